// One launch for many quartet classes of a small system.
//
// A class of a few thousand quartets runs 5 to 30 us, about as long as its launch
// and the gap behind it take; a water energy spent 330 of its 460 us on 19 such
// launches.  Here the workgroups of all those classes run side by side in one
// launch: a workgroup finds its class from a table of block offsets and runs that
// class's body of the straight-line kernels on the class's argument record.  The
// kernel needs the registers of its largest class (512, one wavefront per SIMD),
// so it takes only classes that leave the chip mostly idle when run alone.
#include "vsvb_internal.h"

namespace vsvb {

namespace {

template <int kMode>
__device__ __forceinline__ void small_class(int q, const QuartetArgs& a, const Place& at, double* btab) {
#define VSVB_CLASS(LA, LB, LC, LD)                                  \
  case quartet_class(LA, LB, LC, LD):                               \
    stage_boys<LA + LB + LC + LD>(a.boys, btab);                    \
    if constexpr (kMode == 0)                                       \
      quartet_part<LA, LB, LC, LD, 0>(a, at, btab);                 \
    else if constexpr (LA == LC && LB == LD)                        \
      quartet_part<LA, LB, LC, LD, 1>(a, at, btab);                 \
    else                                                            \
      quartet_part<LA, LB, LC, LD, 2>(a, at, btab);                 \
    break;
  switch (q) {
    VSVB_CLASS(0, 0, 0, 0)
    VSVB_CLASS(1, 0, 0, 0)
    VSVB_CLASS(1, 0, 1, 0)
    VSVB_CLASS(1, 1, 0, 0)
    VSVB_CLASS(1, 1, 1, 0)
    VSVB_CLASS(1, 1, 1, 1)
    VSVB_CLASS(2, 0, 0, 0)
    VSVB_CLASS(2, 0, 1, 0)
    VSVB_CLASS(2, 0, 1, 1)
    VSVB_CLASS(2, 0, 2, 0)
    VSVB_CLASS(2, 1, 0, 0)
    VSVB_CLASS(2, 1, 1, 0)
    VSVB_CLASS(2, 1, 1, 1)
    VSVB_CLASS(2, 1, 2, 0)
    VSVB_CLASS(2, 1, 2, 1)
    VSVB_CLASS(2, 2, 0, 0)
    VSVB_CLASS(2, 2, 1, 0)
    VSVB_CLASS(2, 2, 1, 1)
    VSVB_CLASS(2, 2, 2, 0)
  }
#undef VSVB_CLASS
}

// kMode 0: energy; 1: J/K, classes of different bra and ket transposed.
template <int kMode>
__global__ void __launch_bounds__(256) small_kernel(SmallLaunch s, const QuartetArgs* __restrict__ gs) {
  __shared__ __attribute__((aligned(16))) double btab[kBoysCLen];
  int k = 0;
  while (k + 1 < s.n && blockIdx.x >= (unsigned)s.block0[k + 1]) ++k;  // uniform
  const unsigned local = blockIdx.x - (unsigned)s.block0[k], blocks = (unsigned)s.blocks[k];
  const QuartetArgs a = gs[k];
  small_class<kMode>(s.q[k], a, Place{local % blocks, blocks, local / blocks}, btab);
}

}  // namespace

hipError_t launch_small(const SmallLaunch& s, const QuartetArgs* gs, bool jk, hipStream_t st) {
  if (s.total <= 0) return hipSuccess;
  if (jk)
    hipLaunchKernelGGL(small_kernel<1>, dim3(s.total), dim3(256), s.lds, st, s, gs);
  else
    hipLaunchKernelGGL(small_kernel<0>, dim3(s.total), dim3(256), 0, st, s, gs);
  return hipGetLastError();
}

}  // namespace vsvb

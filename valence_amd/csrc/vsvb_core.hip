// VSVB energy path on MI355X: context, schedule and launch plans, dense products,
// energy and adjoint gradient, batches, C ABI.
//
// Per call (all on the context's stream, inputs already resident):
//   geometry  -> primitive-pair data, S_ao / h_ao (Obara-Saika), Schwarz bounds (vsvb_pairs.hip)
//   weights   -> effective orbital weights C (NDF expansion, angn scaling) and the
//                reference's per-(orbital, shell) weight screen for the ERIs
//   S = C S_ao C^T, h = C h_ao C^T, P = S^-1 per spin block (closed form of the
//   first- and second-order cofactors of the spin-orbital overlap), R = C' P C'^T
//   E1 = sum_s w_s tr(h_s P_s), E2 from the shell-quartet kernels, E = E1 + E2 + E_nuc
//   gradient: J/K from the same quartets (computed anew by every call), then
//   dE/dC_s = 2 P_s C_s F_s (1 - R_s S_ao) with F_s = dE/dR_s.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstdio>
#include <cstring>
#include <map>
#include <memory>
#include <mutex>
#include <numeric>
#include <string>
#include <vector>

#include "vsvb_internal.h"

namespace vsvb {
#include "eri_flops.inc"
}

using namespace vsvb;

// ---------------------------------------------------------------------------
// errors
// ---------------------------------------------------------------------------
namespace vsvb {
thread_local std::string g_last_error;

int fail(int code, const std::string& msg) {
  g_last_error = msg;
  return code;
}
}  // namespace vsvb

// ---------------------------------------------------------------------------
// host helpers: normalization (norm_prim, valence.F90:2264-2306), angn
// (setangn, valence.F90:2395-2421), Boys table
// ---------------------------------------------------------------------------
static double dblfac(int n) {
  double d = 1.0;
  for (int i = 3; i <= n; i += 2) d *= (double)i;
  return d;
}

static void norm_prim(int l, int n, const double* e, const double* u, double* out) {
  const double pi32 = std::pow(std::acos(-1.0), 1.5);
  const double fac = pi32 * dblfac(2 * l - 1) * std::pow(2.0, -l);
  const double fax = -1.5 - l;
  for (int i = 0; i < n; ++i) out[i] = u[i] * std::pow(fac * std::pow(2.0 * e[i], fax), -0.5);
  double s = 0.0;
  for (int i = 0; i < n; ++i)
    for (int j = 0; j < n; ++j) s += fac * out[i] * out[j] * std::pow(e[i] + e[j], fax);
  s = std::pow(s, -0.5);
  for (int i = 0; i < n; ++i) out[i] *= s;
}

static double angn_of(int lx, int ly, int lz) {
  auto ash = [](int l) {
    double f = 1.0;
    for (int j = 1; j <= 2 * l - 1; j += 2) f *= (double)j;
    return std::sqrt(f);
  };
  return ash(lx + ly + lz) / (ash(lx) * ash(ly) * ash(lz));
}

// F_k(T_i), k < kBoysK, by the positive series in long double then downward recursion.
static std::vector<double> make_boys_table() {
  std::vector<double> tab((size_t)kBoysN * kBoysK);
  for (int i = 0; i < kBoysN; ++i) {
    const long double T = (long double)i * (long double)kBoysDT;
    const int K = kBoysK - 1;
    long double term = 1.0L / (2 * K + 1), sum = term;
    for (int k = 1; k < 2000; ++k) {
      term *= 2.0L * T / (2 * K + 2 * k + 1);
      sum += term;
      if (term < 1e-22L * sum) break;
    }
    const long double ex = expl(-T);
    long double F[kBoysK];
    F[K] = ex * sum;
    for (int m = K - 1; m >= 0; --m) F[m] = (2.0L * T * F[m + 1] + ex) / (2 * m + 1);
    for (int m = 0; m < kBoysK; ++m) tab[(size_t)i * kBoysK + m] = (double)F[m];
  }
  // compact tables: F_{L+k}(T_i) / k! for L = 0..kLTot, k < kBoysCK
  const int KC = kLTot + kBoysCK;
  tab.resize(kBoysCOff + (size_t)(kLTot + 1) * kBoysCLen);
  for (int i = 0; i < kBoysCN; ++i) {
    const long double T = (long double)i * (long double)kBoysCDT;
    const int K = KC - 1;
    long double term = 1.0L / (2 * K + 1), sum = term;
    for (int k = 1; k < 4000; ++k) {
      term *= 2.0L * T / (2 * K + 2 * k + 1);
      sum += term;
      if (term < 1e-22L * sum) break;
    }
    const long double ex = expl(-T);
    long double F[kLTot + kBoysCK];
    F[K] = ex * sum;
    for (int m = K - 1; m >= 0; --m) F[m] = (2.0L * T * F[m + 1] + ex) / (2 * m + 1);
    for (int L = 0; L <= kLTot; ++L) {
      long double fact = 1.0L;
      for (int k = 0; k < kBoysCK; ++k) {
        if (k > 0) fact *= k;
        tab[kBoysCOff + (size_t)L * kBoysCLen + (size_t)i * kBoysCRow + k] = (double)(F[L + k] / fact);
      }
    }
  }
  return tab;
}

// ---------------------------------------------------------------------------
// device: geometry preparation
// ---------------------------------------------------------------------------

// Segments of the shell pairs: consecutive parts of a pair's screened primitive
// list, each a work pair of its own (the contracted integral is the sum over
// bra segments x ket segments, and the contraction with the densities is linear
// in it).  The parent's Schwarz bound comes along, so a quartet of segments is
// screened exactly as the quartet of its parents.
__global__ void k_split(const Pair* __restrict__ pairs, const SegSrc* __restrict__ src, int n,
                        Pair* __restrict__ out) {
  const int t = blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= n) return;
  const SegSrc s = src[t];
  Pair P = pairs[s.pair];
  const int b = s.seg * P.npp / s.nseg, e = (s.seg + 1) * P.npp / s.nseg;
  P.pp0 += b;
  P.npp = e - b;
  P.seg = s.seg;
  out[t] = P;
}

// ---------------------------------------------------------------------------
// device: orbital weights
// ---------------------------------------------------------------------------

// NDF self-overlap scale n_f^-1/2 (normal over the NDF range, valence.F90:144).
__global__ void k_ndf_scale(const OrbEntry* __restrict__ ent, const int* __restrict__ orb_start,
                            const double* __restrict__ coeff, const double* __restrict__ angn,
                            const double* __restrict__ S, int nbf, int first_ndf, int ndf, double* __restrict__ scale) {
  const int f = blockIdx.x * blockDim.x + threadIdx.x;
  if (f >= ndf) return;
  const int o = first_ndf + f;
  double s = 0.0;
  for (int k = orb_start[o]; k < orb_start[o + 1]; ++k)
    for (int l = orb_start[o]; l < orb_start[o + 1]; ++l)
      s += angn[ent[k].tgt] * coeff[k] * angn[ent[l].tgt] * coeff[l] * S[(size_t)ent[k].tgt * nbf + ent[l].tgt];
  scale[f] = 1.0 / sqrt(s);
}

// Effective weights Ct[p][mu] (angn folded, NDFs expanded): one thread per orbital.
__global__ void k_build_orbitals(const OrbEntry* __restrict__ ent, const int* __restrict__ orb_start,
                                 const double* __restrict__ coeff, const double* __restrict__ angn,
                                 const double* __restrict__ ndf_scale, int first_ndf, int nbf, int nsp,
                                 double* __restrict__ Ct) {
  const int p = blockIdx.x * blockDim.x + threadIdx.x;
  if (p >= nsp) return;
  double* c = Ct + (size_t)p * nbf;
  for (int k = orb_start[p]; k < orb_start[p + 1]; ++k) {
    const OrbEntry e = ent[k];
    if (e.kind == 0) {
      c[e.tgt] += angn[e.tgt] * coeff[k];
    } else {
      const int f = e.tgt;
      const double w = coeff[k] * ndf_scale[f - first_ndf];
      for (int l = orb_start[f]; l < orb_start[f + 1]; ++l) c[ent[l].tgt] += angn[ent[l].tgt] * coeff[l] * w;
    }
  }
}

// The reference's per-(orbital, shell) weight screen for the ERIs (int2e,
// valence.F90:3296-3300): the shell is used only if the sum of its squared
// weights, after the orbital is normalized (normal, :2157-2182), exceeds dtol.
// One thread per (orbital, shell); S_pp from the orbital overlap matrix.
__global__ void k_shell_screen(const double* __restrict__ Ct, const double* __restrict__ Sorb, int nsp,
                               const Shell* __restrict__ shells, int nsh, const double* __restrict__ angn, int nbf,
                               double dtol, double* __restrict__ Cs, int* __restrict__ nmasked) {
  const long t = blockIdx.x * (long)blockDim.x + threadIdx.x;
  if (t >= (long)nsp * nsh) return;
  const int p = (int)(t / nsh), sh = (int)(t % nsh);
  const Shell S = shells[sh];
  const double* c = Ct + (size_t)p * nbf + S.ao;
  double* cs = Cs + (size_t)p * nbf + S.ao;
  const double inv = 1.0 / Sorb[(size_t)p * nsp + p];
  const int n = ncart(S.l);
  double sum = 0.0;
  bool nz = false;
  for (int k = 0; k < n; ++k) {
    const double raw = c[k] / angn[S.ao + k];
    sum += raw * raw * inv;
    nz |= c[k] != 0.0;
  }
  const bool keep = sum > dtol;
  for (int k = 0; k < n; ++k) cs[k] = keep ? c[k] : 0.0;
  if (nz && !keep) atomicAdd(nmasked, 1);
}

// ---------------------------------------------------------------------------
// device: small dense algebra (row-major)
// ---------------------------------------------------------------------------
// C[M x N] = alpha * op(A) * op(B) + beta * C;  op(A) is M x K; FP64 matrix cores
// (V_MFMA_F64_16X16X4F64, a SIMD is busy with one for 64 cycles).  Lane layout of
// the instruction (probed on the hardware): A[i][k] is held by lane i + 16k,
// B[k][j] by lane j + 16k, and D[i][j] by lane j + 16 (i mod 4) in its accumulator
// register i / 4.
typedef double v4d __attribute__((ext_vector_type(4)));

__device__ __forceinline__ void gemm_store(double alpha, double beta, double v, double* c) {
  *c = alpha * v + (beta == 0.0 ? 0.0 : beta * *c);
}

// Products with many tiles: a workgroup takes 16 MR x 16 NT elements of C.  MR = 4:
// each of its four wavefronts 16 rows and NT accumulators, so an operand read from
// LDS feeds NT instructions; MR = 2 (at most 32 rows): 16 rows and half of the
// columns each; the next 16 columns of A and rows of B are on their way
// while the current ones are multiplied.  Bounded by the matrix cores and the
// operand loads of the edge tiles: 24576 x 144 x 144 takes 34 us, one
// wavefront per 16 x 16 tile without that overlap took 285.  NT is 3 or 4,
// whichever pads N less.
template <int MR, int NT>
__global__ void __launch_bounds__(256) k_gemm_tile(int M, int N, int K, double alpha, const double* __restrict__ A,
                                                   int lda, int ta, const double* __restrict__ B, int ldb, int tb,
                                                   double beta, double* __restrict__ C, int ldc) {
  constexpr int NC = 16 * NT, RM = 16 * MR, NW = NT * MR / 4;
  __shared__ double As[2][RM][17], Bs[2][16][NC + 1];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wr = 16 * ((tid >> 6) % MR), wc = 16 * NW * ((tid >> 6) / MR);  // the wavefront's corner of the tile
  const int m0 = blockIdx.y * RM, n0 = blockIdx.x * NC;
  const int li = lane & 15, lk = lane >> 4;
  double ra[MR], rb[NT];
  auto fetch = [&](int k0) {
#pragma unroll
    for (int x = 0; x < MR; ++x) {
      const int e = tid + 256 * x, r = m0 + (ta ? e % RM : e >> 4), k = k0 + (ta ? e / RM : e & 15);
      ra[x] = r < M && k < K ? (ta ? A[(size_t)k * lda + r] : A[(size_t)r * lda + k]) : 0.0;
    }
#pragma unroll
    for (int x = 0; x < NT; ++x) {
      const int e = tid + 256 * x, c = n0 + (tb ? e >> 4 : e % NC), k = k0 + (tb ? e & 15 : e / NC);
      rb[x] = c < N && k < K ? (tb ? B[(size_t)c * ldb + k] : B[(size_t)k * ldb + c]) : 0.0;
    }
  };
  auto stage = [&](int buf) {
#pragma unroll
    for (int x = 0; x < MR; ++x) {
      const int e = tid + 256 * x;
      As[buf][ta ? e % RM : e >> 4][ta ? e / RM : e & 15] = ra[x];
    }
#pragma unroll
    for (int x = 0; x < NT; ++x) {
      const int e = tid + 256 * x;
      Bs[buf][tb ? e & 15 : e / NC][tb ? e >> 4 : e % NC] = rb[x];
    }
  };
  v4d acc[NW];
#pragma unroll
  for (int j = 0; j < NW; ++j) acc[j] = v4d{0.0, 0.0, 0.0, 0.0};
  fetch(0);
  stage(0);
  for (int k0 = 0, buf = 0; k0 < K; k0 += 16, buf ^= 1) {
    __syncthreads();  // this step is staged; the other buffer's readers are done
    if (k0 + 16 < K) fetch(k0 + 16);
#pragma unroll
    for (int kk = 0; kk < 16; kk += 4) {
      const double a = As[buf][wr + li][kk + lk];
#pragma unroll
      for (int j = 0; j < NW; ++j)
        acc[j] = __builtin_amdgcn_mfma_f64_16x16x4f64(a, Bs[buf][kk + lk][wc + 16 * j + li], acc[j], 0, 0, 0);
    }
    if (k0 + 16 < K) stage(buf ^ 1);
  }
#pragma unroll
  for (int j = 0; j < NW; ++j)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int row = m0 + wr + lk + 4 * r, col = n0 + wc + 16 * j + li;
      if (row < M && col < N) gemm_store(alpha, beta, acc[j][r], C + (size_t)row * ldc + col);
    }
}

// Few tiles, long K: a workgroup of 16 wavefronts takes one 16 x 16 tile, each
// wavefront a sixteenth of K with its operands straight from memory, eight steps
// of loads in flight (nothing is used twice within a wavefront, so LDS would not
// save a load); the partial tiles are added in LDS in a fixed order.  Bounded by
// the loads' latency, K / 512 of them one after another: 144 x 144 x 4096 takes
// 22 us, 285 with one wavefront walking all of K.
constexpr int kDeepWaves = 16;

__global__ void __launch_bounds__(64 * kDeepWaves)
    k_gemm_deep(int M, int N, int K, double alpha, const double* __restrict__ A, int lda, int ta,
                const double* __restrict__ B, int ldb, int tb, double beta, double* __restrict__ C, int ldc) {
  __shared__ double part[kDeepWaves][256];
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int li = lane & 15, lk = lane >> 4;
  const int row = blockIdx.y * 16 + li, col = blockIdx.x * 16 + li;
  const int per = ((K + 4 * kDeepWaves - 1) / (4 * kDeepWaves)) * 4;  // a multiple of the instruction's four
  const int kb = min(K, wave * per), ke = min(K, kb + per);
  const double* pa = A + (ta ? (size_t)row : (size_t)row * lda);
  const double* pb = B + (tb ? (size_t)col * ldb : (size_t)col);
  const size_t sa = ta ? lda : 1, sb = tb ? 1 : ldb;
  v4d acc = {0.0, 0.0, 0.0, 0.0};
  for (int k0 = kb; k0 < ke; k0 += 32) {
    double a[8], b[8];
#pragma unroll
    for (int x = 0; x < 8; ++x) {
      const int k = k0 + 4 * x + lk;
      a[x] = row < M && k < ke ? pa[(size_t)k * sa] : 0.0;
      b[x] = col < N && k < ke ? pb[(size_t)k * sb] : 0.0;
    }
#pragma unroll
    for (int x = 0; x < 8; ++x) acc = __builtin_amdgcn_mfma_f64_16x16x4f64(a[x], b[x], acc, 0, 0, 0);
  }
#pragma unroll
  for (int r = 0; r < 4; ++r) part[wave][(lk + 4 * r) * 16 + li] = acc[r];
  __syncthreads();
  if (threadIdx.x < 256) {
    double s = 0.0;
#pragma unroll
    for (int w = 0; w < kDeepWaves; ++w) s += part[w][threadIdx.x];
    const int r = blockIdx.y * 16 + (threadIdx.x >> 4), c = blockIdx.x * 16 + (threadIdx.x & 15);
    if (r < M && c < N) gemm_store(alpha, beta, s, C + (size_t)r * ldc + c);
  }
}

// Small products (the orbital algebra of one wave function: tens of thousands
// of multiply-adds per output tile at most) are latency-bound: there vector
// FMAs finish sooner than the matrix-core tiles (FP64 vector and matrix peaks
// are equal on this chip).  A workgroup of kGemmSlices x 256 threads takes one
// 16 x 16 tile: slice s accumulates the 16-wide k-steps s, s + kGemmSlices, ...
// (each thread one output element), with the next step's operands loaded into
// registers while the current one is multiplied, and the slices' partial sums
// are added in LDS at the end.
constexpr int kGemmSlices = 4;

__global__ void __launch_bounds__(256 * kGemmSlices)
    k_gemm_small(int M, int N, int K, double alpha, const double* __restrict__ A, int lda, int ta,
                 const double* __restrict__ B, int ldb, int tb, double beta, double* __restrict__ C, int ldc) {
  __shared__ double As[kGemmSlices][16][17], Bs[kGemmSlices][16][17];
  __shared__ double part[kGemmSlices > 1 ? kGemmSlices - 1 : 1][256];
  const int sl = threadIdx.x >> 8, t = threadIdx.x & 255;
  const int tx = t & 15, ty = t >> 4;
  const int row = blockIdx.y * 16 + ty, col = blockIdx.x * 16 + tx;
  auto load_a = [&](int k0) {
    const int k = k0 + tx;
    return (row < M && k < K) ? (ta ? A[(size_t)k * lda + row] : A[(size_t)row * lda + k]) : 0.0;
  };
  auto load_b = [&](int k0) {
    const int k = k0 + ty;
    return (k < K && col < N) ? (tb ? B[(size_t)col * ldb + k] : B[(size_t)k * ldb + col]) : 0.0;
  };
  const int steps = (K + 16 * kGemmSlices - 1) / (16 * kGemmSlices);  // the same count in every slice
  double acc = 0.0;
  double va = load_a(16 * sl), vb = load_b(16 * sl);
  for (int it = 0; it < steps; ++it) {
    As[sl][ty][tx] = va;
    Bs[sl][ty][tx] = vb;
    __syncthreads();
    const int kn = 16 * (sl + kGemmSlices * (it + 1));  // next step of this slice (zeros past K)
    va = load_a(kn);
    vb = load_b(kn);
#pragma unroll
    for (int k = 0; k < 16; ++k) acc += As[sl][ty][k] * Bs[sl][k][tx];
    __syncthreads();
  }
  if (sl > 0) part[sl - 1][t] = acc;
  __syncthreads();
  if (sl == 0 && row < M && col < N) {
#pragma unroll
    for (int s = 0; s < kGemmSlices - 1; ++s) acc += part[s][t];
    double* c = C + (size_t)row * ldc + col;
    *c = alpha * acc + (beta == 0.0 ? 0.0 : beta * *c);
  }
}

// From this many multiply-adds the matrix cores take a product, and a long K does
// so earlier, since the vector tiles walk it in four slices only (1 x 144 x 4096:
// 71 us there, 22 in k_gemm_deep).  The larger tiles need enough
// workgroups for half of the chip's CUs; below that the 16 x 16 tiles with K split
// spread the work wider.
constexpr double kGemmMfmaMin = 8.0e6;
constexpr int kGemmDeepK = 1024;
constexpr long kGemmTiles = 128;

hipError_t vsvb::gemm(hipStream_t st, int M, int N, int K, double alpha, const double* A, int lda, bool ta,
                      const double* B, int ldb, bool tb, double beta, double* C, int ldc) {
  if (M <= 0 || N <= 0) return hipSuccess;
  const dim3 g((N + 15) / 16, (M + 15) / 16);
  const bool large = (double)M * N * K >= kGemmMfmaMin;
  const int nt = M > 32 && (N + 47) / 48 * 48 < (N + 63) / 64 * 64 ? 3 : 4, mr = M > 32 ? 4 : 2;
  const dim3 gt((N + 16 * nt - 1) / (16 * nt), (M + 16 * mr - 1) / (16 * mr));
  if (large && (long)gt.x * gt.y >= kGemmTiles) {
    if (mr == 2)
      hipLaunchKernelGGL((k_gemm_tile<2, 4>), gt, dim3(256), 0, st, M, N, K, alpha, A, lda, (int)ta, B, ldb, (int)tb,
                         beta, C, ldc);
    else if (nt == 3)
      hipLaunchKernelGGL((k_gemm_tile<4, 3>), gt, dim3(256), 0, st, M, N, K, alpha, A, lda, (int)ta, B, ldb, (int)tb, beta,
                         C, ldc);
    else
      hipLaunchKernelGGL((k_gemm_tile<4, 4>), gt, dim3(256), 0, st, M, N, K, alpha, A, lda, (int)ta, B, ldb, (int)tb, beta,
                         C, ldc);
  } else if (large || K >= kGemmDeepK) {
    hipLaunchKernelGGL(k_gemm_deep, g, dim3(64 * kDeepWaves), 0, st, M, N, K, alpha, A, lda, (int)ta, B, ldb, (int)tb,
                       beta, C, ldc);
  } else {
    hipLaunchKernelGGL(k_gemm_small, g, dim3(256 * kGemmSlices), 0, st, M, N, K, alpha, A, lda, (int)ta, B, ldb,
                       (int)tb, beta, C, ldc);
  }
  return hipGetLastError();
}

// Copy the n x n block starting at (off, off) of an ld-strided matrix.
__global__ void k_copy_block(const double* __restrict__ src, int ld, int off, int n, double* __restrict__ dst) {
  const int t = blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= n * n) return;
  dst[t] = src[(size_t)(off + t / n) * ld + off + t % n];
}

// In-place Gauss-Jordan inverse of an SPD matrix (no pivoting needed: every
// leading block of an SPD matrix has positive diagonal).  One workgroup, for
// matrices of up to kSpdOneBlock rows.
constexpr int kSpdOneBlock = 128;
__global__ void __launch_bounds__(1024) k_spd_inverse(double* __restrict__ a, int n, int* __restrict__ status) {
  extern __shared__ double colk[];
  for (int k = 0; k < n; ++k) {
    const double piv = a[(size_t)k * n + k];
    __syncthreads();
    if (!(piv > 0.0) || !isfinite(piv)) {
      if (threadIdx.x == 0) *status = 1;
      return;
    }
    const double ip = 1.0 / piv;
    for (int i = threadIdx.x; i < n; i += blockDim.x) colk[i] = a[(size_t)i * n + k];
    __syncthreads();
    // scale row k
    for (int j = threadIdx.x; j < n; j += blockDim.x) a[(size_t)k * n + j] = (j == k ? 1.0 : a[(size_t)k * n + j]) * ip;
    __syncthreads();
    // rows by thread / 64 (16 at a time), columns by lane: no index division
    for (int i = threadIdx.x >> 6; i < n; i += blockDim.x >> 6) {
      if (i == k) continue;
      const double f = colk[i];
      for (int j = threadIdx.x & 63; j < n; j += 64) {
        double* aij = a + (size_t)i * n + j;
        *aij = (j == k ? 0.0 : *aij) - f * a[(size_t)k * n + j];
      }
    }
    __syncthreads();
  }
}

// The same Gauss-Jordan elimination for large matrices, one pivot per pair of
// launches so that the whole GPU takes each step (one workgroup would be bound
// by one CU's cache bandwidth: 20 ms for n = 384).  Step k: k_gj_pivot saves
// column k (pivot included) and scales row k off the diagonal; k_gj_update
// eliminates column k from every other row and stores the pivot's inverse.
// The pivot element itself is written only in k_gj_update, after every
// workgroup of k_gj_pivot has read it.
__global__ void k_gj_pivot(double* __restrict__ a, int n, int k, double* __restrict__ colk, int* __restrict__ status) {
  const double piv = a[(size_t)k * n + k];
  if (!(piv > 0.0) || !isfinite(piv)) {
    if (blockIdx.x == 0 && threadIdx.x == 0) *status = 1;
    return;
  }
  const double ip = 1.0 / piv;
  for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) {
    colk[i] = a[(size_t)i * n + k];
    if (i != k) a[(size_t)k * n + i] *= ip;
  }
}

__global__ void k_gj_update(double* __restrict__ a, int n, int k, const double* __restrict__ colk) {
  const int j = blockIdx.x * 64 + (threadIdx.x & 63);
  const int i = blockIdx.y * 4 + (threadIdx.x >> 6);
  if (i >= n || j >= n) return;
  const double ip = 1.0 / colk[k];
  double* aij = a + (size_t)i * n + j;
  if (i == k) {
    if (j == k) *aij = ip;  // row k is otherwise final
    return;
  }
  const double akj = j == k ? ip : a[(size_t)k * n + j];
  *aij = (j == k ? 0.0 : *aij) - colk[i] * akj;
}

// In-place inverse of an SPD matrix: one workgroup for n < grid_min (by
// default up to kSpdOneBlock rows), a pair of launches per pivot from grid_min
// rows up.  colk: n doubles of scratch.
static hipError_t launch_spd_inverse(hipStream_t st, double* a, int n, int* status, double* colk, int grid_min) {
  if (n < grid_min) {
    hipLaunchKernelGGL(k_spd_inverse, dim3(1), dim3(1024), n * sizeof(double), st, a, n, status);
    return hipGetLastError();
  }
  const dim3 g((n + 63) / 64, (n + 3) / 4);
  for (int k = 0; k < n; ++k) {
    hipLaunchKernelGGL(k_gj_pivot, dim3((n + 255) / 256), dim3(256), 0, st, a, n, k, colk, status);
    hipLaunchKernelGGL(k_gj_update, g, dim3(256), 0, st, a, n, k, colk);
  }
  return hipGetLastError();
}

// out[0] += w * sum_ij A[off+i][off+j] * B[i][j]  (A ld-strided block, B n x n)
__global__ void k_trace_prod(const double* __restrict__ A, int ld, int off, const double* __restrict__ B, int n,
                             double w, double* __restrict__ out) {
  __shared__ double red[256];
  double s = 0.0;
  for (int t = blockIdx.x * 256 + threadIdx.x; t < n * n; t += gridDim.x * 256)
    s += A[(size_t)(off + t / n) * ld + off + t % n] * B[t];
  red[threadIdx.x] = s;
  __syncthreads();
  for (int o = 128; o > 0; o >>= 1) {
    if (threadIdx.x < o) red[threadIdx.x] += red[threadIdx.x + o];
    __syncthreads();
  }
  if (threadIdx.x == 0) unsafeAtomicAdd(out, w * red[0]);
}
static unsigned trace_blocks(int n) { return (unsigned)std::clamp(n * (long)n / 4096, 1L, 256L); }

__global__ void k_fill(double* __restrict__ p, size_t n, double v) {
  for (size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x; i < n; i += (size_t)gridDim.x * blockDim.x) p[i] = v;
}

hipError_t vsvb::launch_fill(hipStream_t st, double* p, size_t n, double v) {
  const unsigned nb = (unsigned)std::min<size_t>(1024, (n + 255) / 256 + 1);
  hipLaunchKernelGGL(k_fill, dim3(nb), dim3(256), 0, st, p, n, v);
  return hipGetLastError();
}

// Per-class timing slots before a stage: even words (earliest start) ~0, odd
// words (latest end) 0.  A kernel, not a memset: it may be captured in a graph.
__global__ void k_stamp_reset(unsigned long long* __restrict__ p, int n) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) p[i] = (i & 1) ? 0ull : ~0ull;
}

// After a stage: per class (one workgroup each), the earliest start and the
// latest end over its kStampSlots slot pairs, into out[2 q], out[2 q + 1].
__global__ void __launch_bounds__(kStampSlots) k_stamp_reduce(const unsigned long long* __restrict__ slots,
                                                              unsigned long long* __restrict__ out) {
  __shared__ unsigned long long lo[kStampSlots], hi[kStampSlots];
  const unsigned long long* s = slots + (size_t)blockIdx.x * 2 * kStampSlots;
  lo[threadIdx.x] = s[2 * threadIdx.x];
  hi[threadIdx.x] = s[2 * threadIdx.x + 1];
  __syncthreads();
  for (int o = kStampSlots / 2; o > 0; o >>= 1) {
    if ((int)threadIdx.x < o) {
      lo[threadIdx.x] = lo[threadIdx.x] < lo[threadIdx.x + o] ? lo[threadIdx.x] : lo[threadIdx.x + o];
      hi[threadIdx.x] = hi[threadIdx.x] > hi[threadIdx.x + o] ? hi[threadIdx.x] : hi[threadIdx.x + o];
    }
    __syncthreads();
  }
  if (threadIdx.x == 0) {
    out[2 * blockIdx.x] = lo[0];
    out[2 * blockIdx.x + 1] = hi[0];
  }
}

__global__ void k_fill_u32(uint32_t* __restrict__ p, size_t n, uint32_t v) {
  for (size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x; i < n; i += (size_t)gridDim.x * blockDim.x) p[i] = v;
}

// Clearing counters, flags and status words is done by a kernel, not a memset,
// so that the same code can be captured into a HIP graph.
hipError_t vsvb::launch_zero(hipStream_t st, void* p, size_t bytes) {
  const size_t n = bytes / sizeof(uint32_t);
  hipLaunchKernelGGL(k_fill_u32, dim3((unsigned)std::min<size_t>(256, (n + 255) / 256 + 1)), dim3(256), 0, st,
                     (uint32_t*)p, n, 0u);
  return hipGetLastError();
}

// M <- a*(X + X^T) + b*Y (elementwise, n x n); X, Y may alias nothing of M.
__global__ void k_sym_combine(const double* __restrict__ X, double a, const double* __restrict__ Y, double b, int n,
                              double* __restrict__ M) {
  const size_t t = blockIdx.x * (size_t)blockDim.x + threadIdx.x;
  if (t >= (size_t)n * n) return;
  const int i = (int)(t / n), j = (int)(t % n);
  double v = a * (X[t] + X[(size_t)j * n + i]);
  if (Y) v += b * Y[t];
  M[t] = v;
}

// grad[k] = angn[mu_k] * G[orb_k][mu_k] for the AO entries of occupied orbitals,
// 0 for the rest (the weights involving NDFs follow from k_ndf_grad).
__global__ void k_gather_grad(const OrbEntry* __restrict__ ent, int totlen, int nsp, const double* __restrict__ angn,
                              const double* __restrict__ G, int nbf, double* __restrict__ grad) {
  const int k = blockIdx.x * blockDim.x + threadIdx.x;
  if (k >= totlen) return;
  const OrbEntry e = ent[k];
  grad[k] = (e.kind == 0 && e.orb < nsp) ? angn[e.tgt] * G[(size_t)e.orb * nbf + e.tgt] : 0.0;
}

// Gradient of the weights that involve NDFs (ndf2obs, src/valence.F90:2191-2247,
// with the NDF normalization of :144).  Orbital p's effective AO weights are
//   C_p = sum_{AO entries k} angn c_k e_mu(k) + sum_{entries k -> NDF f} c_k s_f d_f,
//   d_f = sum_{weights l of f} angn c_l e_mu(l),   s_f = (d_f^T S d_f)^(-1/2),
// so that, with G_p = dE/dC_p,
//   entry k -> f of orbital p:   dE/dc_k = s_f (d_f . G_p)
//   weight l of NDF f:           dE/dc_l = s_f angn (g_f - s_f^2 (d_f . g_f) S d_f)[mu(l)],
//   g_f = sum over every entry k -> f (any occupied orbital p) of c_k G_p.
// One workgroup (256 threads) per NDF; dv, gv: [ndf][nbf] scratch.
__global__ void __launch_bounds__(256) k_ndf_grad(const OrbEntry* __restrict__ ent, const int* __restrict__ orb_start,
                                                  const double* __restrict__ coeff, const double* __restrict__ angn,
                                                  const double* __restrict__ ndf_scale, const double* __restrict__ S,
                                                  const double* __restrict__ G, int nsp, int nbf, int first_ndf,
                                                  double* __restrict__ dv, double* __restrict__ gv,
                                                  double* __restrict__ grad) {
  __shared__ double red[256];
  const int f = blockIdx.x, o = first_ndf + f, tid = threadIdx.x;
  double* d = dv + (size_t)f * nbf;
  double* g = gv + (size_t)f * nbf;
  const double sf = ndf_scale[f];
  auto block_sum = [&](double v) {
    red[tid] = v;
    __syncthreads();
    for (int h = 128; h > 0; h >>= 1) {
      if (tid < h) red[tid] += red[tid + h];
      __syncthreads();
    }
    const double r = red[0];
    __syncthreads();
    return r;
  };
  for (int mu = tid; mu < nbf; mu += 256) d[mu] = 0.0;
  __syncthreads();
  if (tid == 0)
    for (int l = orb_start[o]; l < orb_start[o + 1]; ++l) d[ent[l].tgt] += angn[ent[l].tgt] * coeff[l];
  for (int mu = tid; mu < nbf; mu += 256) {
    double t = 0.0;
    for (int p = 0; p < nsp; ++p)
      for (int k = orb_start[p]; k < orb_start[p + 1]; ++k)
        if (ent[k].kind == 1 && ent[k].tgt == o) t += coeff[k] * G[(size_t)p * nbf + mu];
    g[mu] = t;
  }
  __syncthreads();
  double t = 0.0;
  for (int mu = tid; mu < nbf; mu += 256) t += d[mu] * g[mu];
  const double dg = block_sum(t);
  for (int p = 0; p < nsp; ++p)
    for (int k = orb_start[p]; k < orb_start[p + 1]; ++k) {
      if (ent[k].kind != 1 || ent[k].tgt != o) continue;  // the same for every thread
      double u = 0.0;
      for (int mu = tid; mu < nbf; mu += 256) u += d[mu] * G[(size_t)p * nbf + mu];
      const double v = block_sum(u);
      if (tid == 0) grad[k] = sf * v;
    }
  for (int l = orb_start[o]; l < orb_start[o + 1]; ++l) {
    const int mu = ent[l].tgt;
    double u = 0.0;
    for (int nu = tid; nu < nbf; nu += 256) u += S[(size_t)mu * nbf + nu] * d[nu];
    const double sd = block_sum(u);
    if (tid == 0) grad[l] = sf * angn[mu] * (g[mu] - sf * sf * dg * sd);
  }
}

hipError_t vsvb::launch_gather_grad(vsvb_context* c, const double* gradC, double* grad) {
  hipLaunchKernelGGL(k_gather_grad, dim3((c->totlen + 255) / 256), dim3(256), 0, c->stream, c->d_ent.p, c->totlen,
                     c->nsp, c->d_angn.p, gradC, c->nbf, grad);
  if (c->ndf > 0)
    hipLaunchKernelGGL(k_ndf_grad, dim3(c->ndf), dim3(256), 0, c->stream, c->d_ent.p, c->d_orb_start.p, c->d_coeff.p,
                       c->d_angn.p, c->d_ndf_scale.p, c->d_S.p, gradC, c->nsp, c->nbf, c->first_ndf, c->d_ndf_d.p,
                       c->d_ndf_g.p, grad);
  return hipGetLastError();
}

__global__ void k_final_energy(const double* __restrict__ e1, const double* __restrict__ e2, double enuc,
                               double* __restrict__ out) {
  out[0] = e1[0] + e2[0] + enuc;
}

// ---------------------------------------------------------------------------
// context
// ---------------------------------------------------------------------------

static double nuclear_repulsion(int natom, const double* xyz, const double* Z) {
  // get_nuclear_repulsion_energy (src/tools_module.F90:19-40)
  double e = 0.0;
  for (int i = 1; i < natom; ++i)
    for (int j = 0; j < i; ++j) {
      const double zij = Z[i] * Z[j];
      if (std::fabs(zij) > 1e-12) {
        const double dx = xyz[3 * i] - xyz[3 * j], dy = xyz[3 * i + 1] - xyz[3 * j + 1], dz = xyz[3 * i + 2] - xyz[3 * j + 2];
        const double rsq = dx * dx + dy * dy + dz * dz;
        if (rsq > 1e-5) e += zij * std::pow(rsq, -0.5);
      }
    }
  return e;
}

static const int kPairLs[kNPairClass][2] = {{0, 0}, {1, 0}, {1, 1}, {2, 0}, {2, 1}, {2, 2}};

static int pair_class_of(int la, int lb) {
  for (int c = 0; c < kNPairClass; ++c)
    if (kPairLs[c][0] == la && kPairLs[c][1] == lb) return c;
  return -1;
}

static hipError_t launch_quartet_class(int bc, int kc, const QuartetArgs& a, bool jk, bool tr, int nblocks,
                                       size_t lds, hipStream_t st) {
  switch (bc) {
    case 0: return launch_quartet_b0(kc, a, jk, tr, nblocks, lds, st);
    case 1: return launch_quartet_b1(kc, a, jk, tr, nblocks, lds, st);
    case 2: return launch_quartet_b2(kc, a, jk, tr, nblocks, lds, st);
    case 3: return launch_quartet_b3(kc, a, jk, tr, nblocks, lds, st);
    case 4: return launch_quartet_b4(kc, a, jk, tr, nblocks, lds, st);
    case 5: return launch_quartet_b5(kc, a, jk, tr, nblocks, lds, st);
  }
  return hipErrorInvalidValue;
}

static hipError_t launch_groups_class(int bc, int kc, const QuartetArgs* gs, int ng, bool tr, int nblocks, size_t lds,
                                      unsigned long long* stamp, hipStream_t st) {
  switch (bc) {
    case 0: return launch_groups_b0(kc, gs, ng, tr, nblocks, lds, stamp, st);
    case 1: return launch_groups_b1(kc, gs, ng, tr, nblocks, lds, stamp, st);
    case 2: return launch_groups_b2(kc, gs, ng, tr, nblocks, lds, stamp, st);
    case 3: return launch_groups_b3(kc, gs, ng, tr, nblocks, lds, stamp, st);
    case 4: return launch_groups_b4(kc, gs, ng, tr, nblocks, lds, stamp, st);
    case 5: return launch_groups_b5(kc, gs, ng, tr, nblocks, lds, stamp, st);
  }
  return hipErrorInvalidValue;
}

static int class_occupancy(int bc, int kc, bool jk, bool tr, size_t lds) {
  switch (bc) {
    case 0: return occupancy_b0(kc, jk, tr, lds);
    case 1: return occupancy_b1(kc, jk, tr, lds);
    case 2: return occupancy_b2(kc, jk, tr, lds);
    case 3: return occupancy_b3(kc, jk, tr, lds);
    case 4: return occupancy_b4(kc, jk, tr, lds);
    case 5: return occupancy_b5(kc, jk, tr, lds);
  }
  return 1;
}

static int quartet_class_index(int bc, int kc) { return bc * (bc + 1) / 2 + kc; }

static int class_parts(int q, bool jk) { return jk ? kPartsJk[q] : kPartsEnergy[q]; }

static int class_bra(int q) {
  for (int b = 0; b < kNPairClass; ++b)
    if (q < quartet_class_index(b, b) + 1) return b;
  return kNPairClass - 1;
}

// Algorithmic FP64 operations of the density contraction per contracted quartet.
static double digestion_flops(int q, int nspin, bool jk) {
  int bc = 0, kc = 0;
  for (int b = 0; b < kNPairClass; ++b)
    for (int k = 0; k <= b; ++k)
      if (quartet_class_index(b, k) == q) { bc = b; kc = k; }
  const double nab = ncart(kPairLs[bc][0]) * ncart(kPairLs[bc][1]);
  const double ncd = ncart(kPairLs[kc][0]) * ncart(kPairLs[kc][1]);
  return jk ? nab * ncd * (4.0 + 8.0 * nspin) : nab * ncd * (2.0 + 4.0 * nspin) + 2.0 * nab;
}

// Straight-line kernel: energy units are 64-pair bra tiles x chunks of ket
// pairs (one wavefront each, four per workgroup); J/K units are 256-pair bra
// strips x chunks of ket pairs (one workgroup each), with the exchange rows of
// a unit in LDS when lds_on and they fit, or, transposed (tr, bra and ket
// classes differ), ket strips of 256 pairs x chunks of bra pairs.  per_cu = 0:
// as many workgroups as the kernel's occupancy allows (energy: at most 2048,
// measured fastest for the low-AM classes).
constexpr double kEnergyUnitsPerWave = 32.0;
// Work units are 32-bit indices; counters may run past the last unit by at
// most a claim per workgroup, which the margin covers.
constexpr long long kMaxUnits = (long long)INT32_MAX - (1LL << 24);
constexpr double kJkUnitsPerBlock = 16.0;

// Work lists of a quartet class.  A lane evaluates its quartet's primitive
// quartets one after another, about 0.25 us each when few wavefronts share a
// SIMD (a (ss|ss) quartet of six-fold contracted shells: 1296 of them, 330 us),
// so a class with few quartets takes segments of its pairs instead: more lanes,
// each with a shorter chain, for one more density contraction per segment
// quartet.  Of the nine pairs of levels the one with the least estimated time is
// taken: the chain of the longest entries, plus the wavefronts per SIMD times
// the average chain, in units of a primitive quartet, where what a quartet costs
// beside its primitives is `tail` of them.  The tails are fitted to the class
// times of all nine pairs of levels on water, C2H6, C3H8, C5H12, C8H18 and the
// H8 and H12 chains: the pairs chosen sum to 5.43 ms where the best sum to 5.26
// (energy), 14.2 to 13.5 ms (J/K); whole pairs alone 16.5 and 18.1 ms.
constexpr double kTailEnergy = 6.0, kTailJk = 45.0, kTailDensity = 25.0;
static void choose_levels(const vsvb_context* c, int bc, int kc, bool jk, bool tr, int* lb, int* lk) {
  *lb = *lk = 0;
  if (c->nlevels < 2 || c->pair_chunk > 0) return;  // a forced chunk width: whole pairs
  const int q = bc * (bc + 1) / 2 + kc;
  const int nd = jk ? c->ndens : 1;
  const double digest = digestion_flops(q, c->nunpd > 0 ? 2 : 1, jk) * nd;
  const double tail = (jk ? kTailJk + kTailDensity * (nd - 1) : kTailEnergy) +
                      (kFlopsHrr[q] + digest) / kFlopsPerPrimQuartet[q];
  double best = 0.0;
  for (int b = 0; b < c->nlevels; ++b)
    for (int k = 0; k < c->nlevels; ++k) {
      if (bc == kc && b != k) continue;
      const WorkList &B = c->work[bc][b], &K = c->work[kc][k];
      const WorkList &lane = tr ? K : B, &uni = tr ? B : K;
      const double tiles = jk ? 4.0 * ((lane.n + kStripB - 1) / kStripB) : (double)((lane.n + kTileB - 1) / kTileB);
      const double waves = tiles * uni.n * (bc == kc ? 0.5 : 1.0);
      const double t = B.longest * (double)K.longest + tail + waves / (4.0 * c->ncu) * (B.mean * K.mean + tail);
      if ((b == 0 && k == 0) || t < best) {
        best = t;
        *lb = b;
        *lk = k;
      }
    }
}

// Most workgroups (of each part) of a straight-line energy launch.
static int energy_grid(const vsvb_context* c, int bc, int kc) {
  return std::min(2048, class_occupancy(bc, kc, false, false, 0) * c->ncu);
}

static ClassLaunch straight_launch(vsvb_context* c, int bc, int kc, bool jk, int per_cu, bool lds_on, bool tr) {
  ClassLaunch L;
  L.tr = jk && tr && bc != kc;
  choose_levels(c, bc, kc, jk, L.tr, &L.lb, &L.lk);
  const int nb = c->work[bc][L.lb].n, nk = c->work[kc][L.lk].n;
  L.per_cu = per_cu;
  if (nb <= 0 || nk <= 0) return L;
  if (!jk) {
    const int cap = energy_grid(c, bc, kc);
    const int nbt = (nb + kTileB - 1) / kTileB;
    // Ket chunks as wide as still leave kEnergyUnitsPerWave units per resident
    // wavefront: large (and sparse) systems claim up to 64 kets at once and
    // skip the screened ones inside the unit; small ones keep one ket per unit.
    int kch = c->pair_chunk > 0 ? c->pair_chunk : 1;
    while (c->pair_chunk == 0 && kch < 64 &&
           (double)nbt * ((nk + 2 * kch - 1) / (2 * kch)) >= kEnergyUnitsPerWave * 4.0 * cap)
      kch *= 2;
    L.kchunk = kch;
    // one-ket units of one class stop at the diagonal: tile t has 64 (t + 1) kets
    const long long units = kch == 1 && bc == kc ? (long long)kTileB / 2 * nbt * (nbt + 1)
                                                 : (long long)nbt * ((nk + kch - 1) / kch);
    L.overflow = units > kMaxUnits;
    L.units = L.overflow ? 0 : (int)units;
    L.blocks = std::min((L.units + 3) / 4, cap);
    L.strips = (nbt + kSegTiles - 1) / kSegTiles;
    // a wavefront's step over the tiles (one-ket units) or chunks (chunked ones)
    // from round to round: about 0.38 of their number, coprime to it
    const int nw = 4 * L.blocks, period = kch > 1 ? (nk + kch - 1) / kch : (bc != kc ? nbt : 0);
    if (period > 2 && period < nw) {
      int step = std::max(1, (int)std::lround(0.382 * period));
      while (std::gcd(step, period) != 1) ++step;
      L.shift = ((step - nw) % period + period) % period;
    }
    return L;
  }
  const int rows = L.tr ? ncart(kPairLs[bc][0]) + ncart(kPairLs[bc][1]) : ncart(kPairLs[kc][0]) + ncart(kPairLs[kc][1]);
  L.strips = L.tr ? (nk + kStripK - 1) / kStripK : (nb + kStripB - 1) / kStripB;
  const int side = L.tr ? nb : nk;  // pairs claimed from each strip's counter
  const size_t kb = (size_t)c->nbf * rows * sizeof(double);
  L.lds = (lds_on && kb <= kMaxLdsK) ? kb : 0;
  const int occ = class_occupancy(bc, kc, true, L.tr, L.lds);
  const int cap = (per_cu > 0 ? std::min(per_cu, occ) : occ) * c->ncu;
  // Claims of several pairs when that still leaves kJkUnitsPerBlock units per
  // workgroup (large, sparse systems), one pair per claim otherwise.
  int kch = c->pair_chunk > 0 ? c->pair_chunk : 1;
  while (c->pair_chunk == 0 && kch < 64 &&
         (double)L.strips * ((side + 2 * kch - 1) / (2 * kch)) >= kJkUnitsPerBlock * cap)
    kch *= 2;
  L.kchunk = kch;
  const long long units = (long long)L.strips * ((side + kch - 1) / kch);
  L.overflow = units > kMaxUnits;
  L.units = L.overflow ? 0 : (int)units;
  L.blocks = std::min(L.units, cap);
  return L;
}

// Default J/K grid: at most 4 workgroups per CU.  Filling every slot was
// measured slower on the batch tuner's workloads for the low-AM classes (more
// concurrent units thrash the caches: (ss|ss) 1.31 -> 1.05 ms, (ds|ss) 0.52 ->
// 0.30 ms on C8H18); the batch tuner still tries every grid.
constexpr int kDefaultJkPerCu = 4;

// Default J/K orientation of a straight-line class: the one with the smaller
// product of its units (strips of 256 pairs, idle lanes included, times the pairs of
// the other side) and the cost of a unit.  A transposed unit costs `cost` of a
// normal one, from both orientations' times of every class of C8H18 (210 AOs) and of
// LiF slabs of 32, 64 and 128 atoms (384, 768, 1536): (ps|ss) 1.7 at every size (1389
// us against 738, 378 ms against 224); d-heavy bras 0.8 (large bra blocks mean many
// atomics per lane in a normal unit: (dd|ss) 55 us against 315, 5.3 ms against 10.5);
// the bras between 0.85 in small bases and 1.3 in large ones, where the larger number
// of exchange rows of a transposed unit takes LDS from other workgroups ((pp|ps) 231
// us against 406, but 7.1 ms against 6.3 at 768 AOs and 21 against 7.2 at 1536).  For those
// bras an orientation whose exchange rows fit in LDS goes before one whose rows do
// not; d-heavy ones are faster transposed without LDS, too.
constexpr int kLargeBasis = 300;
static bool transposed_default(vsvb_context* c, int bc, int kc) {
  if (bc == kc) return false;
  const int nb = c->pair_off[bc + 1] - c->pair_off[bc], nk = c->pair_off[kc + 1] - c->pair_off[kc];
  if (nb <= 0 || nk <= 0) return false;
  // exchange staging: the normal unit holds NC + ND rows of nbf, the transposed one NA + NB
  const size_t row = (size_t)c->nbf * sizeof(double);
  const bool fit_n = row * (ncart(kPairLs[kc][0]) + ncart(kPairLs[kc][1])) <= kMaxLdsK;
  const bool fit_t = row * (ncart(kPairLs[bc][0]) + ncart(kPairLs[bc][1])) <= kMaxLdsK;
  if (bc < 4 && fit_n != fit_t) return fit_t;
  const double un = (double)((nb + kStripB - 1) / kStripB) * nk, ut = (double)((nk + kStripK - 1) / kStripK) * nb;
  const double cost = bc >= 4 ? 0.8 : bc == 1 ? 1.7 : c->nbf < kLargeBasis ? 0.85 : 1.3;
  return ut * cost < un;
}

// Cooperative kernel: one unit per (bra pair, ket pair); claim = 0 picks about
// units / (4 * workgroups), between 1 and 64, or, for classes large enough to
// leave 16 claims of more than 64 units per workgroup (large, mostly screened
// systems), units / (16 * workgroups) up to 1024.
static ClassLaunch coop_launch(vsvb_context* c, int q, bool jk, int per_cu, int claim) {
  ClassLaunch L;
  L.coop = true;
  L.per_cu = per_cu;
  const int bc = class_bra(q), kc = q - quartet_class_index(bc, 0);
  // few quartets: one wavefront per primitive quartet ((dd|dp) of water, nine
  // contracted quartets of three primitive ones each: 41 -> 17 us)
  if (c->nlevels > 1 && c->pair_chunk == 0 && c->ndens == 1 && c->work[bc][1].n * (double)c->work[kc][1].n <= 8.0 * c->ncu)
    L.lb = L.lk = 1;
  const int nb = c->work[bc][L.lb].n, nk = c->work[kc][L.lk].n;
  if (nb <= 0 || nk <= 0 || c->coop_idx[q] < 0) return L;  // an empty class launches nothing
  L.overflow = (long long)nb * nk > kMaxUnits;
  if (L.overflow) return L;
  L.units = nb * nk;
  const int occ = coop_occupancy(c->coop_idx[q], jk);
  L.blocks = std::min(L.units, (per_cu > 0 ? std::min(per_cu, occ) : occ) * c->ncu);
  const int big = L.units / (16 * L.blocks);
  L.claim = claim > 0 ? std::min(claim, 64)
                      : (big > 64 ? std::min(big, 1024) : std::max(1, std::min(64, L.units / (4 * L.blocks))));
  return L;
}

static ClassLaunch policy_launch(vsvb_context* c, int q, const Policy& p) {
  const int bc = class_bra(q), kc = q - quartet_class_index(bc, 0);
  if (c->coop_idx[q] >= 0) return coop_launch(c, q, true, p.per_cu, p.claim);
  return straight_launch(c, bc, kc, true, p.per_cu, p.lds_on, p.tr);
}

// Most primitive pairs per segment, by level and pair class (ss, ps, pp, ds,
// dp, dd): a quarter and a twelfth of the pairs of six-fold, three-fold and
// uncontracted shells.
constexpr int kSegLen[kLevels][kNPairClass] = {{0, 0, 0, 0, 0, 0}, {9, 6, 3, 3, 1, 1}, {3, 2, 1, 1, 1, 1}};
// Workgroups up to which a class joins the shared launch of a small system: it
// runs one workgroup per CU, so a class that fills the chip is faster alone.  A
// forced chunk width keeps every class apart.
constexpr int kSmallBlocks = 320;
// Shell pairs up to which a context holds segment lists: above, every class
// that matters fills the chip with whole pairs.
constexpr int kSplitMaxPairs = 20000;

// Work lists and class launches for the screened primitive counts kept[pair]
// (scheduled order; null: unscreened, before the first geometry).
static int plan_work(vsvb_context* c, const int* kept) {
  c->h_seg.clear();
  for (int pc = 0; pc < kNPairClass; ++pc) {
    const int b = c->pair_off[pc], e = c->pair_off[pc + 1];
    auto count = [&](int i) { return kept ? kept[i] : c->h_pairs[i].npp; };
    double sum = 0.0;
    int most = 0;
    for (int i = b; i < e; ++i) {
      sum += count(i);
      most = std::max(most, count(i));
    }
    for (int l = 0; l < c->nlevels; ++l) {
      WorkList& W = c->work[pc][l];
      if (l > 0 && !kept) W.n = W.cap;
      if (l > 0 && kept) {
        // segment by segment over the pairs, so that neighbouring lanes hold
        // different pairs (their accumulators' rows differ)
        W.off = (int)c->h_seg.size();
        for (int s = 0, any = 1; any; ++s) {
          any = 0;
          for (int i = b; i < e; ++i) {
            const int ns = std::max(1, (count(i) + kSegLen[l][pc] - 1) / kSegLen[l][pc]);
            if (s < ns) {
              c->h_seg.push_back(SegSrc{i, s, ns});
              any = 1;
            }
          }
        }
        W.n = (int)c->h_seg.size() - W.off;
      }
      W.longest = l > 0 ? std::min(most, kSegLen[l][pc]) : most;
      W.mean = W.n > 0 ? sum / W.n : 0.0;
    }
  }
  c->partial_total = 0;
  for (int m = 0; m < 2; ++m) {
    c->small[m] = SmallLaunch{};
    std::fill(c->in_small[m], c->in_small[m] + kNQuartetClass, false);
  }
  for (int q = 0; q < kNQuartetClass; ++q) {
    const int bc = class_bra(q), kc = q - quartet_class_index(bc, 0);
    const bool coop = c->coop_idx[q] >= 0;  // its step tables are all the class has
    c->le[q] = coop ? coop_launch(c, q, false, 0, 0) : straight_launch(c, bc, kc, false, 0, false, false);
    c->ljk[q] = coop ? coop_launch(c, q, true, 0, 0)
                     : straight_launch(c, bc, kc, true, kDefaultJkPerCu, true, transposed_default(c, bc, kc));
    if (c->le[q].overflow || c->ljk[q].overflow)
      return fail(VSVB_ERR_UNSUPPORTED, "shell-pair classes too large for 32-bit work-unit indices");
    if (c->has_pol[q]) {
      const ClassLaunch cl = policy_launch(c, q, c->pol[q]);
      if (!cl.overflow && (cl.units > 0 || c->ljk[q].units <= 0)) c->ljk[q] = cl;
    }
    if (c->nlevels > 1 && c->pair_chunk == 0 && c->ndens == 1 && c->coop_idx[q] < 0) {
      c->in_small[0][q] = c->le[q].units > 0 && c->le[q].kchunk == 1 && c->le[q].blocks * kPartsEnergy[q] <= kSmallBlocks;
      // the shared J/K launch has the transposed units of classes of different bra and ket
      const ClassLaunch cl = straight_launch(c, bc, kc, true, kDefaultJkPerCu, true, bc != kc);
      if (cl.units > 0 && !cl.overflow && cl.kchunk == 1 && cl.blocks * kPartsJk[q] <= kSmallBlocks) {
        c->in_small[1][q] = true;
        c->ljk[q] = cl;
      }
    }
    // energy kernels write four slots per block and part
    c->partial_per_class[q] = (size_t)c->le[q].blocks * 4 * (c->le[q].coop ? 1 : class_parts(q, false));
    c->partial_total += c->partial_per_class[q];
  }
  // the shared launches: high angular momenta (the longest chains) first
  for (int m = 0; m < 2; ++m) {
    SmallLaunch& s = c->small[m];
    for (int q = kNQuartetClass - 1; q >= 0; --q) {
      if (!c->in_small[m][q]) continue;
      const ClassLaunch& cl = m ? c->ljk[q] : c->le[q];
      s.q[s.n] = q;
      s.block0[s.n] = s.total;
      s.blocks[s.n] = cl.blocks;
      s.total += cl.blocks * class_parts(q, m != 0);
      s.lds = std::max(s.lds, (unsigned)cl.lds);
      ++s.n;
    }
    if (s.n < 2) {  // nothing to share
      std::fill(c->in_small[m], c->in_small[m] + kNQuartetClass, false);
      s = SmallLaunch{};
    }
  }
  return VSVB_OK;
}

// A device buffer of the context: allocated, or carved from the context's
// arena (the allocation-free entry point); an arena too small is reported with
// the size the system needs.
template <typename T>
static hipError_t device_buffer(vsvb_context* c, vsvb::DevBuf<T>& b, size_t count) {
  return c->arena ? b.carve(*c->arena, count) : b.alloc(count);
}

// The orbital algebra of this wave function runs along its entry lists
// (vsvb_orbital.hip): few enough orbitals for its LDS and no more than AOs (its
// m x m results stand in nsp x nbf arrays), no NDFs, no spin-coupled pairs, and no
// spin block that is to be inverted grid-wide.
static bool entry_list_orbitals(const vsvb_context* c) {
  return c->ndf == 0 && c->npair == 0 && c->nsp <= std::min(kOrbMax, c->nbf) && c->nbf <= kOrbMaxBasis &&
         std::max(c->nalpha_rows, c->ndocc) < c->grid_inverse_min;
}

static OrbArgs orb_args(const vsvb_context* c) {
  OrbArgs a{};
  a.ent = c->d_ent.p;
  a.orb_start = c->d_orb_start.p;
  a.ao_ptr = c->d_ao_ptr.p;
  a.ao_orb = c->d_ao_orb.p;
  a.shells = c->d_shells.p;
  a.coeff = c->d_coeff.p;
  a.angn = c->d_angn.p;
  a.S = c->d_S.p;
  a.H = c->d_H.p;
  a.J = c->d_J.p;
  a.K = c->d_K.p;
  a.Ct = c->d_Ct.p;
  a.Cs = c->d_Cs.p;
  a.T = c->d_tmp.p;
  a.TH = c->d_tmp2.p;
  a.Y[0] = c->d_X.p;
  a.Y[1] = c->d_Z.p;
  a.V[0] = c->d_tmp2.p;  // C h is done with by then
  a.V[1] = c->d_Rfull.p;
  a.Sorb = c->d_Sorb.p;
  a.Horb = c->d_Horb.p;
  a.P = c->d_P.p;
  a.R = c->d_R.p;
  a.F = c->d_F.p;
  a.G = c->d_gradC.p;
  a.grad = c->d_grad.p;
  a.partial = c->d_partial.p;
  a.scal = c->d_scal.p;
  a.status = c->d_status.p;
  a.nbf = c->nbf;
  a.nsp = c->nsp;
  a.nsh = c->nsh;
  a.totlen = c->totlen;
  a.nspin = c->nunpd > 0 ? 2 : 1;
  a.nalpha = c->nalpha_rows;
  a.nunpd = c->nunpd;
  a.ndocc = c->ndocc;
  a.dtol = c->dtol;
  return a;
}

static int read_options(const vsvb_system* s, const vsvb_options* opt, vsvb_context* c) {
  if (!s) return fail(VSVB_ERR_ARG, "null system");
  if (s->natom < 1 || s->nshell_type < 1) return fail(VSVB_ERR_ARG, "empty molecule or basis");
  c->device = opt ? opt->device : 0;
  c->tau = (opt && opt->quartet_tau > 0) ? opt->quartet_tau : 1e-17;
  c->pair_chunk = opt ? opt->pair_chunk : 0;
  if (c->pair_chunk < 0 || c->pair_chunk > 64) return fail(VSVB_ERR_ARG, "pair_chunk must be 0 (automatic) or 1..64");
  const int gim = opt ? opt->grid_inverse_min : 0;
  if (gim < 0) return fail(VSVB_ERR_ARG, "grid_inverse_min must be 0 (default) or at least 1");
  c->grid_inverse_min = gim > 0 ? gim : kSpdOneBlock + 1;
  return VSVB_OK;
}

// What a context holds of its system on the host: sizes, shells and shell pairs,
// what a schedule needs of them, orbital entries.
struct HostBasis {
  std::vector<Shell> shells;
  std::vector<double> pexp, pcoef, angn;
  std::vector<int> ao_shell;
};

static int describe_system(const vsvb_system* s, const vsvb_options* opt, vsvb_context* c, HostBasis& hb) {
  std::vector<Shell>& shells = hb.shells;
  std::vector<double>&pexp = hb.pexp, &pcoef = hb.pcoef, &angn = hb.angn;
  std::vector<int>& ao_shell = hb.ao_shell;
  c->natom = s->natom;
  c->npair = s->npair;
  c->nunpd = s->nunpd;
  c->ndocc = s->ndocc;
  c->ndf = s->ndf;
  c->norbs = s->norbs;
  c->totlen = s->totlen;
  c->nsp = 2 * s->npair + s->nunpd + s->ndocc;
  c->nalpha_rows = c->nsp;
  if (opt && opt->beta_only_last) {
    if (opt->beta_only_last != 1) return fail(VSVB_ERR_ARG, "beta_only_last must be 0 or 1");
    if (s->nunpd < 1 || s->ndocc < 1)
      return fail(VSVB_ERR_UNSUPPORTED, "beta_only_last needs nunpd >= 1 and ndocc >= 1");
    c->nalpha_rows = c->nsp - 1;
  }
  if (c->npair > 0) c->ndens = c->nsp * (c->nsp + 1) / 2;  // one Coulomb pass over the orbital-pair densities
  c->first_ndf = s->norbs - s->ndf;
  c->dtol = std::pow(10.0, -(double)s->ntol_d);
  if (c->nsp < 1) return fail(VSVB_ERR_ARG, "no electrons");
  // normalized primitive weights per type shell
  std::vector<double> con((size_t)s->nprim);
  for (int ts = 0; ts < s->nshell_type; ++ts) {
    const int p0 = s->shell_prim_start[ts], p1 = s->shell_prim_start[ts + 1];
    if (s->shell_l[ts] < 0 || s->shell_l[ts] > kLMax) return fail(VSVB_ERR_UNSUPPORTED, "only s, p and d shells");
    norm_prim(s->shell_l[ts], p1 - p0, s->prim_exp + p0, s->prim_coef + p0, con.data() + p0);
  }
  // global shells, per-shell primitive copies, AO map
  std::vector<int> shell_type, atom_sh0(s->natom + 1);
  int ao = 0;
  for (int a = 0; a < s->natom; ++a) {
    const int t = s->atom_type[a];
    if (t < 0 || t >= s->ntype) return fail(VSVB_ERR_ARG, "atom type out of range");
    atom_sh0[a] = (int)shells.size();
    for (int ts = s->type_shell_start[t]; ts < s->type_shell_start[t + 1]; ++ts) {
      Shell sh;
      sh.atom = a;
      sh.l = s->shell_l[ts];
      sh.nprim = s->shell_prim_start[ts + 1] - s->shell_prim_start[ts];
      sh.prim0 = (int)pexp.size();
      shell_type.push_back(ts);
      sh.ao = ao;
      for (int k = 0; k < sh.nprim; ++k) {
        pexp.push_back(s->prim_exp[s->shell_prim_start[ts] + k]);
        pcoef.push_back(con[s->shell_prim_start[ts] + k]);
      }
      for (int i = 0; i <= sh.l; ++i)
        for (int j = 0; j <= i; ++j) {
          angn.push_back(angn_of(sh.l - i, i - j, j));
          ao_shell.push_back((int)shells.size());
        }
      ao += ncart(sh.l);
      shells.push_back(sh);
    }
  }
  atom_sh0[s->natom] = (int)shells.size();
  c->nsh = (int)shells.size();
  c->nbf = ao;
  // shell pairs: class-major, by decreasing primitive-pair count
  struct HP { Pair p; int cls; double r2; };
  std::vector<HP> hp;
  for (int M = 0; M < c->nsh; ++M)
    for (int N = 0; N <= M; ++N) {
      HP h{};
      int A = M, B = N;
      if (shells[A].l < shells[B].l) std::swap(A, B);
      h.p.A = A;
      h.p.B = B;
      h.p.npp = shells[A].nprim * shells[B].nprim;
      h.cls = pair_class_of(shells[A].l, shells[B].l);
      const double* xa = s->coords + 3 * shells[A].atom;
      const double* xb = s->coords + 3 * shells[B].atom;
      h.r2 = (xa[0] - xb[0]) * (xa[0] - xb[0]) + (xa[1] - xb[1]) * (xa[1] - xb[1]) + (xa[2] - xb[2]) * (xa[2] - xb[2]);
      hp.push_back(h);
    }
  std::stable_sort(hp.begin(), hp.end(), [](const HP& x, const HP& y) {
    if (x.cls != y.cls) return x.cls < y.cls;
    if (x.p.npp != y.p.npp) return x.p.npp > y.p.npp;
    return x.r2 < y.r2;
  });
  std::vector<Pair> pairs(hp.size());
  c->npp = 0;
  for (size_t i = 0; i < hp.size(); ++i) {
    pairs[i] = hp[i].p;
    pairs[i].pp0 = c->npp;
    c->npp += pairs[i].npp;
  }
  for (int cl = 0; cl <= kNPairClass; ++cl) c->pair_off[cl] = 0;
  for (auto& h : hp) c->pair_off[h.cls + 1]++;
  for (int cl = 0; cl < kNPairClass; ++cl) c->pair_off[cl + 1] += c->pair_off[cl];
  c->npairs = (int)pairs.size();
  c->nfun = 0;
  for (int cl = 0; cl < kNPairClass; ++cl) {
    c->fun_off[cl] = c->nfun;
    for (int i = c->pair_off[cl]; i < c->pair_off[cl + 1]; ++i)
      c->nfun += ncart(shells[pairs[i].A].l) * ncart(shells[pairs[i].B].l);
  }
  c->h_pairs = pairs;
  // What a schedule needs of every shell pair: its class, its pair of atoms, and the
  // squared distances up to which its primitive pairs pass the screen, descending
  // (|K| > kPrimCut solved for the distance, once per pair of shell types).
  c->pair_cls.resize(pairs.size());
  c->pair_type.resize(pairs.size());
  c->prim_reach.resize((size_t)s->nshell_type * s->nshell_type);
  c->apair_start.assign((size_t)s->natom * (s->natom + 1) / 2 + 1, 0);
  std::vector<int> atoms(pairs.size());
  c->most_prims = 0;
  for (size_t i = 0; i < pairs.size(); ++i) {
    const Shell &A = shells[pairs[i].A], &B = shells[pairs[i].B];
    c->pair_cls[i] = hp[i].cls;
    c->pair_type[i] = shell_type[pairs[i].A] * s->nshell_type + shell_type[pairs[i].B];
    atoms[i] = std::max(A.atom, B.atom) * (std::max(A.atom, B.atom) + 1) / 2 + std::min(A.atom, B.atom);
    ++c->apair_start[atoms[i] + 1];
    c->most_prims = std::max(c->most_prims, pairs[i].npp);
    std::vector<double>& reach = c->prim_reach[c->pair_type[i]];
    if (!reach.empty()) continue;
    for (int ia = 0; ia < A.nprim; ++ia)
      for (int ib = 0; ib < B.nprim; ++ib) {
        const double x = pexp[A.prim0 + ia], y = pexp[B.prim0 + ib];
        const double K0 = std::fabs(pcoef[A.prim0 + ia] * pcoef[B.prim0 + ib]) / (x + y) * kPairFold;
        const double d2 = std::log(K0 / kPrimCut) * (x + y) / (x * y);
        reach.push_back(std::isnan(d2) ? 0.0 : d2);
      }
    std::sort(reach.begin(), reach.end(), std::greater<double>());
  }
  for (size_t k = 1; k < c->apair_start.size(); ++k) c->apair_start[k] += c->apair_start[k - 1];
  c->apair_ids.resize(pairs.size());
  {
    std::vector<int> next(c->apair_start);
    for (size_t i = 0; i < pairs.size(); ++i) c->apair_ids[next[atoms[i]]++] = (int)i;
  }
  // orbital entries: map each weight to an AO of the molecule (OBS-local numbering, xm_input)
  c->ent.resize(std::max(1, s->totlen));
  c->orb_start.assign(s->orb_start, s->orb_start + s->norbs + 1);
  for (int p = 0; p < s->norbs; ++p) {
    const int na = s->orb_natom[p];
    if (na < 1 || na > s->mxctr) return fail(VSVB_ERR_ARG, "orbital OBS atom count out of range");
    for (int k = s->orb_start[p]; k < s->orb_start[p + 1]; ++k) {
      OrbEntry e{p, 0, -1, 0};
      const int xp = s->xpset[k];
      if (xp < 1) {
        const int f = xp + s->norbs - 1;
        if (f < c->first_ndf || f >= s->norbs) return fail(VSVB_ERR_ARG, "NDF reference out of range");
        if (p >= c->first_ndf) return fail(VSVB_ERR_UNSUPPORTED, "an NDF expanded in other NDFs");
        e.kind = 1;
        e.tgt = f;
      } else {
        int kk = xp - 1;
        for (int ia = 0; ia < na; ++ia) {
          const int atom = s->orb_atoms[p * s->mxctr + ia];
          if (atom < 0 || atom >= s->natom) return fail(VSVB_ERR_ARG, "OBS atom out of range");
          const int a0 = shells[atom_sh0[atom]].ao;
          const int a1 = atom_sh0[atom + 1] < c->nsh ? shells[atom_sh0[atom + 1]].ao : c->nbf;
          if (kk < a1 - a0) {
            e.tgt = a0 + kk;
            break;
          }
          kk -= a1 - a0;
        }
        if (e.tgt < 0) return fail(VSVB_ERR_ARG, "AO index beyond the orbital's OBS");
      }
      c->ent[k] = e;
    }
  }
  // the orbitals that hold each AO (each once), for the entry-list orbital algebra
  c->ao_ptr.assign(c->nbf + 1, 0);
  if (c->ndf == 0) {
    std::vector<std::vector<int>> of(c->nbf);
    for (int p = 0; p < c->nsp; ++p)
      for (int k = s->orb_start[p]; k < s->orb_start[p + 1]; ++k) {
        auto& v = of[c->ent[k].tgt];
        if (v.empty() || v.back() != p) v.push_back(p);
      }
    for (int m = 0; m < c->nbf; ++m) {
      c->ao_ptr[m + 1] = c->ao_ptr[m] + (int)of[m].size();
      c->ao_orb.insert(c->ao_orb.end(), of[m].begin(), of[m].end());
    }
  }
  // host copies of inputs
  c->coords.assign(s->coords, s->coords + 3 * s->natom);
  c->charges.resize(s->natom);
  for (int a = 0; a < s->natom; ++a) c->charges[a] = s->nuc_charge[s->atom_type[a]];
  c->coeff.assign(s->coeff, s->coeff + s->totlen);
  return VSVB_OK;
}

// Work lists and counters of a context of c->ncu CUs; the length of its segment lists.
static size_t plan_lists(vsvb_context* c) {
  // work lists: the shell pairs, and for systems of up to kSplitMaxPairs pairs
  // their segments (counts here for unscreened primitive lists, the most a
  // geometry can give)
  size_t seg_cap = 0;
  for (int pc = 0; pc < kNPairClass; ++pc) {
    WorkList& W0 = c->work[pc][0];
    W0.off = c->pair_off[pc];
    W0.n = W0.cap = c->pair_off[pc + 1] - c->pair_off[pc];
    for (int l = 1; l < kLevels; ++l) {
      WorkList& W = c->work[pc][l];
      W.cap = 0;
      for (int i = c->pair_off[pc]; i < c->pair_off[pc + 1]; ++i)
        W.cap += std::max(1, (c->h_pairs[i].npp + kSegLen[l][pc] - 1) / kSegLen[l][pc]);
      seg_cap += W.cap;
    }
  }
  // work counters: per part one per energy segment of kSegTiles bra tiles and one
  // per J/K strip (bra strips, or ket strips transposed); one for the cooperative kernel
  static_assert(kSegTiles * kTileB == kStripB, "an energy segment covers one bra strip");
  const bool split = c->npairs <= kSplitMaxPairs;
  c->ctr_total = 0;
  for (int bc = 0, q = 0; bc < kNPairClass; ++bc)
    for (int kc = 0; kc <= bc; ++kc, ++q) {
      int most = 1;
      for (int l = 0; l < (split ? kLevels : 1); ++l)
        most = std::max({most, (c->work[bc][l].cap + kStripB - 1) / kStripB, (c->work[kc][l].cap + kStripK - 1) / kStripK});
      c->ctr_off[q] = c->ctr_total;
      c->ctr_len[q] = most * std::max(kPartsEnergy[q], kPartsJk[q]);
      c->ctr_total += c->ctr_len[q];
      c->coop_idx[q] = coop_class(kPairLs[bc][0], kPairLs[bc][1], kPairLs[kc][0], kPairLs[kc][1]);
    }
  return split ? seg_cap : 0;
}

// Doubles of d_partial: what an energy at any geometry writes, four per workgroup
// and part of a class.  The longest lists give the largest grids, up to the class's
// limit (chunks of several kets are fewer units).  Fock tiles leave their shares of
// E2 there too, at most 20 x 20 per spin; the allocation-free entry, J/K only, has
// no energy launches.
static size_t partial_slots(const vsvb_context* c) {
  size_t slots = 0;
  for (int bc = 0, q = 0; bc < kNPairClass && !c->arena; ++bc)
    for (int kc = 0; kc <= bc; ++kc, ++q) {
      size_t nb = 0, nk = 0;
      for (int l = 0; l < (c->npairs <= kSplitMaxPairs ? kLevels : 1); ++l) {
        nb = std::max<size_t>(nb, c->work[bc][l].cap);
        nk = std::max<size_t>(nk, c->work[kc][l].cap);
      }
      if (nb == 0 || nk == 0) continue;
      const size_t nbt = (nb + kTileB - 1) / kTileB;
      if (c->coop_idx[q] >= 0)
        slots += 4 * std::min(nb * nk, (size_t)coop_occupancy(c->coop_idx[q], false) * c->ncu);
      else
        slots += 4 * class_parts(q, false) *
                 std::min(((bc == kc ? kTileB / 2 * nbt * (nbt + 1) : nbt * nk) + 3) / 4, (size_t)energy_grid(c, bc, kc));
    }
  return std::max<size_t>(slots, 1024);
}

static int build_context(const vsvb_system* s, const vsvb_options* opt, vsvb_context* c) {
  int rc;
  if ((rc = read_options(s, opt, c))) return rc;
  HIP_OK(hipSetDevice(c->device));
  HIP_OK(hipDeviceGetAttribute(&c->wall_khz, hipDeviceAttributeWallClockRate, c->device));
  if (!c->arena) {  // the allocation-free entry creates no stream or events: it runs on the null stream
    if (!c->stream) HIP_OK(hipStreamCreateWithFlags(&c->stream, hipStreamNonBlocking));
    HIP_OK(hipEventCreate(&c->ev0));
    HIP_OK(hipEventCreate(&c->ev1));
    HIP_OK(hipEventCreateWithFlags(&c->ev_in, hipEventDisableTiming));
    HIP_OK(hipEventCreateWithFlags(&c->ev_out, hipEventDisableTiming));
  }
  HostBasis hb;
  if ((rc = describe_system(s, opt, c, hb))) return rc;
  const std::vector<Shell>& shells = hb.shells;
  const std::vector<double>&pexp = hb.pexp, &pcoef = hb.pcoef, &angn = hb.angn;
  const std::vector<int>& ao_shell = hb.ao_shell;
  const std::vector<Pair>& pairs = c->h_pairs;
  // device allocations (all of them, here)
  const size_t nbf2 = (size_t)c->nbf * c->nbf;
  HIP_OK(device_buffer(c, c->d_shells, c->nsh));
  HIP_OK(device_buffer(c, c->d_pairs, c->npairs));
  HIP_OK(device_buffer(c, c->d_psrc, c->npairs));
  HIP_OK(device_buffer(c, c->d_order, c->npairs));
  HIP_OK(device_buffer(c, c->d_pp, c->npp));
  HIP_OK(device_buffer(c, c->d_pexp, pexp.size()));
  HIP_OK(device_buffer(c, c->d_pcoef, pcoef.size()));
  HIP_OK(device_buffer(c, c->d_xyz, 3 * c->natom));
  HIP_OK(device_buffer(c, c->d_charge, c->natom));
  HIP_OK(device_buffer(c, c->d_boys, kBoysCOff + (size_t)(kLTot + 1) * kBoysCLen));
  HIP_OK(device_buffer(c, c->d_angn, c->nbf));
  HIP_OK(device_buffer(c, c->d_ao_shell, c->nbf));
  HIP_OK(device_buffer(c, c->d_orb_start, s->norbs + 1));
  HIP_OK(device_buffer(c, c->d_colk, std::max(1, c->nsp)));
  HIP_OK(device_buffer(c, c->d_ent, c->ent.size()));
  HIP_OK(device_buffer(c, c->d_coeff, std::max(1, s->totlen)));
  HIP_OK(device_buffer(c, c->d_ndf_scale, std::max(1, s->ndf)));
  HIP_OK(device_buffer(c, c->d_ndf_d, s->ndf > 0 ? (size_t)s->ndf * c->nbf : 1));
  HIP_OK(device_buffer(c, c->d_ndf_g, s->ndf > 0 ? (size_t)s->ndf * c->nbf : 1));
  HIP_OK(device_buffer(c, c->d_S, nbf2));
  HIP_OK(device_buffer(c, c->d_H, nbf2));
  HIP_OK(device_buffer(c, c->d_Ct, (size_t)c->nsp * c->nbf));
  HIP_OK(device_buffer(c, c->d_Cs, (size_t)c->nsp * c->nbf));
  HIP_OK(device_buffer(c, c->d_Sorb, (size_t)c->nsp * c->nsp));
  HIP_OK(device_buffer(c, c->d_Horb, (size_t)c->nsp * c->nsp));
  HIP_OK(device_buffer(c, c->d_P, 2 * (size_t)c->nsp * c->nsp));
  HIP_OK(device_buffer(c, c->d_R, 2 * nbf2));
  HIP_OK(device_buffer(c, c->d_tmp, std::max(nbf2, (size_t)c->nsp * c->nbf)));
  HIP_OK(device_buffer(c, c->d_tmp2, std::max(nbf2, (size_t)c->nsp * c->nbf)));
  HIP_OK(device_buffer(c, c->d_J, nbf2));
  HIP_OK(device_buffer(c, c->d_K, 2 * nbf2));
  HIP_OK(device_buffer(c, c->d_F, 2 * nbf2));
  HIP_OK(device_buffer(c, c->d_gradC, (size_t)c->nsp * c->nbf));
  HIP_OK(device_buffer(c, c->d_Jsym, nbf2));
  HIP_OK(device_buffer(c, c->d_Rfull, nbf2));
  HIP_OK(device_buffer(c, c->d_X, (size_t)c->nsp * c->nbf));
  HIP_OK(device_buffer(c, c->d_Z, (size_t)c->nsp * c->nbf));
  // what a call reads back stands in one block: one copy instead of four, each
  // some 10 us of a water energy's 220
  HIP_OK(device_buffer(c, c->d_out, kOutGrad + std::max(1, s->totlen)));
  c->d_scal.alias(reinterpret_cast<double*>(c->d_out.p), 16);
  c->d_status.alias(reinterpret_cast<int*>(c->d_out.p + kOutStatus), 4);
  c->d_counters.alias(c->d_out.p + kOutCounters, kCounterWords);
  c->d_grad.alias(reinterpret_cast<double*>(c->d_out.p + kOutGrad), std::max(1, s->totlen));
  HIP_OK(device_buffer(c, c->d_stamps, (size_t)2 * kStampSlots * kNQuartetClass));
  // quartet launch geometry (grids sized to the occupancy of each class kernel) and partial buffer
  int ncu = 0;
  HIP_OK(hipDeviceGetAttribute(&ncu, hipDeviceAttributeMultiprocessorCount, c->device));
  c->ncu = ncu;
  const size_t seg_cap = plan_lists(c);
  HIP_OK(device_buffer(c, c->d_tilectr, c->ctr_total));
  HIP_OK(coop_prepare(c->device));
  HIP_OK(device_buffer(c, c->d_partial, partial_slots(c)));
  // segment lists last: in the allocation-free entry they are left out where
  // the static array has no room for them
  const size_t seg_bytes = seg_cap * (sizeof(Pair) + sizeof(SegSrc)) + 2 * kNQuartetClass * sizeof(QuartetArgs) + 1024;
  if (seg_cap > 0 && (!c->arena || c->arena->used + seg_bytes <= c->arena->cap)) {
    HIP_OK(device_buffer(c, c->d_split, seg_cap));
    HIP_OK(device_buffer(c, c->d_segsrc, seg_cap));
    HIP_OK(device_buffer(c, c->d_small, 2 * kNQuartetClass));
    c->nlevels = kLevels;
  }
  const size_t list_bytes = (c->ao_ptr.size() + c->ao_orb.size()) * sizeof(int) + 1024;
  if (entry_list_orbitals(c) && (!c->arena || c->arena->used + list_bytes <= c->arena->cap)) {
    HIP_OK(device_buffer(c, c->d_ao_ptr, c->ao_ptr.size()));
    HIP_OK(device_buffer(c, c->d_ao_orb, c->ao_orb.size()));
    HIP_OK(hipMemcpy(c->d_ao_ptr.p, c->ao_ptr.data(), c->ao_ptr.size() * sizeof(int), hipMemcpyHostToDevice));
    if (!c->ao_orb.empty())
      HIP_OK(hipMemcpy(c->d_ao_orb.p, c->ao_orb.data(), c->ao_orb.size() * sizeof(int), hipMemcpyHostToDevice));
  }
  if ((rc = plan_work(c, nullptr))) return rc;
  // uploads
  static const std::vector<double> boys = make_boys_table();  // the same in every context
  HIP_OK(hipMemcpy(c->d_shells.p, shells.data(), shells.size() * sizeof(Shell), hipMemcpyHostToDevice));
  {
    std::vector<PairSrc> src;
    for (const Pair& P : pairs) src.push_back(PairSrc{P.A, P.B, P.pp0});
    HIP_OK(hipMemcpy(c->d_psrc.p, src.data(), src.size() * sizeof(PairSrc), hipMemcpyHostToDevice));
  }
  HIP_OK(hipMemcpy(c->d_pexp.p, pexp.data(), pexp.size() * sizeof(double), hipMemcpyHostToDevice));
  HIP_OK(hipMemcpy(c->d_pcoef.p, pcoef.data(), pcoef.size() * sizeof(double), hipMemcpyHostToDevice));
  HIP_OK(hipMemcpy(c->d_charge.p, c->charges.data(), c->natom * sizeof(double), hipMemcpyHostToDevice));
  HIP_OK(hipMemcpy(c->d_boys.p, boys.data(), boys.size() * sizeof(double), hipMemcpyHostToDevice));
  HIP_OK(hipMemcpy(c->d_angn.p, angn.data(), angn.size() * sizeof(double), hipMemcpyHostToDevice));
  HIP_OK(hipMemcpy(c->d_ao_shell.p, ao_shell.data(), ao_shell.size() * sizeof(int), hipMemcpyHostToDevice));
  HIP_OK(hipMemcpy(c->d_orb_start.p, c->orb_start.data(), c->orb_start.size() * sizeof(int), hipMemcpyHostToDevice));
  HIP_OK(hipMemcpy(c->d_ent.p, c->ent.data(), c->ent.size() * sizeof(OrbEntry), hipMemcpyHostToDevice));
  HIP_OK(hipMemcpy(c->d_coeff.p, c->coeff.data(), c->totlen * sizeof(double), hipMemcpyHostToDevice));
  if (s->npair > 0) return sc_setup(c, s);
  return VSVB_OK;
}

// geometry-dependent device state
// Work order of the shell pairs at one geometry: inside each class, by the
// number of primitive pairs that survive the primitive screen (descending),
// then by centre distance, so that the 64 lanes of a wavefront run primitive
// loops of nearly equal length and Schwarz-skipped quartets cluster.  The
// order is a schedule only (every unique quartet is still evaluated once); it
// is recomputed when the coordinates change.
static int order_pairs(vsvb_context* c) {
  const int np = c->npairs, nap = c->natom * (c->natom + 1) / 2;
  // Shell pairs of one pair of atoms share the distance: the atom pairs are sorted,
  // and every shell pair goes to the next place of its (class, count) in that order.
  std::vector<std::pair<double, int>> ap(nap);
  for (int i = 0, k = 0; i < c->natom; ++i)
    for (int j = 0; j <= i; ++j, ++k) {
      const double *xa = c->coords.data() + 3 * i, *xb = c->coords.data() + 3 * j;
      ap[k] = {(xa[0] - xb[0]) * (xa[0] - xb[0]) + (xa[1] - xb[1]) * (xa[1] - xb[1]) + (xa[2] - xb[2]) * (xa[2] - xb[2]),
               k};
    }
  std::stable_sort(ap.begin(), ap.end(), [](const auto& x, const auto& y) { return x.first < y.first; });
  const int nk = c->most_prims + 1;
  std::vector<int> kept(np), start((size_t)kNPairClass * nk + 1, 0), skept(np);
  auto cell = [&](int i) { return c->pair_cls[i] * nk + (nk - 1 - kept[i]); };  // class, then most primitive pairs first
  for (const auto& x : ap)
    for (int e = c->apair_start[x.second]; e < c->apair_start[x.second + 1]; ++e) {
      const int i = c->apair_ids[e];
      const std::vector<double>& lim = c->prim_reach[c->pair_type[i]];
      kept[i] = (int)(std::lower_bound(lim.begin(), lim.end(), x.first, std::greater<double>()) - lim.begin());
      ++start[cell(i) + 1];
    }
  for (size_t k = 1; k < start.size(); ++k) start[k] += start[k - 1];
  c->h_order.resize(np);
  for (const auto& x : ap)
    for (int e = c->apair_start[x.second]; e < c->apair_start[x.second + 1]; ++e) {
      const int i = c->apair_ids[e], at = start[cell(i)]++;
      c->h_order[at] = i;
      skept[at] = kept[i];
    }
  return plan_work(c, skept.data());
}

static int schedule_pairs(vsvb_context* c) {
  if (c->sched_coords == c->coords) return VSVB_OK;
  const int rc = order_pairs(c);
  if (rc) return rc;
  HIP_OK(hipMemcpyAsync(c->d_order.p, c->h_order.data(), c->npairs * sizeof(int), hipMemcpyHostToDevice, c->stream));
  if (!c->h_seg.empty())
    HIP_OK(hipMemcpyAsync(c->d_segsrc.p, c->h_seg.data(), c->h_seg.size() * sizeof(SegSrc), hipMemcpyHostToDevice,
                          c->stream));
  c->sched_coords = c->coords;
  return VSVB_OK;
}

int vsvb::prepare_geometry(vsvb_context* c, const double* coords) {
  if (coords) c->coords.assign(coords, coords + 3 * c->natom);
  if (c->geom_ready && !coords) return VSVB_OK;
  hipStream_t st = c->stream;
  int rc;
  if ((rc = schedule_pairs(c))) return rc;
  c->enuc = nuclear_repulsion(c->natom, c->coords.data(), c->charges.data());
  if (!c->capturing)
    HIP_OK(hipMemcpyAsync(c->d_xyz.p, c->coords.data(), 3 * c->natom * sizeof(double), hipMemcpyHostToDevice, st));
  PairArgs a{c->d_psrc.p,  c->d_order.p,  c->d_pairs.p, c->d_shells.p, c->d_pexp.p, c->d_pcoef.p, c->d_xyz.p,
             c->d_charge.p, c->d_boys.p,  c->d_pp.p,    c->d_S.p,      c->d_H.p,    kPairFold,    c->natom,
             c->nbf,        {},           {}};
  std::copy(c->pair_off, c->pair_off + kNPairClass + 1, a.off);
  std::copy(c->fun_off, c->fun_off + kNPairClass, a.fun);
  HIP_OK(launch_pairs(a, st));
  if (!c->h_seg.empty()) {
    const int ns = (int)c->h_seg.size();
    hipLaunchKernelGGL(k_split, dim3((ns + 255) / 256), dim3(256), 0, st, c->d_pairs.p, c->d_segsrc.p, ns, c->d_split.p);
    HIP_OK(hipGetLastError());
  }
  c->geom_ready = true;
  return VSVB_OK;
}

// New weights (from the host or the device) into d_coeff.
static int upload_coeff(vsvb_context* c, const double* coeff_host, const double* coeff_dev) {
  if (coeff_host) {
    c->coeff.assign(coeff_host, coeff_host + c->totlen);
    HIP_OK(hipMemcpyAsync(c->d_coeff.p, c->coeff.data(), c->totlen * sizeof(double), hipMemcpyHostToDevice, c->stream));
  } else if (coeff_dev) {
    HIP_OK(hipMemcpyAsync(c->d_coeff.p, coeff_dev, c->totlen * sizeof(double), hipMemcpyDeviceToDevice, c->stream));
  }
  return VSVB_OK;
}

// weights -> Ct, Cs, orbital S and h, P per spin block, R per spin block, E1.
// Spin blocks (npair = 0): alpha = all spatial orbitals (unpaired then docc),
// beta = the trailing ndocc (docc); closed shell when nunpd = 0.
int vsvb::prepare_orbital_basis(vsvb_context* c, const double* coeff_host, const double* coeff_dev) {
  hipStream_t st = c->stream;
  const int rc = upload_coeff(c, coeff_host, coeff_dev);
  if (rc) return rc;
  const int n = c->nbf, ns = c->nsp;
  hipLaunchKernelGGL(k_fill, dim3(1), dim3(64), 0, st, c->d_scal.p, (size_t)16, 0.0);
  HIP_OK(launch_zero(st, c->d_status.p, 4 * sizeof(int)));
  if (c->ndf > 0) {
    hipLaunchKernelGGL(k_ndf_scale, dim3((c->ndf + 63) / 64), dim3(64), 0, st, c->d_ent.p, c->d_orb_start.p,
                       c->d_coeff.p, c->d_angn.p, c->d_S.p, n, c->first_ndf, c->ndf, c->d_ndf_scale.p);
    HIP_OK(hipGetLastError());
  }
  hipLaunchKernelGGL(k_fill, dim3(256), dim3(256), 0, st, c->d_Ct.p, (size_t)ns * n, 0.0);
  hipLaunchKernelGGL(k_build_orbitals, dim3((ns + 63) / 64), dim3(64), 0, st, c->d_ent.p, c->d_orb_start.p,
                     c->d_coeff.p, c->d_angn.p, c->d_ndf_scale.p, c->first_ndf, n, ns, c->d_Ct.p);
  HIP_OK(hipGetLastError());
  // S_orb = Ct S Ct^T, h_orb = Ct H Ct^T
  HIP_OK(gemm(st, ns, n, n, 1.0, c->d_Ct.p, n, false, c->d_S.p, n, false, 0.0, c->d_tmp.p, n));
  HIP_OK(gemm(st, ns, ns, n, 1.0, c->d_tmp.p, n, false, c->d_Ct.p, n, true, 0.0, c->d_Sorb.p, ns));
  HIP_OK(gemm(st, ns, n, n, 1.0, c->d_Ct.p, n, false, c->d_H.p, n, false, 0.0, c->d_tmp.p, n));
  HIP_OK(gemm(st, ns, ns, n, 1.0, c->d_tmp.p, n, false, c->d_Ct.p, n, true, 0.0, c->d_Horb.p, ns));
  {
    const long nt = (long)ns * c->nsh;
    hipLaunchKernelGGL(k_shell_screen, dim3((unsigned)((nt + 255) / 256)), dim3(256), 0, st, c->d_Ct.p, c->d_Sorb.p,
                       ns, c->d_shells.p, c->nsh, c->d_angn.p, n, c->dtol, c->d_Cs.p, c->d_status.p + 1);
    HIP_OK(hipGetLastError());
  }
  return VSVB_OK;
}

// What the quartet pass (1: energy, 2: J/K into jacc, kacc) needs cleared.
static ZeroArgs pass_zero(vsvb_context* c, int pass, int nwfn, double* jacc, double* kacc) {
  ZeroArgs z;
  if (pass <= 0) return z;
  const size_t nn = (size_t)c->nbf * c->nbf, words = sizeof(double) / sizeof(uint32_t);
  z.p[0] = reinterpret_cast<uint32_t*>(c->d_counters.p);
  z.n[0] = kCtrSlots * kCtrStride * sizeof(unsigned long long) / sizeof(uint32_t);
  z.p[1] = reinterpret_cast<uint32_t*>(c->d_tilectr.p);
  z.n[1] = c->ctr_total;
  if (pass == 2) {
    z.p[2] = reinterpret_cast<uint32_t*>(jacc);
    z.n[2] = nwfn * nn * words;
    z.p[3] = reinterpret_cast<uint32_t*>(kacc);
    z.n[3] = nwfn * (c->nunpd > 0 ? 2 : 1) * nn * words;
  }
  return z;
}

// Orbital stage of one wave function; pass: the quartet pass that follows (1
// energy, 2 J/K of this wave function alone, 0 neither), cleared along by the
// entry-list algebra.
static int prepare_orbitals(vsvb_context* c, const double* coeff_host, const double* coeff_dev, int pass) {
  int rc;
  c->cleared = 0;
  if (c->d_ao_ptr.p) {
    if ((rc = upload_coeff(c, coeff_host, coeff_dev))) return rc;
    HIP_OK(launch_orbital_front(c->stream, orb_args(c), nullptr, 1, pass_zero(c, pass, 1, c->d_J.p, c->d_K.p)));
    c->cleared = pass;
    return VSVB_OK;
  }
  if ((rc = prepare_orbital_basis(c, coeff_host, coeff_dev))) return rc;
  hipStream_t st = c->stream;
  const int n = c->nbf, ns = c->nsp;
  const int nspin = c->nunpd > 0 ? 2 : 1;
  for (int s = 0; s < nspin; ++s) {
    const int off = s == 0 ? 0 : c->nunpd;
    const int m = s == 0 ? c->nalpha_rows : c->ndocc;
    double* P = c->d_P.p + (size_t)s * ns * ns;
    if (m == 0) continue;
    hipLaunchKernelGGL(k_copy_block, dim3((m * m + 255) / 256), dim3(256), 0, st, c->d_Sorb.p, ns, off, m, P);
    HIP_OK(launch_spd_inverse(st, P, m, c->d_status.p, c->d_colk.p, c->grid_inverse_min));
    // E1 += w tr(h_s P_s): closed shell counts both spins (w = 2)
    hipLaunchKernelGGL(k_trace_prod, dim3(trace_blocks(m)), dim3(256), 0, st, c->d_Horb.p, ns, off, P, m, nspin == 1 ? 2.0 : 1.0,
                       c->d_scal.p + 0);
    // R_s = Cs_s^T P_s Cs_s
    const double* Cs = c->d_Cs.p + (size_t)off * n;
    HIP_OK(gemm(st, m, n, m, 1.0, P, m, false, Cs, n, false, 0.0, c->d_tmp.p, n));
    HIP_OK(gemm(st, n, n, m, 1.0, Cs, n, true, c->d_tmp.p, n, false, 0.0, c->d_R.p + (size_t)s * n * n, n));
  }
  if (nspin == 2 && c->ndocc == 0) {
    hipLaunchKernelGGL(k_fill, dim3(256), dim3(256), 0, st, c->d_R.p + (size_t)n * n, (size_t)n * n, 0.0);
  }
  return VSVB_OK;
}

// Shell-quartet stage.  By default it serves this context's own wave function;
// a batch group leader passes nwfn > 1 and group-wide density and J/K arrays.
static QuartetArgs class_args(vsvb_context* c, int bc, int kc, const ClassLaunch& cl, bool jk, int nwfn, int nspin,
                              const double* dens, double* jacc, double* kacc, double* partial, double* eri = nullptr) {
  const int q = quartet_class_index(bc, kc);
  QuartetArgs a{};
  const WorkList &B = c->work[bc][cl.lb], &K = c->work[kc][cl.lk];
  a.bra = (cl.lb ? c->d_split.p : c->d_pairs.p) + B.off;
  a.ket = (cl.lk ? c->d_split.p : c->d_pairs.p) + K.off;
  a.nbra = B.n;
  a.nket = K.n;
  a.pp = c->d_pp.p;
  a.shells = c->d_shells.p;
  a.boys = c->d_boys.p;
  a.same = bc == kc;
  a.ntk = cl.claim;
  a.ntiles = cl.units;
  a.kchunk = cl.coop ? 1 : cl.kchunk;
  a.nkc = (a.nket + a.kchunk - 1) / a.kchunk;
  a.lds_k = jk && cl.lds > 0;
  a.tau = c->tau;
  a.nbf = c->nbf;
  a.nwfn = nwfn;
  a.nspin = nspin;
  a.dens = dens;
  a.partial = partial;
  a.jacc = jacc;
  a.kacc = kacc;
  a.eri = eri;
  a.neri = c->nfun;
  a.fbra = c->pair_off[bc + 1] - c->pair_off[bc];
  a.fket = c->pair_off[kc + 1] - c->pair_off[kc];
  a.counters = c->d_counters.p + 4 * q;
  a.stamp = c->profile ? c->d_stamps.p + (size_t)q * 2 * kStampSlots : nullptr;
  a.tile_ctr = c->d_tilectr.p + c->ctr_off[q];
  a.nstrip = cl.coop ? 1 : cl.strips;
  a.shift = cl.shift;
  return a;
}

static hipError_t launch_class(vsvb_context* c, int bc, int kc, const ClassLaunch& cl, const QuartetArgs& a, bool jk) {
  const int q = quartet_class_index(bc, kc);
  if (cl.coop) return launch_coop(c->coop_idx[q], a, jk, cl.blocks, c->device, c->stream);
  return launch_quartet_class(bc, kc, a, jk, cl.tr, cl.blocks, cl.lds, c->stream);
}

// Before a quartet pass: the first `words` counter words (quartets, primitive
// quartets, skips per class; all words also clear the timing results), the
// work counters and, in J/K mode, the accumulators.
static hipError_t quartet_pass_clear(vsvb_context* c, bool jk, int nwfn, int nspin, double* jacc, double* kacc,
                                     int words) {
  hipStream_t st = c->stream;
  const size_t nn = (size_t)c->nbf * c->nbf;
  hipError_t e = hipSuccess;
  const int cleared = c->cleared;
  c->cleared = 0;
  c->last_jk = jk;
  c->last_nwfn = nwfn;
  c->last_nspin = nspin;
  c->ran_quartets = true;
  c->ev_valid = false;
  if (cleared == (jk ? 2 : 1) && words == kCtrSlots * kCtrStride) return e;
  if ((e = launch_zero(st, c->d_counters.p, words * sizeof(unsigned long long))) != hipSuccess) return e;
  if ((e = launch_zero(st, c->d_tilectr.p, c->ctr_total * sizeof(int))) != hipSuccess) return e;
  if (jk) {
    hipLaunchKernelGGL(k_fill, dim3(1024), dim3(256), 0, st, jacc, nwfn * nn, 0.0);
    hipLaunchKernelGGL(k_fill, dim3(1024), dim3(256), 0, st, kacc, nwfn * nspin * nn, 0.0);
  }
  return hipGetLastError();
}

// nspin_override = 0 turns the J/K launch into a Coulomb-only pass over nwfn
// general symmetric densities (the exchange accumulators are not touched).  eri
// (nfun x nfun, zeroed by the caller): an energy pass stores its integrals there
// instead of contracting them (QuartetArgs::eri).
int vsvb::run_quartets(vsvb_context* c, bool jk, int nwfn, const double* dens, double* jacc,
                       double* kacc, int nspin_override, double* eri) {
  hipStream_t st = c->stream;
  const int nspin = nspin_override >= 0 ? nspin_override : (c->nunpd > 0 ? 2 : 1);
  if (!dens) dens = c->d_R.p;
  if (!jacc) jacc = c->d_J.p;
  if (!kacc) kacc = c->d_K.p;
  HIP_OK(quartet_pass_clear(c, jk, nwfn, nspin, jacc, kacc, kCtrSlots * kCtrStride));
  // Stage timing: HIP events on direct runs (under stream capture a record is
  // only a dependency, so replays take the per-class wall-clock stamps the
  // kernels write when profiling is on).
  const int nslot = 2 * kStampSlots * kNQuartetClass;
  if (c->profile) hipLaunchKernelGGL(k_stamp_reset, dim3((nslot + 255) / 256), dim3(256), 0, st, c->d_stamps.p, nslot);
  if (c->ev0 && !c->capturing) HIP_OK(hipEventRecord(c->ev0, st));
  // Classes in class order, or reversed (c->class_rev); each class's partial
  // sums keep their own offset either way.
  size_t offs[kNQuartetClass], poff = 0;
  for (int q = 0; q < kNQuartetClass; ++q) {
    offs[q] = poff;
    poff += c->partial_per_class[q];
  }
  if (!jk && !eri && poff > c->d_partial.n)
    return fail(VSVB_ERR_UNSUPPORTED, "the energy's partial sums do not fit their buffer");
  const int m = jk ? 1 : 0;
  // Two cooperative classes whose wavefronts all fit the chip at once share a
  // launch: each runs as long as its longest quartet (water: 2 x 36 us one after the
  // other, 46 side by side).  A forced chunk width keeps a launch per class.
  int pair[2] = {-1, -1};
  struct Join {  // on every return path
    hipStream_t st = nullptr;
    hipEvent_t ev = nullptr;
    ~Join() {
      if (ev) (void)hipStreamWaitEvent(st, ev, 0);
    }
  } join;
  bool forked = false;
  {
    int k = 0, blocks = 0, fit = 0;
    for (int q = kNQuartetClass - 1; q >= 0 && k < 2; --q) {
      const ClassLaunch& cl = jk ? c->ljk[q] : c->le[q];
      if (!cl.coop || cl.units <= 0) continue;
      pair[k] = q;
      blocks += cl.blocks;
      fit = k == 0 ? coop_occupancy(c->coop_idx[q], jk) : std::min(fit, coop_occupancy(c->coop_idx[q], jk));
      ++k;
    }
    if (k < 2 || blocks > fit * c->ncu || c->pair_chunk > 0) pair[0] = pair[1] = -1;
  }
  if (pair[0] >= 0) {
    QuartetArgs a[2];
    for (int k = 0; k < 2; ++k) {
      const int q = pair[k], bc = class_bra(q), kc = q - quartet_class_index(bc, 0);
      a[k] = class_args(c, bc, kc, jk ? c->ljk[q] : c->le[q], jk, nwfn, nspin, dens, jacc, kacc, c->d_partial.p + offs[q],
                        eri);
    }
    // beside the shared launch, on a stream of its own: both are chains on a mostly
    // idle chip (a water energy 169 us in one stream, 152 so; batches have their own
    // streams and graphs)
    if (c->small[m].n > 0 && c->own_stream && !c->capturing) {
      if (!c->side) {
        HIP_OK(hipEventCreateWithFlags(&c->ev_fork, hipEventDisableTiming));
        HIP_OK(hipEventCreateWithFlags(&c->ev_join, hipEventDisableTiming));
        HIP_OK(hipStreamCreateWithFlags(&c->side, hipStreamNonBlocking));
      }
      HIP_OK(hipEventRecord(c->ev_fork, st));
      HIP_OK(hipStreamWaitEvent(c->side, c->ev_fork, 0));
      forked = true;
    }
    const ClassLaunch* l = jk ? c->ljk : c->le;
    HIP_OK(launch_coop_pair(c->coop_idx[pair[0]], a[0], l[pair[0]].blocks, c->coop_idx[pair[1]], a[1],
                            l[pair[1]].blocks, jk, c->device, forked ? c->side : st));
    if (forked) {
      HIP_OK(hipEventRecord(c->ev_join, c->side));
      join.st = st;
      join.ev = c->ev_join;
    }
  }
  // Small classes share one launch: their argument records go to the device when
  // they differ from the last ones (under capture nothing is uploaded; records
  // that differ then take separate launches).
  bool shared = c->small[m].n > 0 && (nwfn == 1 || eri);
  if (shared) {
    const SmallLaunch& s = c->small[m];
    std::vector<QuartetArgs> rec(s.n);
    for (int k = 0; k < s.n; ++k) {
      const int q = s.q[k], bc = class_bra(q), kc = q - quartet_class_index(bc, 0);
      rec[k] = class_args(c, bc, kc, jk ? c->ljk[q] : c->le[q], jk, nwfn, nspin, dens, jacc, kacc,
                          c->d_partial.p + offs[q], eri);
    }
    std::vector<QuartetArgs>& old = c->h_small[m];
    QuartetArgs* dev = c->d_small.p + (size_t)m * kNQuartetClass;
    if (old.size() != rec.size() || std::memcmp(old.data(), rec.data(), rec.size() * sizeof(QuartetArgs)) != 0) {
      if (c->capturing) {
        shared = false;
      } else {
        old.swap(rec);
        HIP_OK(hipMemcpyAsync(dev, old.data(), old.size() * sizeof(QuartetArgs), hipMemcpyHostToDevice, st));
      }
    }
    if (shared) HIP_OK(launch_small(s, dev, jk, st));
  }
  for (int t = 0; t < kNQuartetClass; ++t) {
    const int q = c->class_rev ? kNQuartetClass - 1 - t : t;
    if ((shared && c->in_small[m][q]) || q == pair[0] || q == pair[1]) continue;
    const int bc = class_bra(q), kc = q - quartet_class_index(bc, 0);
    const ClassLaunch& cl = jk ? c->ljk[q] : c->le[q];
    const int nb = c->work[bc][0].n, nk = c->work[kc][0].n;
    // a class with pairs on both sides always has work units: a launch
    // configuration without any would drop its quartets silently
    if (nb > 0 && nk > 0 && cl.units <= 0)
      return fail(VSVB_ERR_UNSUPPORTED, "quartet class " + std::to_string(q) + " has no launchable work units");
    const QuartetArgs a = class_args(c, bc, kc, cl, jk, nwfn, nspin, dens, jacc, kacc, c->d_partial.p + offs[q],
                                     eri);
    HIP_OK(launch_class(c, bc, kc, cl, a, jk));
  }
  if (forked) {
    join.ev = nullptr;
    HIP_OK(hipStreamWaitEvent(st, c->ev_join, 0));
  }
  if (c->ev0 && c->ev1 && !c->capturing) {
    HIP_OK(hipEventRecord(c->ev1, st));
    c->ev_valid = true;
  }
  if (c->profile)
    hipLaunchKernelGGL(k_stamp_reduce, dim3(kNQuartetClass), dim3(kStampSlots), 0, st, c->d_stamps.p,
                       c->d_counters.p + kCtrSlots * kCtrStride);
  if (!jk && !eri) HIP_OK(launch_energy_sum(st, c->d_partial.p, (long)poff, c->enuc, c->d_scal.p));
  return VSVB_OK;
}

// Counters of the last quartet stage.  Class times come from the kernels'
// wall-clock stamps (profiling on); the stage time from the HIP events of a direct
// run, or, after a graph replay (whose events were not recorded), from the stamps'
// overall span.
int vsvb::finish_counters(vsvb_context* c) {
  unsigned long long h[kStatWords];
  const unsigned long long *n = c->h_out.data() + kOutCounters, *stamp = n + kCtrSlots * kCtrStride;
  std::copy(n, n + kCtrStride, h);
  for (int s = 1; s < kCtrSlots; ++s)
    for (int k = 0; k < kCtrStride; ++k) h[k] += n[s * kCtrStride + k];
  std::copy(stamp, stamp + 2 * kNQuartetClass, h + kCtrStride);
  return finish_counters(c, h, false);
}

int vsvb::finish_counters(vsvb_context* c, const unsigned long long* h, bool replayed) {
  if (!c->ran_quartets) {  // a batch-group member: its integrals were counted by the leader
    std::memset(c->class_stats, 0, sizeof(c->class_stats));
    std::memset(c->last_counters, 0, sizeof(c->last_counters));
    return VSVB_OK;
  }
  c->ran_quartets = false;
  const unsigned long long* stamp = h + kCtrStride;
  const double tick_ms = c->wall_khz > 0 ? 1.0 / c->wall_khz : 0.0;
  const int nspin = c->last_nspin;
  double tot[3] = {0, 0, 0};
  unsigned long long t0 = ~0ull, t1 = 0;
  for (int q = 0; q < kNQuartetClass; ++q) {
    for (int k = 0; k < 3; ++k) tot[k] += (double)h[4 * q + k];
    const bool launched = (c->last_jk ? c->ljk[q].units : c->le[q].units) > 0;
    double cms = 0.0;
    if (c->profile && launched && stamp[2 * q + 1] >= stamp[2 * q]) {
      cms = (double)(stamp[2 * q + 1] - stamp[2 * q]) * tick_ms;
      t0 = std::min(t0, stamp[2 * q]);
      t1 = std::max(t1, stamp[2 * q + 1]);
    }
    c->class_stats[q][0] = cms;
    c->class_stats[q][1] = (double)h[4 * q];
    c->class_stats[q][2] = (double)h[4 * q + 1];
    c->class_stats[q][3] = (double)h[4 * q + 2];
    c->class_stats[q][4] = (double)h[4 * q + 1] * kFlopsPerPrimQuartet[q] +
                           (double)h[4 * q] * (kFlopsHrr[q] + c->last_nwfn * digestion_flops(q, nspin, c->last_jk));
    c->class_stats[q][5] = launched ? 1.0 : 0.0;
  }
  double ms = std::nan("");
  if (!replayed && c->ev_valid) {
    float evms = 0.0f;
    HIP_OK(hipEventElapsedTime(&evms, c->ev0, c->ev1));
    ms = evms;
  } else if (c->profile && t1 >= t0) {
    ms = (double)(t1 - t0) * tick_ms;
  }
  c->last_counters[0] = tot[0];
  c->last_counters[1] = tot[1];
  c->last_counters[2] = tot[2];
  c->last_counters[3] = ms;
  return VSVB_OK;
}

int vsvb::fetch_out(vsvb_context* c, bool grad) {
  const size_t words = kOutGrad + (grad ? (size_t)c->totlen : 0);
  c->h_out.resize(words);
  HIP_OK(hipMemcpyAsync(c->h_out.data(), c->d_out.p, words * sizeof(unsigned long long), hipMemcpyDeviceToHost,
                        c->stream));
  HIP_OK(hipStreamSynchronize(c->stream));
  return VSVB_OK;
}

int vsvb::check_status(vsvb_context* c, bool for_grad) {
  int st[4];
  std::memcpy(st, c->h_out.data() + kOutStatus, sizeof(st));
  if (st[0]) return fail(VSVB_ERR_NUMERIC, "orbital overlap block is not positive definite (linearly dependent orbitals)");
  if (st[2])
    return fail(VSVB_ERR_NUMERIC, "a transition overlap between two determinants of the spin-coupled expansion is "
                                  "exactly singular (cofactors of singular blocks are not implemented)");
  if (for_grad && st[1])
    return fail(VSVB_ERR_UNSUPPORTED, "gradient requested while the per-shell weight screen drops shells (raise ntol_d)");
  return VSVB_OK;
}

// Enqueue one plain-energy evaluation on the context stream (no host sync).
static int enqueue_energy(vsvb_context* c, const double* coords, const double* coeff) {
  int rc;
  if ((rc = prepare_geometry(c, coords))) return rc;
  if ((rc = prepare_orbitals(c, coeff, nullptr, 1))) return rc;
  return run_quartets(c, false);
}

static int finish_energy(vsvb_context* c, double* energy, double* parts) {
  int rc;
  if ((rc = fetch_out(c, false))) return rc;
  const double* h = reinterpret_cast<const double*>(c->h_out.data());
  if ((rc = check_status(c, false))) return rc;
  if ((rc = finish_counters(c))) return rc;
  if (!std::isfinite(h[2])) return fail(VSVB_ERR_NUMERIC, "non-finite energy");
  if (energy) *energy = h[2];
  if (parts) {
    parts[0] = h[0] + h[1];
    parts[1] = 1.0;
    parts[2] = h[0];
    parts[3] = c->enuc;
  }
  return VSVB_OK;
}

static int energy_impl(vsvb_context* c, const double* coords, const double* coeff, double* energy, double* parts) {
  int rc;
  HIP_OK(hipSetDevice(c->device));
  if (c->npair > 0) {
    if ((rc = prepare_geometry(c, coords))) return rc;
    if ((rc = prepare_orbital_basis(c, coeff, nullptr))) return rc;
    if ((rc = sc_enqueue(c, false, nullptr))) return rc;
    return sc_finish(c, energy, parts, nullptr);
  }
  if ((rc = enqueue_energy(c, coords, coeff))) return rc;
  return finish_energy(c, energy, parts);
}

// Gradient assembly from the J/K accumulators.
//   J = A + A^T (Coulomb matrix of RT),  Kx_s = B_s + B_s^T (x_s * exchange matrix of D_s)
//   F2_s = dE2/dD_s = cfac J - Kx_s,  E2 = 1/2 sum_s tr(D_s F2_s)
//   F_s = w1 h + F2_s,  dE/dC_s = 2 P_s C_s F_s (1 - R_s S_ao)   (row-major C_s = orbital rows)
static int gradient_impl(vsvb_context* c, double* grad_dev) {
  hipStream_t st = c->stream;
  if (c->d_ao_ptr.p) {
    HIP_OK(launch_orbital_back(st, orb_args(c), nullptr, 1, grad_dev));
    return VSVB_OK;
  }
  const int n = c->nbf, ns = c->nsp;
  const size_t nn = (size_t)n * n;
  const int nspin = c->nunpd > 0 ? 2 : 1;
  const int T = 256;
  const int gb = (int)((nn + T - 1) / T);
  const double cfac = nspin == 1 ? 2.0 : 1.0, w1 = nspin == 1 ? 2.0 : 1.0;
  hipLaunchKernelGGL(k_sym_combine, dim3(gb), dim3(T), 0, st, c->d_J.p, 1.0, (const double*)nullptr, 0.0, n,
                     c->d_Jsym.p);
  hipLaunchKernelGGL(k_fill, dim3(1024), dim3(256), 0, st, c->d_gradC.p, (size_t)ns * n, 0.0);
  for (int s = 0; s < nspin; ++s) {
    const int off = s == 0 ? 0 : c->nunpd;
    const int m = s == 0 ? c->nalpha_rows : c->ndocc;
    if (m == 0) continue;
    double* F = c->d_F.p + (size_t)s * nn;
    hipLaunchKernelGGL(k_sym_combine, dim3(gb), dim3(T), 0, st, c->d_K.p + (size_t)s * nn, -1.0, c->d_Jsym.p, cfac,
                       n, F);
    hipLaunchKernelGGL(k_trace_prod, dim3(trace_blocks(n)), dim3(256), 0, st, c->d_R.p + (size_t)s * nn, n, 0, F, n, 0.5,
                       c->d_scal.p + 3);
    hipLaunchKernelGGL(k_sym_combine, dim3(gb), dim3(T), 0, st, c->d_H.p, 0.5 * w1, F, 1.0, n, F);
    const double* Ct = c->d_Ct.p + (size_t)off * n;
    const double* P = c->d_P.p + (size_t)s * ns * ns;
    HIP_OK(gemm(st, m, n, m, 1.0, P, m, false, Ct, n, false, 0.0, c->d_X.p, n));                   // X = P C
    HIP_OK(gemm(st, n, n, m, 1.0, Ct, n, true, c->d_X.p, n, false, 0.0, c->d_Rfull.p, n));       // R = C^T P C
    HIP_OK(gemm(st, m, n, n, 1.0, Ct, n, false, F, n, false, 0.0, c->d_X.p, n));                  // X = C F
    HIP_OK(gemm(st, m, n, n, 1.0, c->d_X.p, n, false, c->d_Rfull.p, n, false, 0.0, c->d_Z.p, n)); // Z = X R
    HIP_OK(gemm(st, m, n, n, -1.0, c->d_Z.p, n, false, c->d_S.p, n, false, 1.0, c->d_X.p, n));    // X -= Z S
    HIP_OK(gemm(st, m, n, m, 2.0, P, m, false, c->d_X.p, n, false, 1.0, c->d_gradC.p + (size_t)off * n, n));
  }
  HIP_OK(launch_gather_grad(c, c->d_gradC.p, grad_dev));
  return VSVB_OK;
}

static int enqueue_energy_grad(vsvb_context* c, const double* coords, const double* coeff_host,
                               const double* coeff_dev, double* grad_dev) {
  int rc;
  if ((rc = prepare_geometry(c, coords))) return rc;
  if ((rc = prepare_orbitals(c, coeff_host, coeff_dev, 2))) return rc;
  if ((rc = run_quartets(c, true))) return rc;
  return gradient_impl(c, grad_dev);
}

static int finish_energy_grad(vsvb_context* c, double* energy, double* grad) {
  int rc;
  if ((rc = fetch_out(c, grad != nullptr))) return rc;
  const double* h = reinterpret_cast<const double*>(c->h_out.data());
  if (grad) std::memcpy(grad, h + kOutGrad, c->totlen * sizeof(double));
  if ((rc = check_status(c, true))) return rc;
  if ((rc = finish_counters(c))) return rc;
  const double e = h[0] + h[3] + c->enuc;
  if (!std::isfinite(e)) return fail(VSVB_ERR_NUMERIC, "non-finite energy");
  if (energy) *energy = e;
  return VSVB_OK;
}

// First batched mode: one context per wave function, every evaluation enqueued
// on its own stream before any host synchronization, so independent wave
// functions overlap on the device.
// Wave functions on the same molecule (geometry, atom types and basis) and of
// the same spin type form a group: the group leader owns the geometry data and
// runs one shell-quartet pass whose thread blocks contract each ERI block with
// every member's density; members alias the leader's geometry buffers and use
// slices of the group's density / Coulomb / exchange arrays.
// Members of a group (wave functions on one geometry) from which their J and K come
// from stored integrals, and most memory for them.  32 wave functions of C8H18 took
// 46.0 ms quartet by quartet and take 13.9 so: 4.3 for the integrals, 8.2 for passes
// over the two 4 GB orders of the matrix that do not grow with the members, 1.5 for
// the members' own algebra; at 8 members the two are about even.  A single C2H6 or
// C3H8 wave function (0.70 and 1.19 ms) lost 7 and 10 % by it.
constexpr int kStoredMembers = 8;
constexpr size_t kStoredGroupBytes = (size_t)16 << 30;

struct BatchGroup {
  std::vector<int> members;  // indices into vsvb_batch::ctx; members[0] leads
  DevBuf<double> dens, jacc, kacc;
  DevBuf<OrbArgs> orec;           // the members' orbital records, when they have entry lists
  std::vector<OrbArgs> h_orec;
  StoredIntegrals stored;         // of a group of many densities
};

// The first run of a batch is enqueued directly and then captured whole
// (every group's geometry, orbital, quartet and gradient launches, then a
// gather of all energies, gradients, status words and counters into four
// device arrays) into one HIP graph; later runs replay it: one graph launch
// and one copy to pinned host memory per run.  The systems of a batch are fixed
// at creation, so the captured work never changes.
constexpr int kTuneBuckets = 2;  // groups of one wave function (and of a few), groups of more
constexpr int kTuneCols = 8;
constexpr int kBatchLanes = 4;  // streams the groups of a batch run on
// Group-launch chunks per lane: 0 (one quartet pass per group) by default.  On
// the 96-wave-function C8H18 batch (MI355X) one launch per class over a
// stream's groups cut the serialized quartet time from 423 to 336 ms per run
// (one stream: 471 -> 379 ms per run), but on four streams the per-group
// passes overlap better with the groups' orbital and gradient work: 338-340 ms
// against 348-365 ms for 1-3 chunks on 2-4 streams.
constexpr int kDefaultChunks = 0;

// One launch of a quartet class over several groups of a lane (the argument
// records d_qargs[off, off + ng)).
struct GroupLaunch {
  int q = 0, lane = 0, off = 0, ng = 0, blocks = 0;
  int coop_idx = -1;  // cooperative kernel (step-table index), or -1: straight-line kernel
  bool tr = false;    // straight-line: transposed J/K units
  size_t lds = 0;     // dynamic LDS: the largest of the groups' exchange staging
  std::vector<int> groups;  // the groups whose records it takes, in record order
  double ms = 0.0, flops = 0.0;  // last run: span of the launch (profiling on), algorithmic FLOPs of its groups
};

// Groups of one lane that run as one unit: their geometry and orbital work,
// then one launch per class over all of them, then their gradients.
struct LaneChunk {
  int lane = 0;
  std::vector<int> groups;  // in enqueue order
  int l0 = 0, l1 = 0;       // its launches glaunch[l0, l1)
};

struct GatherItem {
  const unsigned long long* out;  // vsvb_context::d_out
  double enuc;
  size_t goff;
  int len, spin_coupled;
};

struct vsvb_batch {
  std::vector<vsvb_context*> ctx;
  std::vector<BatchGroup> groups;
  std::vector<int> order;                // groups in enqueue order (estimated cost, largest first)
  std::vector<int> lane_of;              // lane of each group
  std::vector<double> gcost;             // estimated work of each group
  // Class launches over many groups (vsvb_batch_set_group_launch): chunks per
  // lane (0: every group launches its own classes), the plan of the last
  // direct run, its argument records on the device and the launches' timing.
  int chunks = kDefaultChunks;
  bool planned = false;
  std::vector<LaneChunk> lchunks;
  std::vector<GroupLaunch> glaunch;
  std::vector<QuartetArgs> h_qargs;
  DevBuf<QuartetArgs> d_qargs;
  DevBuf<unsigned long long> d_lstamp;   // kStampSlots slot pairs per launch
  DevBuf<unsigned long long> d_lspan;    // per launch: first wavefront start, last wavefront end
  std::vector<unsigned long long> h_lspan;
  double lstats[kNQuartetClass][2] = {};  // per class: summed launch time (ms), launches
  hipStream_t stream = nullptr;          // the run's own stream: fork, join, gather, graph launch
  std::vector<hipStream_t> lanes;        // group streams (default priority), forked from and joined to stream
  hipEvent_t ev_fork = nullptr;
  std::vector<hipEvent_t> ev_join;
  int runs = 0;
  bool tuned = false;
  // per bucket and class: coop, per_cu, lds, claim, transposed, best ms, default ms, tuned
  double tuning[kTuneBuckets][kNQuartetClass][kTuneCols] = {};
  bool graph_failed = false;
  bool graph_off = false;        // runs stay direct (vsvb_batch_set_graph)
  bool graph_hold = false;       // new coordinates were set: the next run is direct and is not captured
  std::string graph_error;
  hipGraphExec_t exec = nullptr;
  std::vector<size_t> goff;      // offset of each wave function's gradient in d_g
  std::vector<char> ran;         // the wave function ran the quartet stage itself (group leader)
  DevBuf<GatherItem> d_items;
  DevBuf<double> d_e, d_g;
  DevBuf<int> d_st;
  DevBuf<unsigned long long> d_cnt;
  double* h_e = nullptr;
  double* h_g = nullptr;
  int* h_st = nullptr;
  unsigned long long* h_cnt = nullptr;
  ~vsvb_batch() {
    if (exec) (void)hipGraphExecDestroy(exec);
    if (h_e) (void)hipHostFree(h_e);
    if (h_g) (void)hipHostFree(h_g);
    if (h_st) (void)hipHostFree(h_st);
    if (h_cnt) (void)hipHostFree(h_cnt);
    groups.clear();
    for (auto* c : ctx) vsvb_context_destroy(c);
    for (auto e : ev_join) (void)hipEventDestroy(e);
    if (ev_fork) (void)hipEventDestroy(ev_fork);
    for (auto s : lanes) (void)hipStreamDestroy(s);
    if (stream) (void)hipStreamDestroy(stream);
  }
};

// Groups go to the lane streams longest first, each to the lane with the least
// estimated work so far, and every lane enqueues its groups in that order, so
// that one large group (many densities on one molecule) does not end up
// behind a lane's share of small ones.  Estimated work of a group: squared
// shell-pair count (quartets) times 1 + (densities - 1) / 5 (the quartet
// pass of 32 C8H18 densities measured about 7x that of one).
static void assign_lanes(vsvb_batch* b, int nl) {
  const size_t ng = b->groups.size();
  std::vector<double> cost(ng);
  for (size_t k = 0; k < ng; ++k) {
    const vsvb_context* lead = b->ctx[b->groups[k].members[0]];
    const double np = lead->npairs;
    cost[k] = np * np * (1.0 + 0.2 * ((double)b->groups[k].members.size() - 1.0));
  }
  b->order.resize(ng);
  for (size_t k = 0; k < ng; ++k) b->order[k] = (int)k;
  std::stable_sort(b->order.begin(), b->order.end(), [&](int x, int y) { return cost[x] > cost[y]; });
  std::vector<double> load(nl, 0.0);
  b->lane_of.assign(ng, 0);
  b->gcost = cost;
  for (int gi : b->order) {
    const int l = (int)(std::min_element(load.begin(), load.end()) - load.begin());
    load[l] += cost[gi];
    b->lane_of[gi] = l;
    for (int i : b->groups[gi].members) b->ctx[i]->stream = b->lanes[l];
  }
  b->planned = false;
}

constexpr int kCnt = kStatWords;  // counters and timing stamps per context

// All device work of one batch run, no host synchronization.  The groups run
// on the lane streams, which fork from the batch stream at the start and join
// it at the end (in a captured graph: parallel branches).
static int batch_enqueue_groups(vsvb_batch* b);

static int batch_enqueue(vsvb_batch* b) {
  HIP_OK(hipEventRecord(b->ev_fork, b->stream));
  for (auto s : b->lanes) HIP_OK(hipStreamWaitEvent(s, b->ev_fork, 0));
  int rc = batch_enqueue_groups(b);
  // Every lane joins the batch stream, also after a failure: under stream
  // capture a lane that never joins would stay in capture mode.
  for (size_t k = 0; k < b->lanes.size(); ++k) {
    const hipError_t e1 = hipEventRecord(b->ev_join[k], b->lanes[k]);
    const hipError_t e2 = hipStreamWaitEvent(b->stream, b->ev_join[k], 0);
    if (!rc && (e1 != hipSuccess || e2 != hipSuccess))
      rc = fail(VSVB_ERR_DEVICE, std::string("joining the group streams: ") +
                                     hipGetErrorString(e1 != hipSuccess ? e1 : e2));
  }
  return rc;
}

static hipError_t launch_group_rec(vsvb_batch* b, const GroupLaunch& r, unsigned long long* stamp) {
  const QuartetArgs* gs = b->d_qargs.p + r.off;
  hipStream_t st = b->lanes[r.lane];
  if (r.coop_idx >= 0) return launch_coop_groups(r.coop_idx, gs, r.ng, r.blocks, b->ctx[0]->device, stamp, st);
  const int bc = class_bra(r.q), kc = r.q - quartet_class_index(bc, 0);
  return launch_groups_class(bc, kc, gs, r.ng, r.tr, r.blocks, r.lds, stamp, st);
}

template <typename T>
static hipError_t ensure_buffer(DevBuf<T>& d, size_t count) {
  if (d.p && d.n >= count) return hipSuccess;
  if (d.p && d.own) (void)hipFree(d.p);
  d.p = nullptr;
  return d.alloc(count);
}

// Plan of the class launches over many groups: every lane's closed- and
// high-spin groups (a spin-coupled group runs its own pass) in `chunks`
// consecutive chunks of about equal estimated work; per chunk and class one
// launch over the chunk's groups, or one per kernel variant when the groups'
// launch policies differ (cooperative or straight-line kernel, orientation).
// Each group keeps its own work units, claims and buffers (its argument
// record); the launch takes the largest grid and exchange staging among them.
// The records go to the device here, on a direct run before any capture, and
// stay unchanged while a captured graph refers to them.
static int batch_plan(vsvb_batch* b) {
  b->planned = false;
  b->lchunks.clear();
  b->glaunch.clear();
  b->h_qargs.clear();
  if (b->chunks <= 0) return VSVB_OK;
  for (auto& g : b->groups) {  // the argument records hold the work lists of the geometry to be run
    const int rc = schedule_pairs(b->ctx[g.members[0]]);
    if (rc) return rc;
  }
  for (int l = 0; l < (int)b->lanes.size(); ++l) {
    std::vector<int> gl;
    double tot = 0.0;
    for (int gi : b->order)
      if (b->lane_of[gi] == l) {
        gl.push_back(gi);
        tot += b->gcost[gi];
      }
    if (gl.empty()) continue;
    const int K = std::min<int>(b->chunks, (int)gl.size());
    const size_t c0 = b->lchunks.size();
    for (int k = 0; k < K; ++k) {
      b->lchunks.emplace_back();
      b->lchunks.back().lane = l;
    }
    double run = 0.0;
    for (int gi : gl) {
      const int k = std::min(K - 1, (int)(run * K / std::max(tot, 1e-300)));
      b->lchunks[c0 + k].groups.push_back(gi);
      run += b->gcost[gi];
    }
  }
  for (auto& ch : b->lchunks) {
    ch.l0 = (int)b->glaunch.size();
    for (int q = 0; q < kNQuartetClass; ++q) {
        const int bc = class_bra(q), kc = q - quartet_class_index(bc, 0);
        // kernel variants of this class in the chunk: key -1 - coop index (cooperative), 0 / 1 (orientation)
        std::vector<int> keys;
        std::vector<std::vector<QuartetArgs>> args;
        std::vector<GroupLaunch> recs;
        for (int gi : ch.groups) {
          BatchGroup& g = b->groups[gi];
          vsvb_context* lead = b->ctx[g.members[0]];
          if (lead->npair > 0 || g.stored.M.p) continue;  // (runs its own pass)
          const int nb = lead->pair_off[bc + 1] - lead->pair_off[bc], nk = lead->pair_off[kc + 1] - lead->pair_off[kc];
          if (nb <= 0 || nk <= 0) continue;
          const ClassLaunch& cl = lead->ljk[q];
          if (cl.units <= 0)
            return fail(VSVB_ERR_UNSUPPORTED, "quartet class " + std::to_string(q) + " has no launchable work units");
          const int nwfn = (int)g.members.size();
          const int nspin = lead->nunpd > 0 ? 2 : 1;
          QuartetArgs a = class_args(lead, bc, kc, cl, true, nwfn, nspin, nwfn > 1 ? g.dens.p : lead->d_R.p,
                                     nwfn > 1 ? g.jacc.p : lead->d_J.p, nwfn > 1 ? g.kacc.p : lead->d_K.p,
                                     lead->d_partial.p);
          a.stamp = nullptr;  // the launch is timed as a whole
          const int key = cl.coop ? -1 - lead->coop_idx[q] : (cl.tr ? 1 : 0);
          size_t v = 0;
          while (v < keys.size() && keys[v] != key) ++v;
          if (v == keys.size()) {
            keys.push_back(key);
            args.emplace_back();
            GroupLaunch r;
            r.q = q;
            r.lane = ch.lane;
            r.coop_idx = cl.coop ? lead->coop_idx[q] : -1;
            r.tr = !cl.coop && cl.tr;
            recs.push_back(r);
          }
          args[v].push_back(a);
          recs[v].groups.push_back(gi);
          recs[v].blocks = std::max(recs[v].blocks, cl.blocks);
          recs[v].lds = std::max(recs[v].lds, cl.coop ? (size_t)0 : cl.lds);
        }
        for (size_t v = 0; v < keys.size(); ++v) {
          recs[v].off = (int)b->h_qargs.size();
          recs[v].ng = (int)args[v].size();
          b->h_qargs.insert(b->h_qargs.end(), args[v].begin(), args[v].end());
          b->glaunch.push_back(recs[v]);
        }
      }
    ch.l1 = (int)b->glaunch.size();
  }
  const size_t nlaunch = b->glaunch.size();
  HIP_OK(ensure_buffer(b->d_qargs, std::max<size_t>(b->h_qargs.size(), 1)));
  HIP_OK(ensure_buffer(b->d_lstamp, std::max<size_t>(nlaunch, 1) * 2 * kStampSlots));
  HIP_OK(ensure_buffer(b->d_lspan, std::max<size_t>(nlaunch, 1) * 2));
  if (!b->h_qargs.empty())
    HIP_OK(hipMemcpy(b->d_qargs.p, b->h_qargs.data(), b->h_qargs.size() * sizeof(QuartetArgs), hipMemcpyHostToDevice));
  b->h_lspan.assign(2 * nlaunch, 0);
  b->planned = true;
  return VSVB_OK;
}

// Every member's orbital algebra runs along its entry lists: the group shares its launches.
static bool group_one_launch(const vsvb_batch* b, const BatchGroup& g) {
  if (g.members.size() < 2) return false;
  const vsvb_context* lead = b->ctx[g.members[0]];
  for (int i : g.members) {
    const vsvb_context* c = b->ctx[i];
    if (!c->d_ao_ptr.p || c->nbf != lead->nbf || c->nalpha_rows != lead->nalpha_rows || c->ndocc != lead->ndocc ||
        c->nunpd != lead->nunpd)
      return false;
  }
  return true;
}

// The members' orbital stage; pass 2: the group's J/K pass follows, and its
// counters and accumulators are cleared along.
static int group_orbitals(vsvb_batch* b, BatchGroup& g, int pass) {
  vsvb_context* lead = b->ctx[g.members[0]];
  int rc;
  const int nwfn = (int)g.members.size();
  if (!group_one_launch(b, g)) {
    for (int i : g.members)
      if ((rc = prepare_orbitals(b->ctx[i], nullptr, nullptr, nwfn == 1 ? pass : 0))) return rc;
    return VSVB_OK;
  }
  if (g.h_orec.empty()) {  // constant over the batch's life; written on a direct run, before any capture
    if (lead->capturing) return fail(VSVB_ERR_DEVICE, "orbital records of a batch group are not on the device");
    for (int i : g.members) g.h_orec.push_back(orb_args(b->ctx[i]));
    HIP_OK(g.orec.alloc(g.h_orec.size()));
    HIP_OK(hipMemcpyAsync(g.orec.p, g.h_orec.data(), g.h_orec.size() * sizeof(OrbArgs), hipMemcpyHostToDevice,
                          lead->stream));
  }
  HIP_OK(launch_orbital_front(lead->stream, g.h_orec[0], g.orec.p, nwfn,
                              pass_zero(lead, pass, nwfn, g.jacc.p, g.kacc.p)));
  lead->cleared = pass;
  return VSVB_OK;
}

// Geometry and orbital work of one group, and, for a spin-coupled group, its
// whole pass; with own = true also its own quartet pass and its gradients.
static int group_front(vsvb_batch* b, BatchGroup& g, bool own) {
  int rc;
  vsvb_context* lead = b->ctx[g.members[0]];
  for (int i : g.members)
    for (int k = 0; k < b->ctx[i]->totlen; ++k)
      if (b->ctx[i]->ent[k].kind != 0) return fail(VSVB_ERR_UNSUPPORTED, "batched wave functions with NDFs");
  // geometry-dependent data are rebuilt every run: passing the coordinates forces it
  if ((rc = prepare_geometry(lead, lead->coords.data()))) return rc;
  if (lead->npair > 0) {
    if ((rc = prepare_orbital_basis(lead, nullptr, nullptr))) return rc;
    return sc_enqueue(lead, true, lead->d_grad.p);
  }
  const int nwfn = (int)g.members.size();
  if (g.stored.M.p) {
    if ((rc = group_orbitals(b, g, 1))) return rc;
    return stored_jk(lead, g.stored, nwfn, g.dens.p, g.jacc.p, g.kacc.p);
  }
  if ((rc = group_orbitals(b, g, own ? 2 : 0))) return rc;
  if (!own) {
    const int nspin = lead->nunpd > 0 ? 2 : 1;
    HIP_OK(quartet_pass_clear(lead, true, nwfn, nspin, nwfn > 1 ? g.jacc.p : lead->d_J.p,
                              nwfn > 1 ? g.kacc.p : lead->d_K.p, kCounterWords));
    return VSVB_OK;
  }
  if (nwfn > 1) {
    if ((rc = run_quartets(lead, true, nwfn, g.dens.p, g.jacc.p, g.kacc.p))) return rc;
  } else if ((rc = run_quartets(lead, true))) {
    return rc;
  }
  return VSVB_OK;
}

static int group_gradients(vsvb_batch* b, BatchGroup& g) {
  vsvb_context* lead = b->ctx[g.members[0]];
  if (lead->npair > 0) return VSVB_OK;
  if (group_one_launch(b, g)) {
    for (int i : g.members) b->ctx[i]->enuc = lead->enuc;
    HIP_OK(launch_orbital_back(lead->stream, g.h_orec[0], g.orec.p, (int)g.members.size(), nullptr));
    return VSVB_OK;
  }
  for (int i : g.members) {
    vsvb_context* m = b->ctx[i];
    m->enuc = lead->enuc;
    const int rc = gradient_impl(m, m->d_grad.p);
    if (rc) return rc;
  }
  return VSVB_OK;
}

// Every group's device work on its lane stream.  Every wave function goes
// through the J/K (adjoint-ready) contraction; the energy is assembled from it,
// and the gradient when asked for.  With a plan of group launches, each lane
// chunk runs its groups' geometry and orbital work, then one launch per class
// over the chunk, then the gradients; otherwise every group runs its own pass.
static int batch_enqueue_groups(vsvb_batch* b) {
  int rc;
  if (!b->planned || b->chunks <= 0) {
    // Groups on odd lanes run their classes in reverse order, so concurrent
    // lanes tend to pair the VALU-bound low-angular-momentum classes with the
    // latency-bound cooperative (d-heavy) ones.  Measured on the 96-member
    // C8H18 batch over four runs each: 360-362 evals/s against 350-361.
    for (int gi : b->order) {
      BatchGroup& g = b->groups[gi];
      b->ctx[g.members[0]]->class_rev = b->lane_of[gi] & 1;
      if ((rc = group_front(b, g, true))) return rc;
      if ((rc = group_gradients(b, g))) return rc;
    }
    return VSVB_OK;
  }
  const bool prof = b->ctx[0]->profile;
  for (const auto& ch : b->lchunks) {
    for (int gi : ch.groups)
      if ((rc = group_front(b, b->groups[gi], false))) return rc;
    hipStream_t st = b->lanes[ch.lane];
    const int nl = ch.l1 - ch.l0;
    unsigned long long* stamps = b->d_lstamp.p + (size_t)ch.l0 * 2 * kStampSlots;
    if (prof && nl > 0) {
      const int nslot = nl * 2 * kStampSlots;
      hipLaunchKernelGGL(k_stamp_reset, dim3((nslot + 255) / 256), dim3(256), 0, st, stamps, nslot);
    }
    for (int r = ch.l0; r < ch.l1; ++r)
      HIP_OK(launch_group_rec(b, b->glaunch[r], prof ? b->d_lstamp.p + (size_t)r * 2 * kStampSlots : nullptr));
    if (prof && nl > 0)
      hipLaunchKernelGGL(k_stamp_reduce, dim3(nl), dim3(kStampSlots), 0, st, stamps, b->d_lspan.p + 2 * (size_t)ch.l0);
    HIP_OK(hipGetLastError());
    for (int gi : ch.groups)
      if ((rc = group_gradients(b, b->groups[gi]))) return rc;
  }
  return VSVB_OK;
}

// Per-class launch times of the last run's group launches (profiling on).
static int batch_launch_stats(vsvb_batch* b) {
  std::memset(b->lstats, 0, sizeof(b->lstats));
  if (!b->planned || b->chunks <= 0) return VSVB_OK;
  const bool prof = b->ctx[0]->profile;
  if (prof && !b->glaunch.empty())
    HIP_OK(hipMemcpy(b->h_lspan.data(), b->d_lspan.p, b->h_lspan.size() * sizeof(unsigned long long),
                     hipMemcpyDeviceToHost));
  const double tick_ms = b->ctx[0]->wall_khz > 0 ? 1.0 / b->ctx[0]->wall_khz : 0.0;
  for (size_t r = 0; r < b->glaunch.size(); ++r) {
    GroupLaunch& L = b->glaunch[r];
    const int q = L.q;
    b->lstats[q][1] += 1.0;
    const unsigned long long t0 = b->h_lspan[2 * r], t1 = b->h_lspan[2 * r + 1];
    L.ms = (prof && t1 >= t0) ? (double)(t1 - t0) * tick_ms : 0.0;
    b->lstats[q][0] += L.ms;
    L.flops = 0.0;  // the groups' leads counted their quartets (finish_counters ran before)
    for (int gi : L.groups) L.flops += b->ctx[b->groups[gi].members[0]]->class_stats[q][4];
  }
  return VSVB_OK;
}

// Results of every wave function into the arrays a replay reads back, a workgroup each.
__global__ void k_gather(const GatherItem* __restrict__ items, double* __restrict__ e, double* __restrict__ g,
                         int* __restrict__ st, unsigned long long* __restrict__ cnt) {
  const GatherItem x = items[blockIdx.x];
  const double* scal = reinterpret_cast<const double*>(x.out);
  const int* status = reinterpret_cast<const int*>(x.out + kOutStatus);
  if (threadIdx.x == 0) e[blockIdx.x] = x.spin_coupled ? scal[2] : scal[0] + scal[3] + x.enuc;
  if (threadIdx.x < 4) st[4 * blockIdx.x + threadIdx.x] = status[threadIdx.x];
  for (int k = threadIdx.x; k < kCnt; k += blockDim.x) {  // the copies added up, then the stamps
    const unsigned long long* n = x.out + kOutCounters;
    unsigned long long s = k < kCtrStride ? 0 : n[kCtrSlots * kCtrStride + k - kCtrStride];
    for (int m = 0; m < (k < kCtrStride ? kCtrSlots : 0); ++m) s += n[m * kCtrStride + k];
    cnt[(size_t)kCnt * blockIdx.x + k] = s;
  }
  for (int k = threadIdx.x; k < x.len; k += blockDim.x)
    g[x.goff + k] = reinterpret_cast<const double*>(x.out + kOutGrad)[k];
}

// The items of the batch's geometries (the nuclear repulsion is one of their
// numbers), uploaded before the capture that reads them.
static int batch_gather_items(vsvb_batch* b) {
  std::vector<GatherItem> items;
  for (size_t i = 0; i < b->ctx.size(); ++i) {
    const vsvb_context* c = b->ctx[i];
    items.push_back(GatherItem{c->d_out.p, c->enuc, b->goff[i], c->totlen, c->npair > 0});
  }
  HIP_OK(ensure_buffer(b->d_items, items.size()));
  HIP_OK(hipMemcpy(b->d_items.p, items.data(), items.size() * sizeof(GatherItem), hipMemcpyHostToDevice));
  return VSVB_OK;
}

static int batch_gather(vsvb_batch* b) {
  hipLaunchKernelGGL(k_gather, dim3((unsigned)b->ctx.size()), dim3(256), 0, b->stream, b->d_items.p, b->d_e.p, b->d_g.p,
                     b->d_st.p, b->d_cnt.p);
  HIP_OK(hipGetLastError());
  return VSVB_OK;
}

// Launch tuner of the batch (J/K mode), run before the first run.  Groups of
// one wave function (one density per quartet pass) and groups of more than
// kFewDensities (J/K contractions of many densities per quartet) are tuned
// apart: for each bucket a representative closed- or high-spin group leader --
// single: the molecule size that occurs most often; many: the group with the
// most density work -- times every candidate configuration of every class on its
// own data: the straight-line kernel with 1 or 2 workgroups per CU, with or
// without the LDS exchange staging, in both orientations (classes with
// different bra and ket classes); for classes with step tables the cooperative
// kernel with automatic, 1-, 8- or 64-unit claims and 8, 4 or 2 workgroups
// per CU.  Both kernels stay below their occupancy: a class timed alone often
// ranks 4 or as many straight-line workgroups per CU as fit first, and as many
// cooperative ones as fit, but in the batch four lane streams run classes side
// by side.  On the 96-member C8H18 batch, capping the straight-line launches at
// 2 per CU measured 330-333 -> 339-347 evals/s (1 per CU: 331-338), then
// dropping the cooperative kernel's as-many-as-fit candidate 340 -> 349-358
// (cooperative candidates 4 and 2 only: 340-341).  The
// fastest (best of two launches) becomes the class policy of every group of
// the bucket if it beats the default (the first candidate) by 3% or more (a
// candidate already 1.5x slower than the best after one launch gets no
// second).  The launches accumulate into the leader's J/K arrays,
// which the first run clears again.
static int tune_leader(vsvb_batch* b, BatchGroup* gs, double (*tuning)[kTuneCols], std::vector<Policy>& best) {
  vsvb_context* L = b->ctx[gs->members[0]];
  int rc;
  if ((rc = prepare_geometry(L, L->coords.data()))) return rc;
  if ((rc = group_orbitals(b, *gs, 0))) return rc;
  const int nwfn = (int)gs->members.size();
  const double* dens = nwfn > 1 ? gs->dens.p : L->d_R.p;
  double* jacc = nwfn > 1 ? gs->jacc.p : L->d_J.p;
  double* kacc = nwfn > 1 ? gs->kacc.p : L->d_K.p;
  const int nspin = L->nunpd > 0 ? 2 : 1;
  struct Events {  // released on every return path
    hipEvent_t a = nullptr, b = nullptr;
    ~Events() {
      if (a) (void)hipEventDestroy(a);
      if (b) (void)hipEventDestroy(b);
    }
  } ev;
  HIP_OK(hipEventCreate(&ev.a));
  HIP_OK(hipEventCreate(&ev.b));
  hipEvent_t e0 = ev.a, e1 = ev.b;
  best.assign(kNQuartetClass, Policy{});
  for (int bc = 0; bc < kNPairClass; ++bc)
    for (int kc = 0; kc <= bc; ++kc) {
      const int q = quartet_class_index(bc, kc);
      if (L->ljk[q].units <= 0 || L->in_small[1][q]) continue;  // (small classes share one launch)
      std::vector<Policy> cand;
      const bool coop = L->coop_idx[q] >= 0;
      Policy d0;  // the default
      d0.tr = L->ljk[q].tr;
      d0.per_cu = coop ? 8 : 2;
      cand.push_back(d0);
      if (coop) {
        for (int pc : {8, 4, 2})
          for (int cl : {0, 1, 8, 64}) {
            Policy p;
            p.per_cu = pc;
            p.claim = cl;
            cand.push_back(p);
          }
      } else {
        for (int pc : {1, 2})
          for (bool lds : {true, false}) {
            Policy p;
            p.per_cu = pc;
            p.lds_on = lds;
            cand.push_back(p);
            if (bc != kc && lds) {
              p.tr = true;
              cand.push_back(p);
            }
          }
        if (bc != kc) {
          Policy p;
          p.tr = true;
          p.lds_on = false;
          p.per_cu = 2;
          cand.push_back(p);
        }
      }
      double tbest = 1e30, tdef = 0.0;
      for (size_t k = 0; k < cand.size(); ++k) {
        const ClassLaunch cl = policy_launch(L, q, cand[k]);
        if (cl.overflow) continue;  // not a launch this class can take
        const QuartetArgs a = class_args(L, bc, kc, cl, true, nwfn, nspin, dens, jacc, kacc, L->d_partial.p);
        float tmin = 1e30f;
        for (int rep = 0; rep < 2; ++rep) {
          HIP_OK(launch_zero(L->stream, L->d_tilectr.p + L->ctr_off[q], L->ctr_len[q] * sizeof(int)));
          HIP_OK(hipEventRecord(e0, L->stream));
          HIP_OK(launch_class(L, bc, kc, cl, a, true));
          HIP_OK(hipEventRecord(e1, L->stream));
          HIP_OK(hipEventSynchronize(e1));
          float ms = 0.0f;
          HIP_OK(hipEventElapsedTime(&ms, e0, e1));
          tmin = std::min(tmin, ms);
          if (tmin > 1.5 * tbest) break;  // clearly slower: no second launch
        }
        if (k == 0) tdef = tmin;
        if (tmin < tbest) {
          tbest = tmin;
          best[q] = cand[k];
        }
      }
      // A candidate replaces the default only if it is at least 3% faster:
      // closer races resolved differently from process to process, and some
      // of those picks overlapped worse in the batch (six batch runs each on
      // the 96-member C8H18 batch: 352-361 evals/s, one run in six at 352,
      // against 359-363 with the margin).
      if (tdef > 0.0 && tbest > 0.97 * tdef) {
        best[q] = cand[0];
        tbest = tdef;
      }
      double* t = tuning[q];
      t[0] = coop ? 1 : 0;
      t[1] = best[q].per_cu;
      t[2] = best[q].lds_on ? 1 : 0;
      t[3] = best[q].claim;
      t[4] = best[q].tr ? 1 : 0;
      t[5] = tbest;
      t[6] = tdef;
      t[7] = 1;
    }
  return VSVB_OK;
}

// Groups of up to this many densities take the single-density policies (their
// launches behave like one density's: measured 245 -> 247 evaluations/s on the
// 96-wave-function batch, whose alkanes come in groups of two).
constexpr size_t kFewDensities = 4;

static int tune_batch(vsvb_batch* b) {
  // representatives: single-density groups -- the most frequent molecule size
  // (ties: the larger); groups of more than kFewDensities -- the most nwfn * nbf^2
  std::map<int, int> freq;
  for (auto& g : b->groups) {
    vsvb_context* l = b->ctx[g.members[0]];
    if (l->npair == 0 && g.members.size() == 1) ++freq[l->nbf];
  }
  int nbf1 = -1, f1 = 0;
  for (auto& kv : freq)
    if (kv.second >= f1) {
      f1 = kv.second;
      nbf1 = kv.first;
    }
  BatchGroup* rep[kTuneBuckets] = {nullptr, nullptr};
  double wmax = 0.0;
  for (auto& g : b->groups) {
    vsvb_context* l = b->ctx[g.members[0]];
    if (l->npair > 0 || g.stored.M.p) continue;
    if (g.members.size() == 1) {
      if (!rep[0] && l->nbf == nbf1) rep[0] = &g;
    } else if (g.members.size() > kFewDensities) {
      const double w = (double)g.members.size() * l->nbf * l->nbf;
      if (w > wmax) {
        wmax = w;
        rep[1] = &g;
      }
    }
  }
  std::vector<Policy> best[kTuneBuckets];
  for (int k = 0; k < kTuneBuckets; ++k) {
    if (!rep[k]) continue;
    const int rc = tune_leader(b, rep[k], b->tuning[k], best[k]);
    if (rc) return rc;
  }
  for (auto& g : b->groups) {
    const int k = g.members.size() > kFewDensities ? 1 : 0;
    if (!rep[k] || g.stored.M.p) continue;
    for (int i : g.members) {
      vsvb_context* c = b->ctx[i];
      if (c->npair > 0) continue;
      for (int q = 0; q < kNQuartetClass; ++q) {
        if (b->tuning[k][q][7] <= 0.0) continue;
        // the representative's best launch may not fit a larger molecule of the
        // bucket (too many work units for 32-bit indices): that group keeps its
        // own default launch, which its context was created with
        c->pol[q] = best[k][q];
        c->has_pol[q] = true;
        if (c->in_small[1][q]) continue;  // runs in the shared launch
        const ClassLaunch cl = policy_launch(c, q, best[k][q]);
        if (!cl.overflow && (cl.units > 0 || c->ljk[q].units <= 0)) c->ljk[q] = cl;
      }
    }
  }
  return VSVB_OK;
}

static int batch_capture(vsvb_batch* b) {
  int rc = batch_gather_items(b);
  if (rc) return rc;
  for (auto* c : b->ctx) c->capturing = true;
  hipError_t e = hipStreamBeginCapture(b->stream, hipStreamCaptureModeThreadLocal);
  if (e == hipSuccess) {
    rc = batch_enqueue(b);
    if (!rc) rc = batch_gather(b);
    hipGraph_t g = nullptr;
    const hipError_t e2 = hipStreamEndCapture(b->stream, &g);
    if (!rc && e2 == hipSuccess && g) {
      e = hipGraphInstantiate(&b->exec, g, nullptr, nullptr, 0);
      if (e != hipSuccess) b->exec = nullptr;
    } else if (e2 != hipSuccess) {
      e = e2;
    }
    if (g) (void)hipGraphDestroy(g);
  }
  for (size_t i = 0; i < b->ctx.size(); ++i) {
    b->ran[i] = b->ctx[i]->ran_quartets;
    b->ctx[i]->capturing = false;
  }
  if (rc || e != hipSuccess || !b->exec) {
    b->graph_failed = true;
    b->graph_error = rc ? g_last_error : std::string(hipGetErrorString(e));
    (void)hipGetLastError();
    return VSVB_ERR_DEVICE;
  }
  return VSVB_OK;
}

static int batch_replay(vsvb_batch* b, int32_t want_grad, double* energies, double* const* grads) {
  hipStream_t st = b->stream;
  const size_t n = b->ctx.size();
  HIP_OK(hipGraphLaunch(b->exec, st));
  HIP_OK(hipMemcpyAsync(b->h_e, b->d_e.p, n * sizeof(double), hipMemcpyDeviceToHost, st));
  HIP_OK(hipMemcpyAsync(b->h_st, b->d_st.p, 4 * n * sizeof(int), hipMemcpyDeviceToHost, st));
  HIP_OK(hipMemcpyAsync(b->h_g, b->d_g.p, b->goff[n] * sizeof(double), hipMemcpyDeviceToHost, st));
  HIP_OK(hipMemcpyAsync(b->h_cnt, b->d_cnt.p, kCnt * n * sizeof(unsigned long long), hipMemcpyDeviceToHost, st));
  HIP_OK(hipStreamSynchronize(st));
  for (size_t i = 0; i < n; ++i) {
    vsvb_context* c = b->ctx[i];
    const int* s4 = b->h_st + 4 * i;
    if (s4[0]) return fail(VSVB_ERR_NUMERIC, "wave function " + std::to_string(i) + ": orbital overlap block is not positive definite");
    if (s4[2]) return fail(VSVB_ERR_NUMERIC, "wave function " + std::to_string(i) + ": exactly singular spin-coupled transition overlap");
    if (want_grad && s4[1]) return fail(VSVB_ERR_UNSUPPORTED, "wave function " + std::to_string(i) + ": gradient with masked shells");
    if (want_grad && c->npair > 0 && s4[3])
      return fail(VSVB_ERR_UNSUPPORTED, "wave function " + std::to_string(i) + ": gradient at a singular spin-coupled transition overlap");
    if (!std::isfinite(b->h_e[i])) return fail(VSVB_ERR_NUMERIC, "wave function " + std::to_string(i) + ": non-finite energy");
    if (energies) energies[i] = b->h_e[i];
    if (want_grad && grads && grads[i]) std::memcpy(grads[i], b->h_g + b->goff[i], c->totlen * sizeof(double));
    c->ran_quartets = b->ran[i];
    int rc;
    if ((rc = finish_counters(c, b->h_cnt + kCnt * i, true))) return rc;
  }
  return VSVB_OK;
}

static bool same_molecule(const vsvb_system* a, const vsvb_system* b) {
  if (a->natom != b->natom || a->ntype != b->ntype || a->nshell_type != b->nshell_type || a->nprim != b->nprim)
    return false;
  if ((a->nunpd > 0) != (b->nunpd > 0) || a->nspinc != b->nspinc || a->npair != b->npair) return false;
  if (a->npair > 0) return false;  // spin-coupled wave functions run their own pass
  auto eq = [](const void* x, const void* y, size_t n) { return std::memcmp(x, y, n) == 0; };
  return eq(a->atom_type, b->atom_type, sizeof(int32_t) * a->natom) &&
         eq(a->coords, b->coords, sizeof(double) * 3 * a->natom) &&
         eq(a->nuc_charge, b->nuc_charge, sizeof(double) * a->ntype) &&
         eq(a->type_shell_start, b->type_shell_start, sizeof(int32_t) * (a->ntype + 1)) &&
         eq(a->shell_l, b->shell_l, sizeof(int32_t) * a->nshell_type) &&
         eq(a->shell_prim_start, b->shell_prim_start, sizeof(int32_t) * (a->nshell_type + 1)) &&
         eq(a->prim_exp, b->prim_exp, sizeof(double) * a->nprim) && eq(a->prim_coef, b->prim_coef, sizeof(double) * a->nprim);
}

// Make member m of a group share the leader's geometry data.
static void share_geometry(vsvb_context* lead, vsvb_context* m) {
  m->d_shells.alias(lead->d_shells.p, lead->d_shells.n);
  m->d_pairs.alias(lead->d_pairs.p, lead->d_pairs.n);
  m->d_psrc.alias(lead->d_psrc.p, lead->d_psrc.n);
  m->d_order.alias(lead->d_order.p, lead->d_order.n);
  m->d_pp.alias(lead->d_pp.p, lead->d_pp.n);
  m->d_pexp.alias(lead->d_pexp.p, lead->d_pexp.n);
  m->d_pcoef.alias(lead->d_pcoef.p, lead->d_pcoef.n);
  m->d_xyz.alias(lead->d_xyz.p, lead->d_xyz.n);
  m->d_charge.alias(lead->d_charge.p, lead->d_charge.n);
  m->d_boys.alias(lead->d_boys.p, lead->d_boys.n);
  m->d_S.alias(lead->d_S.p, lead->d_S.n);
  m->d_H.alias(lead->d_H.p, lead->d_H.n);
  m->geom_ready = true;  // members never rebuild geometry; the leader does
}

// Device Boys function at given arguments (diagnostics / tests).
template <int L>
__global__ void k_boys_probe(const double* __restrict__ T, int n, const double* __restrict__ tab, int compact,
                             double* __restrict__ out) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  double F[L + 1];
  if (compact)
    boys_eval_c<L>(T[i], 1.0, tab + kBoysCOff + (size_t)L * kBoysCLen, F);
  else
    boys_eval<L>(T[i], tab, F);
#pragma unroll
  for (int m = 0; m <= L; ++m) out[(size_t)i * (L + 1) + m] = F[m];
}

// ---------------------------------------------------------------------------
// C ABI
// ---------------------------------------------------------------------------
// Device scratch of the allocation-free entry point (vsvb_energy_grad_static):
// every device buffer of its transient context is carved from this array.
// Each GPU holds its own copy from module load until the process ends; host
// code uses the per-device address from hipGetSymbolAddress, never the name.
// Calls on one GPU are serialized by a host lock (they would race on the
// array); the array keeps the last call's contents, and every buffer the
// pipeline reads is written or cleared earlier in the same call.
constexpr size_t kScratchBytes = (size_t)32 << 20;
constexpr int kScratchDevices = 64;
static __device__ __align__(256) unsigned char scratch[kScratchBytes];
static void* g_scratch_ptr[kScratchDevices] = {};
static std::mutex g_scratch_mu[kScratchDevices];

extern "C" {

int vsvb_debug_boys(int32_t L, const double* T, int32_t n, double* out) {
  const int compact = L >= 16 ? 1 : 0;
  if (compact) L -= 16;
  if (L < 0 || L > kLTot || n < 1 || !T || !out) return fail(VSVB_ERR_ARG, "invalid Boys probe arguments");
  auto tab = make_boys_table();
  DevBuf<double> dt, dT, dout;
  HIP_OK(dt.alloc(tab.size()));
  HIP_OK(dT.alloc(n));
  HIP_OK(dout.alloc((size_t)n * (L + 1)));
  HIP_OK(hipMemcpy(dt.p, tab.data(), tab.size() * sizeof(double), hipMemcpyHostToDevice));
  HIP_OK(hipMemcpy(dT.p, T, n * sizeof(double), hipMemcpyHostToDevice));
  const dim3 g((n + 63) / 64), b(64);
  switch (L) {
#define BP(LL) case LL: hipLaunchKernelGGL(k_boys_probe<LL>, g, b, 0, 0, dT.p, n, dt.p, compact, dout.p); break;
    BP(0) BP(1) BP(2) BP(3) BP(4) BP(5) BP(6) BP(7) BP(8)
#undef BP
  }
  HIP_OK(hipGetLastError());
  HIP_OK(hipMemcpy(out, dout.p, (size_t)n * (L + 1) * sizeof(double), hipMemcpyDeviceToHost));
  return VSVB_OK;
}

// Lowest root of H c = E S c (S symmetric positive definite, m small): Cholesky
// S = L L^T, cyclic Jacobi rotations on M = L^-1 H L^-T, c = L^-T y.  Returns
// false when S is not positive definite.
static bool lowest_root(int m, const std::vector<double>& H, const std::vector<double>& S, double* eig,
                        double* vec) {
  std::vector<double> L((size_t)m * m, 0.0);
  for (int j = 0; j < m; ++j) {
    double d = S[(size_t)j * m + j];
    for (int k = 0; k < j; ++k) d -= L[(size_t)j * m + k] * L[(size_t)j * m + k];
    if (!(d > 0.0)) return false;
    L[(size_t)j * m + j] = std::sqrt(d);
    for (int i = j + 1; i < m; ++i) {
      double v = S[(size_t)i * m + j];
      for (int k = 0; k < j; ++k) v -= L[(size_t)i * m + k] * L[(size_t)j * m + k];
      L[(size_t)i * m + j] = v / L[(size_t)j * m + j];
    }
  }
  // W = L^-1 H (forward substitution per column), M = W L^-T (per row)
  std::vector<double> W((size_t)m * m), M((size_t)m * m);
  for (int c = 0; c < m; ++c)
    for (int i = 0; i < m; ++i) {
      double v = H[(size_t)i * m + c];
      for (int k = 0; k < i; ++k) v -= L[(size_t)i * m + k] * W[(size_t)k * m + c];
      W[(size_t)i * m + c] = v / L[(size_t)i * m + i];
    }
  for (int r = 0; r < m; ++r)
    for (int i = 0; i < m; ++i) {
      double v = W[(size_t)r * m + i];
      for (int k = 0; k < i; ++k) v -= L[(size_t)i * m + k] * M[(size_t)r * m + k];
      M[(size_t)r * m + i] = v / L[(size_t)i * m + i];
    }
  for (int i = 0; i < m; ++i)
    for (int j = 0; j < i; ++j) M[(size_t)i * m + j] = M[(size_t)j * m + i] = 0.5 * (M[(size_t)i * m + j] + M[(size_t)j * m + i]);
  std::vector<double> V((size_t)m * m, 0.0);
  for (int i = 0; i < m; ++i) V[(size_t)i * m + i] = 1.0;
  for (int sweep = 0; sweep < 100; ++sweep) {
    double off = 0.0, tot = 0.0;
    for (int i = 0; i < m; ++i)
      for (int j = 0; j < m; ++j) {
        tot += M[(size_t)i * m + j] * M[(size_t)i * m + j];
        if (i != j) off += M[(size_t)i * m + j] * M[(size_t)i * m + j];
      }
    if (off <= 1e-30 * tot || off == 0.0) break;
    for (int p = 0; p < m; ++p)
      for (int q = p + 1; q < m; ++q) {
        const double apq = M[(size_t)p * m + q];
        if (apq == 0.0) continue;
        const double th = 0.5 * (M[(size_t)q * m + q] - M[(size_t)p * m + p]) / apq;
        const double t = (th >= 0 ? 1.0 : -1.0) / (std::fabs(th) + std::sqrt(th * th + 1.0));
        const double cs = 1.0 / std::sqrt(t * t + 1.0), sn = t * cs;
        for (int k = 0; k < m; ++k) {  // M <- J^T M J, V <- V J
          const double mkp = M[(size_t)k * m + p], mkq = M[(size_t)k * m + q];
          M[(size_t)k * m + p] = cs * mkp - sn * mkq;
          M[(size_t)k * m + q] = sn * mkp + cs * mkq;
        }
        for (int k = 0; k < m; ++k) {
          const double mpk = M[(size_t)p * m + k], mqk = M[(size_t)q * m + k];
          M[(size_t)p * m + k] = cs * mpk - sn * mqk;
          M[(size_t)q * m + k] = sn * mpk + cs * mqk;
        }
        for (int k = 0; k < m; ++k) {
          const double vkp = V[(size_t)k * m + p], vkq = V[(size_t)k * m + q];
          V[(size_t)k * m + p] = cs * vkp - sn * vkq;
          V[(size_t)k * m + q] = sn * vkp + cs * vkq;
        }
      }
  }
  int lo = 0;
  for (int i = 1; i < m; ++i)
    if (M[(size_t)i * m + i] < M[(size_t)lo * m + lo]) lo = i;
  *eig = M[(size_t)lo * m + lo];
  // c = L^-T y (back substitution), y = column lo of V
  for (int i = m - 1; i >= 0; --i) {
    double v = V[(size_t)i * m + lo];
    for (int k = i + 1; k < m; ++k) v -= L[(size_t)k * m + i] * vec[k];
    vec[i] = v / L[(size_t)i * m + i];
  }
  int big = 0;
  for (int i = 1; i < m; ++i)
    if (std::fabs(vec[i]) > std::fabs(vec[big])) big = i;
  if (vec[big] < 0.0)
    for (int i = 0; i < m; ++i) vec[i] = -vec[i];
  return true;
}

static int spin_context(vsvb_context* c, const double* coeff) {
  if (c->npair == 0) return fail(VSVB_ERR_ARG, "the wave function has no spin-coupled pairs");
  int rc;
  HIP_OK(hipSetDevice(c->device));
  if ((rc = prepare_geometry(c, nullptr))) return rc;
  return prepare_orbital_basis(c, coeff, nullptr);
}

int vsvb_spin_matrices(vsvb_context* c, const double* coeff, double* ham, double* ovl) {
  if (!c || !ham || !ovl) return fail(VSVB_ERR_ARG, "null argument");
  int rc;
  if ((rc = spin_context(c, coeff))) return rc;
  return sc_matrices(c, ham, ovl);
}

int vsvb_spin_opt(vsvb_context* c, const double* coeff, double* energy, double* coeff_sc) {
  if (!c || !energy || !coeff_sc) return fail(VSVB_ERR_ARG, "null argument");
  int rc;
  if ((rc = spin_context(c, coeff))) return rc;
  const int m = c->sc.nspinc;
  std::vector<double> H((size_t)m * m), S((size_t)m * m);
  if ((rc = sc_matrices(c, H.data(), S.data()))) return rc;
  double eig = 0.0;
  if (!lowest_root(m, H, S, &eig, coeff_sc))
    return fail(VSVB_ERR_NUMERIC, "overlap matrix of the spin couplings is not positive definite");
  *energy = eig + c->enuc;
  return VSVB_OK;
}

int vsvb_set_spin_coupling(vsvb_context* c, const double* coeff_sc) {
  if (!c || !coeff_sc) return fail(VSVB_ERR_ARG, "null argument");
  if (c->npair == 0) return fail(VSVB_ERR_ARG, "the wave function has no spin-coupled pairs");
  for (int i = 0; i < c->sc.nspinc; ++i)
    if (!std::isfinite(coeff_sc[i])) return fail(VSVB_ERR_ARG, "non-finite spin-coupling weight");
  HIP_OK(hipSetDevice(c->device));
  return sc_set_coupling(c, coeff_sc);
}

int vsvb_debug_gemm(int32_t M, int32_t N, int32_t K, int32_t ta, int32_t tb, double alpha, const double* A,
                    const double* B, double beta, double* C) {
  if (M < 1 || N < 1 || K < 1 || !A || !B || !C) return fail(VSVB_ERR_ARG, "invalid GEMM probe arguments");
  const size_t na = (size_t)M * K, nb = (size_t)K * N, nc = (size_t)M * N;
  DevBuf<double> dA, dB, dC;
  HIP_OK(dA.alloc(na));
  HIP_OK(dB.alloc(nb));
  HIP_OK(dC.alloc(nc));
  HIP_OK(hipMemcpy(dA.p, A, na * sizeof(double), hipMemcpyHostToDevice));
  HIP_OK(hipMemcpy(dB.p, B, nb * sizeof(double), hipMemcpyHostToDevice));
  HIP_OK(hipMemcpy(dC.p, C, nc * sizeof(double), hipMemcpyHostToDevice));
  // row-major storage: op(A) is M x K, so A is stored K x M when transposed
  HIP_OK(gemm(nullptr, M, N, K, alpha, dA.p, ta ? M : K, ta != 0, dB.p, tb ? K : N, tb != 0, beta, dC.p, N));
  HIP_OK(hipMemcpy(C, dC.p, nc * sizeof(double), hipMemcpyDeviceToHost));
  return VSVB_OK;
}

int vsvb_debug_plan(const vsvb_system* sys, const vsvb_options* opt, int32_t ncu, double* plan, int64_t* partial) {
  if (!sys || ncu < 1 || !plan || !partial) return fail(VSVB_ERR_ARG, "invalid plan probe arguments");
  vsvb_context c;  // host state only
  c.own_stream = false;
  HostBasis hb;
  int rc;
  if ((rc = read_options(sys, opt, &c))) return rc;
  if ((rc = describe_system(sys, opt, &c, hb))) return rc;
  c.ncu = ncu;
  if (plan_lists(&c) > 0) c.nlevels = kLevels;
  partial[1] = (int64_t)partial_slots(&c);
  if ((rc = plan_work(&c, nullptr))) return rc;
  const size_t unscreened = c.partial_total;
  if ((rc = order_pairs(&c))) return rc;
  partial[0] = (int64_t)std::max(unscreened, c.partial_total);
  for (int m = 0; m < 2; ++m)
    for (int q = 0; q < kNQuartetClass; ++q) {
      const ClassLaunch& l = m ? c.ljk[q] : c.le[q];
      const double row[8] = {(double)l.coop, (double)l.lb, (double)l.lk, (double)l.units, (double)l.blocks,
                             l.coop ? (double)l.claim : (double)l.kchunk, (double)l.tr, (double)c.in_small[m][q]};
      std::copy(row, row + 8, plan + (m * kNQuartetClass + q) * 8);
    }
  return VSVB_OK;
}

int vsvb_debug_stored(const vsvb_system* sys, const vsvb_options* opt, int32_t nwfn) {
  if (!sys || nwfn < 1) return fail(VSVB_ERR_ARG, "invalid stored-integral probe arguments");
  vsvb_context c;  // host state only
  c.own_stream = false;
  HostBasis hb;
  StoredIntegrals s;
  int rc;
  if ((rc = read_options(sys, opt, &c))) return rc;
  if ((rc = describe_system(sys, opt, &c, hb))) return rc;
  (void)hipSetDevice(c.device);
  if (c.npair > 0)
    stored_setup(&c, s, 0, 0, kStoredBytes);
  else
    stored_setup(&c, s, nwfn, c.nunpd > 0 ? 2 : 1, kStoredGroupBytes);
  return s.M.p ? 1 : 0;
}

const char* vsvb_last_error(void) { return g_last_error.c_str(); }

const char* vsvb_version(void) { return "vsvb-mi355x 0.1 (gfx950, FP64 OS/HGP)"; }

int vsvb_context_create(const vsvb_system* sys, const vsvb_options* opt, vsvb_context** ctx) {
  if (!ctx) return fail(VSVB_ERR_ARG, "null ctx pointer");
  *ctx = nullptr;
  auto* c = new vsvb_context();
  const int rc = build_context(sys, opt, c);
  if (rc != VSVB_OK) {
    vsvb_context_destroy(c);
    return rc;
  }
  *ctx = c;
  return VSVB_OK;
}

void vsvb_context_destroy(vsvb_context* c) {
  if (!c) return;
  (void)hipSetDevice(c->device);
  if (c->side) (void)hipStreamSynchronize(c->side);
  if (c->stream) (void)hipStreamSynchronize(c->stream);
  if (c->ev0) (void)hipEventDestroy(c->ev0);
  if (c->ev1) (void)hipEventDestroy(c->ev1);
  if (c->ev_fork) (void)hipEventDestroy(c->ev_fork);
  if (c->ev_join) (void)hipEventDestroy(c->ev_join);
  if (c->side) (void)hipStreamDestroy(c->side);
  if (c->ev_in) (void)hipEventDestroy(c->ev_in);
  if (c->ev_out) (void)hipEventDestroy(c->ev_out);
  hipStream_t st = c->own_stream ? c->stream : nullptr;
  delete c;
  if (st) (void)hipStreamDestroy(st);
}

int vsvb_energy(vsvb_context* c, const double* coords, const double* coeff, double* energy, double* parts) {
  if (!c) return fail(VSVB_ERR_ARG, "null context");
  return energy_impl(c, coords, coeff, energy, parts);
}

int vsvb_energy_parts(vsvb_context* c, const double* coeff, double* num, double* wfnorm) {
  double parts[4];
  const int rc = vsvb_energy(c, nullptr, coeff, nullptr, parts);
  if (rc) return rc;
  if (num) *num = parts[0];
  if (wfnorm) *wfnorm = parts[1];
  return VSVB_OK;
}

int vsvb_energy_grad(vsvb_context* c, const double* coords, const double* coeff, double* energy, double* grad) {
  if (!c) return fail(VSVB_ERR_ARG, "null context");
  HIP_OK(hipSetDevice(c->device));
  int rc;
  if (c->npair > 0) {
    if ((rc = prepare_geometry(c, coords))) return rc;
    if ((rc = prepare_orbital_basis(c, coeff, nullptr))) return rc;
    if ((rc = sc_enqueue(c, true, c->d_grad.p))) return rc;
    return sc_finish(c, energy, nullptr, grad);
  }
  rc = enqueue_energy_grad(c, coords, coeff, nullptr, c->d_grad.p);
  if (rc) return rc;
  return finish_energy_grad(c, energy, grad);
}

int vsvb_energy_grad_static(const vsvb_system* sys, const vsvb_options* opt, double* energy, double* grad) {
  if (!sys || !energy) return fail(VSVB_ERR_ARG, "null argument");
  if (sys->npair > 0)
    return fail(VSVB_ERR_UNSUPPORTED, "the allocation-free entry covers wave functions without spin-coupled pairs "
                                      "(npair = 0); use vsvb_context_create and vsvb_energy_grad");
  const int dev = opt ? opt->device : 0;
  if (dev < 0 || dev >= kScratchDevices) return fail(VSVB_ERR_ARG, "device ordinal out of range");
  HIP_OK(hipSetDevice(dev));
  std::lock_guard<std::mutex> lk(g_scratch_mu[dev]);
  if (!g_scratch_ptr[dev]) {  // once per device, with that device current
    void* p = nullptr;
    HIP_OK(hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)));
    g_scratch_ptr[dev] = p;
  }
  vsvb::Arena arena;
  arena.base = static_cast<char*>(g_scratch_ptr[dev]);
  arena.cap = kScratchBytes;
  vsvb_context c;  // transient: no stream, no events, every device buffer in the arena
  c.arena = &arena;
  c.own_stream = false;
  int rc = build_context(sys, opt, &c);
  if (rc != VSVB_OK && arena.need > arena.cap)
    return fail(VSVB_ERR_UNSUPPORTED, "the system needs more than the " + std::to_string(kScratchBytes >> 20) +
                                          " MiB of device scratch the allocation-free entry holds (" +
                                          std::to_string(arena.need >> 20) + " MiB requested before it ran out); "
                                          "use vsvb_context_create and vsvb_energy_grad");
  if (rc != VSVB_OK) return rc;
  if ((rc = enqueue_energy_grad(&c, nullptr, nullptr, nullptr, c.d_grad.p))) return rc;
  return finish_energy_grad(&c, energy, grad);
}

int vsvb_energy_grad_device(vsvb_context* c, const double* coeff_device, double* energy_device, double* grad_device,
                            void* stream) {
  if (!c || !coeff_device || !energy_device || !grad_device) return fail(VSVB_ERR_ARG, "null argument");
  HIP_OK(hipSetDevice(c->device));
  hipStream_t caller = (hipStream_t)stream;
  // the caller's earlier work (that produced coeff) -> the context stream -> the caller's later work
  HIP_OK(hipEventRecord(c->ev_in, caller));
  HIP_OK(hipStreamWaitEvent(c->stream, c->ev_in, 0));
  int rc;
  if ((rc = prepare_geometry(c, nullptr))) return rc;
  if (c->npair > 0) {
    if ((rc = prepare_orbital_basis(c, nullptr, coeff_device))) return rc;
    if ((rc = sc_enqueue(c, true, grad_device))) return rc;
    HIP_OK(hipMemcpyAsync(energy_device, c->d_scal.p + 2, sizeof(double), hipMemcpyDeviceToDevice, c->stream));
  } else {
    if ((rc = prepare_orbitals(c, nullptr, coeff_device, 2))) return rc;
    if ((rc = run_quartets(c, true))) return rc;
    if ((rc = gradient_impl(c, grad_device))) return rc;
    hipLaunchKernelGGL(k_final_energy, dim3(1), dim3(1), 0, c->stream, c->d_scal.p, c->d_scal.p + 3, c->enuc,
                       energy_device);
    HIP_OK(hipGetLastError());
  }
  HIP_OK(hipEventRecord(c->ev_out, c->stream));
  HIP_OK(hipStreamWaitEvent(caller, c->ev_out, 0));
  // numerical status (singular blocks, masked shells) is known only after the work ran
  if ((rc = fetch_out(c, false))) return rc;
  if ((rc = check_status(c, true))) return rc;
  if (c->npair > 0 && reinterpret_cast<const int*>(c->h_out.data() + kOutStatus)[3])
    return fail(VSVB_ERR_UNSUPPORTED, "gradient at a singular spin-coupled transition overlap");
  return finish_counters(c);
}

int vsvb_debug_buffer(vsvb_context* c, const char* name, double* out, int64_t n) {
  if (!c || !name || !out) return fail(VSVB_ERR_ARG, "null argument");
  struct { const char* nm; const DevBuf<double>* b; } tab[] = {
      {"S_ao", &c->d_S}, {"h_ao", &c->d_H}, {"C", &c->d_Ct}, {"C_eri", &c->d_Cs}, {"S_orb", &c->d_Sorb},
      {"h_orb", &c->d_Horb}, {"P", &c->d_P}, {"R", &c->d_R}, {"J", &c->d_J}, {"K", &c->d_K}, {"F", &c->d_F},
      {"gradC", &c->d_gradC}, {"scalars", &c->d_scal}};
  for (auto& t : tab)
    if (!std::strcmp(t.nm, name)) {
      if ((size_t)n > t.b->n) return fail(VSVB_ERR_ARG, "request larger than the buffer");
      HIP_OK(hipStreamSynchronize(c->stream));
      HIP_OK(hipMemcpy(out, t.b->p, n * sizeof(double), hipMemcpyDeviceToHost));
      return VSVB_OK;
    }
  return fail(VSVB_ERR_ARG, std::string("unknown buffer ") + name);
}

int vsvb_set_profiling(vsvb_context* c, int32_t on) {
  if (!c) return fail(VSVB_ERR_ARG, "null context");
  HIP_OK(hipSetDevice(c->device));
  c->profile = on != 0;
  return VSVB_OK;
}

int vsvb_batch_set_profiling(vsvb_batch* b, int32_t on) {
  if (!b) return fail(VSVB_ERR_ARG, "null batch");
  // a captured graph holds the per-class event nodes of the switch it was
  // captured with: release it, the next run is direct and captures again
  if (b->exec && (on != 0) != b->ctx[0]->profile) {
    HIP_OK(hipSetDevice(b->ctx[0]->device));
    HIP_OK(hipStreamSynchronize(b->stream));
    HIP_OK(hipGraphExecDestroy(b->exec));
    b->exec = nullptr;
  }
  for (auto* c : b->ctx) {
    const int rc = vsvb_set_profiling(c, on);
    if (rc) return rc;
  }
  return VSVB_OK;
}

/* Sum of the per-class statistics of every wave function of the last run; with
   group launches the time and launch columns are those of the launches. */
int vsvb_batch_class_stats(vsvb_batch* b, double* out) {
  if (!b || !out) return fail(VSVB_ERR_ARG, "null argument");
  std::memset(out, 0, sizeof(double) * kNQuartetClass * 6);
  for (auto* c : b->ctx)
    for (int q = 0; q < kNQuartetClass; ++q)
      for (int k = 0; k < 6; ++k) out[q * 6 + k] += c->class_stats[q][k];
  if (b->planned && b->chunks > 0)
    for (int q = 0; q < kNQuartetClass; ++q) {
      out[q * 6] = b->lstats[q][0];
      out[q * 6 + 5] = b->lstats[q][1];
    }
  return VSVB_OK;
}

int vsvb_class_stats(vsvb_context* c, double* out) {
  if (!c || !out) return fail(VSVB_ERR_ARG, "null argument");
  std::memcpy(out, c->class_stats, sizeof(c->class_stats));
  return VSVB_OK;
}

int vsvb_last_counters(vsvb_context* c, double* out4) {
  if (!c || !out4) return fail(VSVB_ERR_ARG, "null argument");
  std::memcpy(out4, c->last_counters, sizeof(c->last_counters));
  return VSVB_OK;
}

int vsvb_batch_create(int32_t nwfn, const vsvb_system* const* systems, const vsvb_options* opt, vsvb_batch** b) {
  if (!b || !systems || nwfn < 1) return fail(VSVB_ERR_ARG, "invalid batch arguments");
  *b = nullptr;
  std::unique_ptr<vsvb_batch> own(new vsvb_batch());  // released on every failure path
  vsvb_batch* bt = own.get();
  HIP_OK(hipSetDevice(opt ? opt->device : 0));
  HIP_OK(hipStreamCreateWithFlags(&bt->stream, hipStreamNonBlocking));
  for (int i = 0; i < nwfn; ++i) {
    auto* c = new vsvb_context();
    c->stream = bt->stream;
    c->own_stream = false;
    const int rc = build_context(systems[i], opt, c);
    if (rc) {
      g_last_error = "wave function " + std::to_string(i) + ": " + g_last_error;
      vsvb_context_destroy(c);
      return rc;
    }
    bt->ctx.push_back(c);
  }
  // group wave functions that share the molecule
  std::vector<int> gid(nwfn, -1);
  for (int i = 0; i < nwfn; ++i) {
    if (gid[i] >= 0) continue;
    gid[i] = (int)bt->groups.size();
    bt->groups.emplace_back();
    bt->groups.back().members.push_back(i);
    for (int j = i + 1; j < nwfn; ++j)
      if (gid[j] < 0 && same_molecule(systems[i], systems[j])) {
        gid[j] = gid[i];
        bt->groups.back().members.push_back(j);
      }
  }
  // group streams
  const int nl = std::min<int>(kBatchLanes, (int)bt->groups.size());
  HIP_OK(hipEventCreateWithFlags(&bt->ev_fork, hipEventDisableTiming));
  for (int k = 0; k < nl; ++k) {
    hipStream_t s = nullptr;
    HIP_OK(hipStreamCreateWithFlags(&s, hipStreamNonBlocking));
    bt->lanes.push_back(s);
    hipEvent_t e = nullptr;
    HIP_OK(hipEventCreateWithFlags(&e, hipEventDisableTiming));
    bt->ev_join.push_back(e);
  }
  assign_lanes(bt, nl);
  for (auto& g : bt->groups) {
    vsvb_context* lead = bt->ctx[g.members[0]];
    if (g.members.size() < 2) continue;
    if ((int)g.members.size() >= kStoredMembers && lead->npair == 0 && lead->pair_chunk == 0)
      stored_setup(lead, g.stored, (int)g.members.size(), lead->nunpd > 0 ? 2 : 1, kStoredGroupBytes);
    // its work lists are planned with the first geometry
    lead->ndens = g.stored.M.p ? 1 : (int)g.members.size();
    const size_t nn = (size_t)lead->nbf * lead->nbf;
    const int nspin = lead->nunpd > 0 ? 2 : 1;
    const size_t G = g.members.size();
    HIP_OK(g.dens.alloc(G * nspin * nn));
    HIP_OK(g.jacc.alloc(G * nn));
    HIP_OK(g.kacc.alloc(G * nspin * nn));
    for (size_t k = 0; k < G; ++k) {
      vsvb_context* m = bt->ctx[g.members[k]];
      if (k > 0) share_geometry(lead, m);
      m->d_R.alias(g.dens.p + k * nspin * nn, nspin * nn);
      m->d_J.alias(g.jacc.p + k * nn, nn);
      m->d_K.alias(g.kacc.p + k * nspin * nn, nspin * nn);
    }
  }
  // gather arrays for graph replays
  bt->goff.assign(nwfn + 1, 0);
  for (int i = 0; i < nwfn; ++i) bt->goff[i + 1] = bt->goff[i] + std::max(1, bt->ctx[i]->totlen);
  bt->ran.assign(nwfn, 0);
  HIP_OK(bt->d_e.alloc(nwfn));
  HIP_OK(bt->d_g.alloc(bt->goff[nwfn]));
  HIP_OK(bt->d_st.alloc(4 * (size_t)nwfn));
  HIP_OK(bt->d_cnt.alloc((size_t)kCnt * nwfn));
  HIP_OK(hipHostMalloc((void**)&bt->h_e, nwfn * sizeof(double), hipHostMallocDefault));
  HIP_OK(hipHostMalloc((void**)&bt->h_g, bt->goff[nwfn] * sizeof(double), hipHostMallocDefault));
  HIP_OK(hipHostMalloc((void**)&bt->h_st, 4 * (size_t)nwfn * sizeof(int), hipHostMallocDefault));
  HIP_OK(hipHostMalloc((void**)&bt->h_cnt, (size_t)kCnt * nwfn * sizeof(unsigned long long), hipHostMallocDefault));
  *b = own.release();
  return VSVB_OK;
}

int vsvb_batch_run(vsvb_batch* b, int32_t want_grad, double* energies, double* const* grads) {
  if (!b) return fail(VSVB_ERR_ARG, "null batch");
  int rc;
  HIP_OK(hipSetDevice(b->ctx[0]->device));
  if (!b->tuned) {
    b->tuned = true;
    if ((rc = tune_batch(b))) return rc;
  }
  ++b->runs;
  if (b->exec) {
    if ((rc = batch_replay(b, want_grad, energies, grads))) return rc;
    return batch_launch_stats(b);
  }
  if ((rc = batch_plan(b))) return rc;
  if ((rc = batch_enqueue(b))) return rc;
  for (size_t i = 0; i < b->ctx.size(); ++i) {
    vsvb_context* c = b->ctx[i];
    double* e = energies ? energies + i : nullptr;
    double* g = (want_grad && grads) ? grads[i] : nullptr;
    if ((rc = c->npair > 0 ? sc_finish(c, e, nullptr, g) : finish_energy_grad(c, e, g))) return rc;
  }
  if ((rc = batch_launch_stats(b))) return rc;
  // capturing runs nothing: the graph is built now, after the first (direct) run,
  // and replayed from the next run on; on failure runs stay direct
  if (!b->graph_failed && !b->graph_off && !b->graph_hold) (void)batch_capture(b);
  b->graph_hold = false;
  return VSVB_OK;
}

int vsvb_batch_set_coords(vsvb_batch* b, const double* coords) {
  if (!b || !coords) return fail(VSVB_ERR_ARG, "null argument");
  const size_t n = b->ctx.size();
  std::vector<size_t> off(n + 1, 0);
  for (size_t i = 0; i < n; ++i) off[i + 1] = off[i] + 3 * (size_t)b->ctx[i]->natom;
  for (size_t i = 0; i < off[n]; ++i)
    if (!std::isfinite(coords[i])) return fail(VSVB_ERR_ARG, "non-finite coordinate");
  // wave functions that share one quartet pass share one geometry
  for (auto& g : b->groups)
    for (size_t k = 1; k < g.members.size(); ++k)
      if (std::memcmp(coords + off[g.members[k]], coords + off[g.members[0]], 3 * sizeof(double) *
                      b->ctx[g.members[0]]->natom) != 0)
        return fail(VSVB_ERR_ARG, "wave functions " + std::to_string(g.members[0]) + " and " +
                                      std::to_string(g.members[k]) +
                                      " were created on one geometry and share its quartet pass: give them the same "
                                      "coordinates");
  HIP_OK(hipSetDevice(b->ctx[0]->device));
  HIP_OK(hipStreamSynchronize(b->stream));
  for (auto s : b->lanes) HIP_OK(hipStreamSynchronize(s));
  for (size_t i = 0; i < n; ++i) b->ctx[i]->coords.assign(coords + off[i], coords + off[i + 1]);
  // a captured graph holds the old nuclear repulsion and skips the coordinate upload
  if (b->exec) {
    HIP_OK(hipGraphExecDestroy(b->exec));
    b->exec = nullptr;
  }
  b->graph_hold = true;
  return VSVB_OK;
}

// calcsurface (src/valence_api_nitrogen.F90:17-27): coordinates in angstrom
// (tools_module angs2bohr factor), energy in cm^-1.
constexpr double kAngs2Bohr = 1.889725987722;
constexpr double kHartree2Wavenumber = 219474.631;

int vsvb_surface(vsvb_context* c, const double* x_angstrom, double* v_cm1) {
  if (!c || !x_angstrom || !v_cm1) return fail(VSVB_ERR_ARG, "null argument");
  std::vector<double> x(3 * (size_t)c->natom);
  for (size_t i = 0; i < x.size(); ++i) x[i] = x_angstrom[i] * kAngs2Bohr;
  double e = 0.0;
  const int rc = vsvb_energy(c, x.data(), nullptr, &e, nullptr);
  if (rc) return rc;
  *v_cm1 = e * kHartree2Wavenumber;
  return VSVB_OK;
}

int vsvb_surface_batch(vsvb_batch* b, const double* x_angstrom, double* v_cm1) {
  if (!b || !x_angstrom || !v_cm1) return fail(VSVB_ERR_ARG, "null argument");
  size_t tot = 0;
  for (auto* c : b->ctx) tot += 3 * (size_t)c->natom;
  std::vector<double> x(tot);
  for (size_t i = 0; i < tot; ++i) x[i] = x_angstrom[i] * kAngs2Bohr;
  int rc;
  if ((rc = vsvb_batch_set_coords(b, x.data()))) return rc;
  if ((rc = vsvb_batch_run(b, 0, v_cm1, nullptr))) return rc;
  for (size_t i = 0; i < b->ctx.size(); ++i) v_cm1[i] *= kHartree2Wavenumber;
  return VSVB_OK;
}

int vsvb_batch_set_lanes(vsvb_batch* b, int32_t n) {
  if (!b) return fail(VSVB_ERR_ARG, "null batch");
  if (n < 1) return fail(VSVB_ERR_ARG, "lane count must be at least 1");
  const int nl = std::min<int>(n, (int)b->lanes.size());
  HIP_OK(hipStreamSynchronize(b->stream));
  for (auto s : b->lanes) HIP_OK(hipStreamSynchronize(s));
  if (b->exec) {
    HIP_OK(hipGraphExecDestroy(b->exec));
    b->exec = nullptr;
  }
  assign_lanes(b, nl);
  return VSVB_OK;
}

/* The last run's group launches, rows of 6: class, kernel (0 straight-line, 1
   straight-line transposed, 2 cooperative), groups, stream, ms, FLOPs. */
int vsvb_batch_launches(vsvb_batch* b, double* out, int32_t cap, int32_t* n) {
  if (!b || !n || (cap > 0 && !out)) return fail(VSVB_ERR_ARG, "null argument");
  const bool on = b->planned && b->chunks > 0;
  *n = on ? (int32_t)b->glaunch.size() : 0;
  for (int32_t r = 0; r < std::min(*n, cap); ++r) {
    const GroupLaunch& L = b->glaunch[r];
    double* o = out + 6 * (size_t)r;
    o[0] = L.q;
    o[1] = L.coop_idx >= 0 ? 2 : (L.tr ? 1 : 0);
    o[2] = L.ng;
    o[3] = L.lane;
    o[4] = L.ms;
    o[5] = L.flops;
  }
  return VSVB_OK;
}

int vsvb_batch_set_group_launch(vsvb_batch* b, int32_t chunks) {
  if (!b) return fail(VSVB_ERR_ARG, "null batch");
  if (chunks < 0 || chunks > 64) return fail(VSVB_ERR_ARG, "group-launch chunks per lane must be 0..64");
  HIP_OK(hipSetDevice(b->ctx[0]->device));
  HIP_OK(hipStreamSynchronize(b->stream));
  for (auto s : b->lanes) HIP_OK(hipStreamSynchronize(s));
  if (b->exec) {
    HIP_OK(hipGraphExecDestroy(b->exec));
    b->exec = nullptr;
  }
  b->chunks = chunks;
  b->planned = false;
  return VSVB_OK;
}

int vsvb_batch_set_graph(vsvb_batch* b, int32_t on) {
  if (!b) return fail(VSVB_ERR_ARG, "null batch");
  b->graph_off = on == 0;
  if (b->graph_off && b->exec) {
    HIP_OK(hipStreamSynchronize(b->stream));
    HIP_OK(hipGraphExecDestroy(b->exec));
    b->exec = nullptr;
  }
  return VSVB_OK;
}

int vsvb_batch_tuning(vsvb_batch* b, double* out) {
  if (!b || !out) return fail(VSVB_ERR_ARG, "null argument");
  std::memcpy(out, b->tuning, sizeof(b->tuning));
  return VSVB_OK;
}

int vsvb_batch_stored_groups(vsvb_batch* b) {
  if (!b) return fail(VSVB_ERR_ARG, "null batch");
  return (int)std::count_if(b->groups.begin(), b->groups.end(), [](const BatchGroup& g) { return g.stored.M.p != nullptr; });
}

int vsvb_batch_uses_graph(vsvb_batch* b) {
  if (!b) return fail(VSVB_ERR_ARG, "null batch");
  if (b->graph_failed) g_last_error = "graph capture failed: " + b->graph_error;
  return b->exec ? 1 : 0;
}

void vsvb_batch_destroy(vsvb_batch* b) { delete b; }

}  // extern "C"

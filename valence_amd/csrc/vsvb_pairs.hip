// What a new geometry needs of every shell pair: its primitive pairs, its block of
// the one-electron matrices, its Schwarz bound.  Small systems run all of it in two
// launches (thirteen before): a class of a few hundred pairs is a launch of 5 to 25
// us whose wavefronts fill a corner of the chip.
#include "vsvb_internal.h"

namespace vsvb {

namespace {

// ---------------------------------------------------------------------------
// primitive pairs
// ---------------------------------------------------------------------------

// One wavefront per shell pair, a lane per primitive pair, for the vector between
// the centres and the primitive pairs kept by the screen: those with
// |K_ab| > kPrimCut (K carries the contraction weights and exp(-ab/(a+b) |AB|^2)),
// in their order; their number becomes the pair's npp.  A dropped primitive pair
// changes any ERI by less than kPrimCut * (the largest K) * (a bounded Boys/angular
// factor).  Measured: at 1e-14 every energy of the oracle fixtures (C8H18, C12H26,
// H12, LiF8, the reference's inputs) is the same as at 1e-20 to 1e-13 Eh, and the
// C8H18 J/K pass drops 10% of its primitive quartets' time; 1e-13 starts to move
// C12H26's energy (7e-12 Eh).  K does not depend on the orbital weights, so the
// weight gradient stays the exact derivative of the screened energy.
//
// Bounded by one chain of loads and an exp: C8H18 8 us; in three launches,
// the screen a thread per shell pair walking its list, 61.
__global__ void __launch_bounds__(256) k_pairs(PairArgs a) {
  const int t = __builtin_amdgcn_readfirstlane((int)(blockIdx.x * 4 + (threadIdx.x >> 6))), lane = threadIdx.x & 63;
  if (t >= a.off[kNPairClass]) return;  // whole wavefront
  const PairSrc P = a.src[a.order[t]];
  const Shell A = a.shells[P.A], B = a.shells[P.B];
  const double Ax = a.xyz[3 * A.atom], Ay = a.xyz[3 * A.atom + 1], Az = a.xyz[3 * A.atom + 2];
  const double Bx = a.xyz[3 * B.atom], By = a.xyz[3 * B.atom + 1], Bz = a.xyz[3 * B.atom + 2];
  const double ABx = Ax - Bx, ABy = Ay - By, ABz = Az - Bz;
  int kept = 0;
  for (int i0 = 0; i0 < A.nprim * B.nprim; i0 += 64) {
    const int i = i0 + lane;
    PrimPair o{};
    bool keep = false;
    if (i < A.nprim * B.nprim) {
      const int ia = A.prim0 + i / B.nprim, ib = B.prim0 + i % B.nprim;
      const double x = a.pexp[ia], y = a.pexp[ib], p = x + y, rp = 1.0 / p;
      o.p = p;
      o.oo2p = 0.5 * rp;
      o.Px = (x * Ax + y * Bx) * rp;
      o.Py = (x * Ay + y * By) * rp;
      o.Pz = (x * Az + y * Bz) * rp;
      o.PAx = o.Px - Ax;
      o.PAy = o.Py - Ay;
      o.PAz = o.Pz - Az;
      o.K = a.pcoef[ia] * a.pcoef[ib] * exp(-x * y * rp * (ABx * ABx + ABy * ABy + ABz * ABz)) * rp * a.kfold;
      o.pad = 0.0;
      keep = fabs(o.K) > kPrimCut;
    }
    const unsigned long long m = __ballot(keep);
    if (keep) a.pp[P.pp0 + kept + __popcll(m & ((1ull << lane) - 1))] = o;
    kept += __popcll(m);
  }
  if (lane == 0) {
    int cl = 0;
    while (t >= a.off[cl + 1]) ++cl;
    a.pairs[t] = Pair{P.A, P.B, P.pp0, kept, a.fun[cl] + t - a.off[cl], 0, ABx, ABy, ABz, 0.0};
  }
}

// ---------------------------------------------------------------------------
// device: one-electron integrals (Obara-Saika), one wavefront per shell pair
// ---------------------------------------------------------------------------
// cartesian tuples of total order 0..4 in CCA order, cumulative index
__device__ __forceinline__ constexpr int cart_off(int l) { return l * (l + 1) * (l + 2) / 6; }
__device__ __forceinline__ constexpr int cart_idx(int lx, int ly, int lz) {
  return cart_off(lx + ly + lz) + ((ly + lz) * (ly + lz + 1)) / 2 + lz;
}
__device__ __forceinline__ void cart_of(int l, int c, int& lx, int& ly, int& lz) {
  int i = 0;
  while ((i + 1) * (i + 2) / 2 <= c) ++i;
  const int j = c - i * (i + 1) / 2;
  lx = l - i;
  ly = i - j;
  lz = j;
}

// The lanes of the wavefront take the (primitive pair, nuclear centre) items of
// the pair in turn; the item of centre 0 also adds the primitive pair's overlap
// and kinetic terms.  Lane sums are reduced across the wavefront at the end.
template <int LA, int LB>
__device__ __forceinline__ void one_e(const PairArgs& g, int t) {
  constexpr int NA = ncart(LA), NB = ncart(LB), L = LA + LB;
  constexpr int NE = cart_off(L + 1);        // cartesians of order 0..L
  constexpr int NBc = cart_off(LB + 1);      // cartesians of order 0..LB
  const int lane = threadIdx.x & 63, natom = g.natom, nbf = g.nbf;
  const Shell* __restrict__ shells = g.shells;
  const double *__restrict__ pexp = g.pexp, *__restrict__ pcoef = g.pcoef, *__restrict__ xyz = g.xyz,
               *__restrict__ charge = g.charge, *__restrict__ boys = g.boys;
  double *__restrict__ S = g.S, *__restrict__ H = g.H;
  const Pair PR = g.pairs[t];
  const Shell A = shells[PR.A], B = shells[PR.B];
  const double Ax = xyz[3 * A.atom], Ay = xyz[3 * A.atom + 1], Az = xyz[3 * A.atom + 2];
  const double Bx = xyz[3 * B.atom], By = xyz[3 * B.atom + 1], Bz = xyz[3 * B.atom + 2];
  const double AB[3] = {Ax - Bx, Ay - By, Az - Bz};
  double s[NA * NB], tk[NA * NB], v[NA * NB];
#pragma unroll
  for (int k = 0; k < NA * NB; ++k) s[k] = tk[k] = v[k] = 0.0;
  const int nitem = A.nprim * B.nprim * natom;
  for (int item = lane; item < nitem; item += 64) {
    const int ipp = item / natom, c = item - ipp * natom;
    const int ia = ipp / B.nprim, ib = ipp - ia * B.nprim;
    {
      const double a = pexp[A.prim0 + ia], b = pexp[B.prim0 + ib], p = a + b, rp = 1.0 / p;
      const double mu = a * b * rp;
      const double cc = pcoef[A.prim0 + ia] * pcoef[B.prim0 + ib];
      const double Pc[3] = {(a * Ax + b * Bx) * rp, (a * Ay + b * By) * rp, (a * Az + b * Bz) * rp};
      const double PA[3] = {Pc[0] - Ax, Pc[1] - Ay, Pc[2] - Az};
      const double PB[3] = {Pc[0] - Bx, Pc[1] - By, Pc[2] - Bz};
      if (c == 0) {
      // 1D overlaps, i <= LA, j <= LB + 2
      double S1[3][LA + 1][LB + 3];
#pragma unroll
      for (int d = 0; d < 3; ++d) {
        S1[d][0][0] = sqrt(M_PI * rp) * exp(-mu * AB[d] * AB[d]);
#pragma unroll
        for (int i = 0; i <= LA; ++i)
#pragma unroll
          for (int j = 0; j <= LB + 2; ++j) {
            if (i == 0 && j == 0) continue;
            double val;
            if (i > 0) {
              val = PA[d] * S1[d][i - 1][j];
              if (i > 1) val += (i - 1) * 0.5 * rp * S1[d][i - 2][j];
              if (j > 0) val += j * 0.5 * rp * S1[d][i - 1][j - 1];
            } else {
              val = PB[d] * S1[d][i][j - 1];
              if (j > 1) val += (j - 1) * 0.5 * rp * S1[d][i][j - 2];
            }
            S1[d][i][j] = val;
          }
      }
#pragma unroll
      for (int ca = 0; ca < NA; ++ca)
#pragma unroll
        for (int cb = 0; cb < NB; ++cb) {
          int ax, ay, az, bx, by, bz;
          cart_of(LA, ca, ax, ay, az);
          cart_of(LB, cb, bx, by, bz);
          const int ai[3] = {ax, ay, az}, bj[3] = {bx, by, bz};
          double sv[3], tv[3];
#pragma unroll
          for (int d = 0; d < 3; ++d) {
            const int i = ai[d], j = bj[d];
            sv[d] = S1[d][i][j];
            const double km = j >= 2 ? S1[d][i][j - 2] : 0.0;
            tv[d] = -0.5 * (j * (j - 1) * km - 2.0 * b * (2 * j + 1) * sv[d] + 4.0 * b * b * S1[d][i][j + 2]);
          }
          s[ca * NB + cb] += cc * sv[0] * sv[1] * sv[2];
          tk[ca * NB + cb] += cc * (tv[0] * sv[1] * sv[2] + sv[0] * tv[1] * sv[2] + sv[0] * sv[1] * tv[2]);
        }
      }
      // nuclear attraction of centre c: VRR [e|0]^(m), |e| <= L, then HRR to [a|b]
      const double pre = 2.0 * M_PI * rp * exp(-mu * (AB[0] * AB[0] + AB[1] * AB[1] + AB[2] * AB[2])) * cc;
      {
        const double Z = charge[c];
        if (fabs(Z) <= 1e-12) continue;  // int1e skips |Z| <= 1e-12 (valence.F90:3146)
        const double PC[3] = {Pc[0] - xyz[3 * c], Pc[1] - xyz[3 * c + 1], Pc[2] - xyz[3 * c + 2]};
        double F[L + 1];
        boys_eval<L>(p * (PC[0] * PC[0] + PC[1] * PC[1] + PC[2] * PC[2]), boys, F);
        double Vm[L + 1][NE];
#pragma unroll
        for (int m = 0; m <= L; ++m) Vm[m][0] = -Z * pre * F[m];
#pragma unroll
        for (int l = 1; l <= L; ++l)
#pragma unroll
          for (int c2 = 0; c2 < ncart(l); ++c2) {
            int ex, ey, ez;
            cart_of(l, c2, ex, ey, ez);
            const int e[3] = {ex, ey, ez};
            const int i = ex > 0 ? 0 : (ey > 0 ? 1 : 2);
            int e1[3] = {ex, ey, ez};
            e1[i] -= 1;
            const int i1 = cart_idx(e1[0], e1[1], e1[2]);
            const int nn = e1[i];
            int i2 = 0;
            if (nn > 0) {
              int e2[3] = {e1[0], e1[1], e1[2]};
              e2[i] -= 1;
              i2 = cart_idx(e2[0], e2[1], e2[2]);
            }
            const int ie = cart_off(l) + c2;
#pragma unroll
            for (int m = 0; m <= L - l; ++m) {
              double val = PA[i] * Vm[m][i1] - PC[i] * Vm[m + 1][i1];
              if (nn > 0) val += nn * 0.5 * rp * (Vm[m][i2] - Vm[m + 1][i2]);
              Vm[m][ie] = val;
            }
            (void)e;
          }
        // HRR on b: W[e][b] = W[e+1_i][b-1_i] + AB_i W[e][b-1_i]
        double W[NE][NBc];
#pragma unroll
        for (int ie = 0; ie < NE; ++ie) W[ie][0] = Vm[0][ie];
#pragma unroll
        for (int lb = 1; lb <= LB; ++lb)
#pragma unroll
          for (int cbb = 0; cbb < ncart(lb); ++cbb) {
            int bx, by, bz;
            cart_of(lb, cbb, bx, by, bz);
            const int i = bx > 0 ? 0 : (by > 0 ? 1 : 2);
            int b1[3] = {bx, by, bz};
            b1[i] -= 1;
            const int ib1 = cart_idx(b1[0], b1[1], b1[2]);
            const int ibb = cart_off(lb) + cbb;
#pragma unroll
            for (int le = 0; le <= L - lb; ++le)
#pragma unroll
              for (int ce = 0; ce < ncart(le); ++ce) {
                int ex, ey, ez;
                cart_of(le, ce, ex, ey, ez);
                int ep[3] = {ex, ey, ez};
                ep[i] += 1;
                const int iep = cart_idx(ep[0], ep[1], ep[2]);
                const int iee = cart_off(le) + ce;
                W[iee][ibb] = W[iep][ib1] + AB[i] * W[iee][ib1];
              }
          }
#pragma unroll
        for (int ca = 0; ca < NA; ++ca)
#pragma unroll
          for (int cb = 0; cb < NB; ++cb) v[ca * NB + cb] += W[cart_off(LA) + ca][cart_off(LB) + cb];
      }
    }
  }
#pragma unroll
  for (int ca = 0; ca < NA; ++ca)
#pragma unroll
    for (int cb = 0; cb < NB; ++cb) {
      const double sv = vsvb::wave_sum(s[ca * NB + cb]), hv = vsvb::wave_sum(tk[ca * NB + cb] + v[ca * NB + cb]);
      if (lane == 0) {
        const int mu = A.ao + ca, nu = B.ao + cb;
        S[(size_t)mu * nbf + nu] = sv;
        S[(size_t)nu * nbf + mu] = sv;
        H[(size_t)mu * nbf + nu] = hv;
        H[(size_t)nu * nbf + mu] = hv;
      }
    }
}

// ---------------------------------------------------------------------------
// Schwarz bounds
// ---------------------------------------------------------------------------
// Q = sqrt(max_ab |(ab|ab)|) of a shell pair: one wavefront per pair, the lanes
// split the bra primitive pairs and the partial diagonal integrals are summed
// across the wave.
template <int LA, int LB>
__device__ __forceinline__ void schwarz(const PairArgs& a, int t) {
  constexpr int NAB = ncart(LA) * ncart(LB);
  const int lane = threadIdx.x & 63;
  const Pair P = a.pairs[t];
  double dsum[NAB];
#pragma unroll
  for (int k = 0; k < NAB; ++k) dsum[k] = 0.0;
  for (int b = lane; b < P.npp; b += 64) {
    double v[NAB * NAB];
    eri_block<LA, LB, LA, LB, -1>(a.pp + P.pp0 + b, 1, a.pp + P.pp0, P.npp, P.ABx, P.ABy, P.ABz, P.ABx, P.ABy, P.ABz,
                                  a.boys + kBoysCOff + (size_t)(2 * (LA + LB)) * kBoysCLen, v);
#pragma unroll
    for (int k = 0; k < NAB; ++k) dsum[k] += v[k * NAB + k];
  }
  double m = 0.0;
#pragma unroll
  for (int k = 0; k < NAB; ++k) m = fmax(m, fabs(wave_sum(dsum[k])));
  if (lane == 0) a.pairs[t].Q = sqrt(m);
}

// ---------------------------------------------------------------------------
// launches
// ---------------------------------------------------------------------------
// The work of a launch: kind 2 pc + 1 the Schwarz bounds of pair class pc, 2 pc its
// one-electron integrals.
template <int kKind>
__device__ __forceinline__ void pair_work(const PairArgs& a, int t) {
  constexpr int pc = kKind / 2, LA = pc == 0 ? 0 : (pc < 3 ? 1 : 2), LB = pc - LA * (LA + 1) / 2;
  if constexpr (kKind % 2)
    schwarz<LA, LB>(a, t);
  else
    one_e<LA, LB>(a, t);
}

template <int kKind>
__global__ void __launch_bounds__(256) k_pair_work(PairArgs a) {
  const int t = a.off[kKind / 2] + __builtin_amdgcn_readfirstlane((int)(blockIdx.x * 4 + (threadIdx.x >> 6)));
  if (t >= a.off[kKind / 2 + 1]) return;  // whole wavefront
  pair_work<kKind>(a, t);
}

// Every kind side by side, the longest chains ((dd) first) in front: block0[k] is
// the first workgroup of the k-th in that order.
struct PairBlocks {
  int block0[2 * kNPairClass + 1];
};

__global__ void __launch_bounds__(256) k_pair_all(PairArgs a, PairBlocks s) {
  int k = 0;
  while (blockIdx.x >= (unsigned)s.block0[k + 1]) ++k;  // uniform
  const int kind = 2 * kNPairClass - 1 - k;
  const int t = a.off[kind / 2] +
                __builtin_amdgcn_readfirstlane((int)((blockIdx.x - s.block0[k]) * 4 + (threadIdx.x >> 6)));
  if (t >= a.off[kind / 2 + 1]) return;  // whole wavefront
  switch (kind) {
    case 0: pair_work<0>(a, t); break;
    case 1: pair_work<1>(a, t); break;
    case 2: pair_work<2>(a, t); break;
    case 3: pair_work<3>(a, t); break;
    case 4: pair_work<4>(a, t); break;
    case 5: pair_work<5>(a, t); break;
    case 6: pair_work<6>(a, t); break;
    case 7: pair_work<7>(a, t); break;
    case 8: pair_work<8>(a, t); break;
    case 9: pair_work<9>(a, t); break;
    case 10: pair_work<10>(a, t); break;
    case 11: pair_work<11>(a, t); break;
  }
}

template <int kKind>
void launch_kinds(const PairArgs& a, hipStream_t st) {
  const int np = a.off[kKind / 2 + 1] - a.off[kKind / 2];
  if (np > 0) hipLaunchKernelGGL(k_pair_work<kKind>, dim3((np + 3) / 4), dim3(256), 0, st, a);
  if constexpr (kKind > 0) launch_kinds<kKind - 1>(a, st);
}

// Shell pairs up to which everything shares one launch.  That launch has the
// registers of its largest kind, one wavefront per SIMD, where low angular momenta
// alone have four to eight: water 117 us instead of 234 (the sum of twelve, without
// the gaps), C8H18 98 instead of 279, a slab of 32 atoms (15576 pairs) 193
// instead of 322, one of 64 (62128) 1003 instead of 674.
constexpr int kSharedPairs = 32768;

}  // namespace

hipError_t launch_pairs(const PairArgs& a, hipStream_t st) {
  const int np = a.off[kNPairClass];
  hipLaunchKernelGGL(k_pairs, dim3((np + 3) / 4), dim3(256), 0, st, a);
  if (np <= kSharedPairs) {
    PairBlocks s{};
    for (int k = 0; k < 2 * kNPairClass; ++k) {
      const int pc = (2 * kNPairClass - 1 - k) / 2;
      s.block0[k + 1] = s.block0[k] + (a.off[pc + 1] - a.off[pc] + 3) / 4;
    }
    hipLaunchKernelGGL(k_pair_all, dim3(s.block0[2 * kNPairClass]), dim3(256), 0, st, a, s);
  } else {
    launch_kinds<2 * kNPairClass - 1>(a, st);
  }
  return hipGetLastError();
}

}  // namespace vsvb

// Orbital algebra of closed- and high-spin wave functions of up to kOrbMax
// orbitals, from the weights to the AO densities and from the Fock matrices to the
// weight gradient.
//
// The orbitals of a VSVB wave function are expanded over one or two atoms (20 to
// 30 of C8H18's 210 AOs), so products with C run over an orbital's own entries:
// C S and S_orb cost 0.16 M multiply-adds instead of 1.7 M, R = C^T P C 0.4 M
// instead of 1.7 M, and the gradient needs C F and m x m products only, since
//   dE/dC = 2 P C F (1 - R S) = 2 P (Y - W T),  Y = C F, T = C S, W = (Y C^T) P
// (four dense products of 1.5 M before).  What bounds these kernels is latency:
// dependent phases, and a pivot loop of two barriers a step.  Kernel time of an
// energy and gradient of C8H18: 240 us in 33 launches (products, inverse, traces,
// fills) before, 148 in eight now (the inverse with S_orb 65, the m x m products
// 34); of water's energy 55 us in 17 launches before, 26 in two now.  The wave
// functions of a batch group run side by side in the same launches.
#include "vsvb_internal.h"

namespace vsvb {

namespace {

constexpr int kOrbThreads = 1024;
constexpr int kOrbOneLaunch = 64;

// Sum over the workgroup (every thread gets it); red: one double per wavefront.
__device__ __forceinline__ double block_sum(double v, double* red) {
  v = wave_sum(v);
  __syncthreads();  // the previous sum's values are read
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
  __syncthreads();
  double s = 0.0;
  for (int w = 0; w < (int)(blockDim.x >> 6); ++w) s += red[w];
  return s;
}

// In-place Gauss-Jordan inverse of the SPD matrix M (m x m, m <= kOrbMax, in
// LDS): every thread holds its elements' new values in registers between the
// two barriers of a pivot step.  False at a pivot that is not positive.
__device__ bool invert_lds(double* M, int m) {
  constexpr int kPer = kOrbMax * kOrbMax / kOrbThreads;
  int ei[kPer], ej[kPer];
  double v[kPer];
#pragma unroll
  for (int t = 0; t < kPer; ++t) {
    const int e = threadIdx.x + t * kOrbThreads;
    ei[t] = e < m * m ? e / m : -1;
    ej[t] = e < m * m ? e - ei[t] * m : 0;
  }
  for (int k = 0; k < m; ++k) {
    const double piv = M[k * m + k];
    if (!(piv > 0.0) || !isfinite(piv)) return false;  // the same value in every thread
    const double ip = 1.0 / piv;
#pragma unroll
    for (int t = 0; t < kPer; ++t)
      if (ei[t] >= 0) {
        const int i = ei[t], j = ej[t];
        const double akj = (j == k ? 1.0 : M[k * m + j]) * ip;
        v[t] = i == k ? akj : (j == k ? 0.0 : M[i * m + j]) - M[i * m + k] * akj;
      }
    __syncthreads();
#pragma unroll
    for (int t = 0; t < kPer; ++t)
      if (ei[t] >= 0) M[ei[t] * m + ej[t]] = v[t];
    __syncthreads();
  }
  return true;
}

constexpr int kOrbEntries = 64;

// The threads that share a row: a workgroup, or one wavefront of it.
struct Row {
  int tid, nt;
  bool wave;
  __device__ __forceinline__ void sync() const {
    if (wave) {
      __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
      __builtin_amdgcn_wave_barrier();
    } else {
      __syncthreads();
    }
  }
};
__device__ __forceinline__ Row block_row() { return {(int)threadIdx.x, (int)blockDim.x, false}; }
__device__ __forceinline__ Row wave_row() { return {(int)threadIdx.x & 63, 64, true}; }
// LDS of a row: entries, or rows of the orbitals' matrices.
struct RowScratch {
  double w[2 * kOrbMax];
  int tgt[kOrbEntries];
};

// Orbital p: its effective weights Ct, T = C S and C h, kOrbEntries entries at a time.
__device__ __forceinline__ void orbital_row(const OrbArgs& a, Row r, int p, RowScratch& lds) {
  const int tid = r.tid, nt = r.nt, n = a.nbf;
  double* w = lds.w;
  int* tgt = lds.tgt;
  const int k0 = a.orb_start[p], k1 = a.orb_start[p + 1];
  for (int v = tid; v < n; v += nt) {
    a.Ct[(size_t)p * n + v] = 0.0;
    a.T[(size_t)p * n + v] = 0.0;
    a.TH[(size_t)p * n + v] = 0.0;
  }
  for (int kb = k0; kb < k1; kb += kOrbEntries) {
    const int len = min(kOrbEntries, k1 - kb);
    r.sync();  // the row is zeroed; the previous entries are done with
    for (int k = tid; k < len; k += nt) {
      tgt[k] = a.ent[kb + k].tgt;
      w[k] = a.angn[tgt[k]] * a.coeff[kb + k];
    }
    r.sync();
    for (int k = tid; k < len; k += nt) {
      double x = 0.0;
      bool first = true;  // an AO that an orbital lists twice is written once, with the sum
      for (int l = 0; l < len; ++l)
        if (tgt[l] == tgt[k]) {
          first &= l >= k;
          x += w[l];
        }
      if (first) a.Ct[(size_t)p * n + tgt[k]] += x;
    }
    for (int v = tid; v < n; v += nt) {
      double s = a.T[(size_t)p * n + v], h = a.TH[(size_t)p * n + v];
      for (int k = 0; k < len; ++k) {
        s += w[k] * a.S[(size_t)tgt[k] * n + v];
        h += w[k] * a.H[(size_t)tgt[k] * n + v];
      }
      a.T[(size_t)p * n + v] = s;
      a.TH[(size_t)p * n + v] = h;
    }
  }
}

// S_orb, h_orb, the screened weights Cs, and per spin P and E1.
__device__ void orbital_middle(const OrbArgs& a, double* M, double* red) {
  const int tid = threadIdx.x, n = a.nbf, ns = a.nsp;
  if (tid < 16) a.scal[tid] = 0.0;
  if (tid < 4) a.status[tid] = 0;
  for (int e = tid; e < ns * ns; e += kOrbThreads) {
    const int p = e / ns, q = e - p * ns;
    double s = 0.0, h = 0.0;
    for (int k = a.orb_start[q]; k < a.orb_start[q + 1]; ++k) {
      const int mu = a.ent[k].tgt;
      const double w = a.angn[mu] * a.coeff[k];
      s += w * a.T[(size_t)p * n + mu];
      h += w * a.TH[(size_t)p * n + mu];
    }
    a.Sorb[e] = s;
    a.Horb[e] = h;
  }
  __syncthreads();
  // the reference's per-(orbital, shell) weight screen (k_shell_screen)
  for (int e = tid; e < ns * a.nsh; e += kOrbThreads) {
    const int p = e / a.nsh;
    const Shell S = a.shells[e - p * a.nsh];
    const double* c = a.Ct + (size_t)p * n + S.ao;
    double* cs = a.Cs + (size_t)p * n + S.ao;
    const double inv = 1.0 / a.Sorb[(size_t)p * ns + p];
    double sum = 0.0;
    bool nz = false;
    for (int k = 0; k < ncart(S.l); ++k) {
      const double raw = c[k] / a.angn[S.ao + k];
      sum += raw * raw * inv;
      nz |= c[k] != 0.0;
    }
    const bool keep = sum > a.dtol;
    for (int k = 0; k < ncart(S.l); ++k) cs[k] = keep ? c[k] : 0.0;
    if (nz && !keep) atomicAdd(a.status + 1, 1);
  }
  double e1 = 0.0;
  for (int s = 0; s < a.nspin; ++s) {
    const int off = s == 0 ? 0 : a.nunpd, m = s == 0 ? a.nalpha : a.ndocc;
    if (m == 0) continue;
    __syncthreads();  // the previous spin is done with M
    for (int e = tid; e < m * m; e += kOrbThreads) M[e] = a.Sorb[(size_t)(off + e / m) * ns + off + e % m];
    __syncthreads();
    if (!invert_lds(M, m) && tid == 0) a.status[0] = 1;
    __syncthreads();
    double t = 0.0;
    for (int e = tid; e < m * m; e += kOrbThreads) {
      a.P[(size_t)s * ns * ns + e] = M[e];
      t += a.Horb[(size_t)(off + e / m) * ns + off + e % m] * M[e];
    }
    e1 += (a.nspin == 1 ? 2.0 : 1.0) * block_sum(t, red);
  }
  if (tid == 0) a.scal[0] = e1;
}

// Row mu of R_s = C^T P C: u = (C^T P)[mu][:] over the orbitals that hold AO mu,
// then u C.
__device__ __forceinline__ void density_row(const OrbArgs& a, Row w, int s, int mu, RowScratch& lds) {
  const int tid = w.tid, nt = w.nt, n = a.nbf, ns = a.nsp;
  double* u = lds.w;
  const int off = s == 0 ? 0 : a.nunpd, m = s == 0 ? a.nalpha : a.ndocc;
  const double* P = a.P + (size_t)s * ns * ns;
  double* R = a.R + (size_t)s * n * n + (size_t)mu * n;
  w.sync();  // the previous row is done with u
  for (int q = tid; q < m; q += nt) {
    double x = 0.0;
    for (int k = a.ao_ptr[mu]; k < a.ao_ptr[mu + 1]; ++k) {
      const int o = a.ao_orb[k];
      if (o >= off && o < off + m) x += a.Cs[(size_t)o * n + mu] * P[(size_t)(o - off) * m + q];
    }
    u[q] = x;
  }
  w.sync();
  for (int v = tid; v < n; v += nt) {
    double r = 0.0;
    for (int q = 0; q < m; ++q) r += u[q] * a.Cs[(size_t)(off + q) * n + v];
    R[v] = r;
  }
}

// Up to kOrbOneLaunch AOs a wave function is one workgroup of one launch, a
// wavefront per row (a row is at most a load per lane; water's front 21 us, where
// three launches and their gaps take as long by themselves); above, the stages are
// launches of a workgroup per row (C8H18: front 86 us and back 62, in one workgroup
// each 242 and 124).
template <bool kArray>
__device__ __forceinline__ OrbArgs record(const OrbArgs& one, const OrbArgs* __restrict__ recs, int w) {
  if constexpr (kArray)
    return recs[w];
  else
    return one;
}

__device__ __forceinline__ void clear(const ZeroArgs& z, unsigned block, unsigned blocks) {
  const size_t t0 = (size_t)block * blockDim.x + threadIdx.x, step = (size_t)blocks * blockDim.x;
  for (int k = 0; k < 4; ++k)
    for (size_t i = t0; i < z.n[k]; i += step) z.p[k][i] = 0u;
}

// Workgroups [0, nrec) take a wave function each; the rest clear what the
// quartet pass accumulates into.
template <bool kArray>
__global__ void __launch_bounds__(kOrbThreads) k_orbital_front(OrbArgs one, const OrbArgs* __restrict__ recs, int nrec,
                                                               ZeroArgs z) {
  __shared__ double M[kOrbMax * kOrbMax], red[kOrbThreads / 64];
  __shared__ RowScratch row[kOrbThreads / 64];
  if ((int)blockIdx.x >= nrec) {
    clear(z, blockIdx.x - nrec, gridDim.x - nrec);
    return;
  }
  const OrbArgs a = record<kArray>(one, recs, blockIdx.x);
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  for (int p = wave; p < a.nsp; p += kOrbThreads / 64) orbital_row(a, wave_row(), p, row[wave]);
  __syncthreads();
  orbital_middle(a, M, red);
  __syncthreads();
  for (int s = 0; s < a.nspin; ++s)
    for (int mu = wave; mu < a.nbf; mu += kOrbThreads / 64) density_row(a, wave_row(), s, mu, row[wave]);
}

// Grid (orbital, wave function); the last kClearBlocks orbitals' places clear.
constexpr int kClearBlocks = 32;
template <bool kArray>
__global__ void __launch_bounds__(256) k_orbital_rows(OrbArgs one, const OrbArgs* __restrict__ recs, ZeroArgs z) {
  __shared__ RowScratch row;
  const int nsp = (int)gridDim.x - kClearBlocks;
  if ((int)blockIdx.x >= nsp) {
    clear(z, blockIdx.y * kClearBlocks + blockIdx.x - nsp, gridDim.y * kClearBlocks);
    return;
  }
  orbital_row(record<kArray>(one, recs, blockIdx.y), block_row(), blockIdx.x, row);
}

template <bool kArray>
__global__ void __launch_bounds__(kOrbThreads) k_orbital_middle(OrbArgs one, const OrbArgs* __restrict__ recs) {
  __shared__ double M[kOrbMax * kOrbMax], red[kOrbThreads / 64];
  orbital_middle(record<kArray>(one, recs, blockIdx.x), M, red);
}

// Grid (AO, wave function, spin).
template <bool kArray>
__global__ void __launch_bounds__(256) k_density_rows(OrbArgs one, const OrbArgs* __restrict__ recs) {
  __shared__ RowScratch row;
  density_row(record<kArray>(one, recs, blockIdx.y), block_row(), blockIdx.z, blockIdx.x, row);
}

// F_s = w1 h + cfac (A + A^T) - (B_s + B_s^T) from the J/K accumulators, one
// 32 x 32 tile per workgroup (the transposed tile through LDS), and the tile's
// share of E2 = 1/2 tr(R_s (F_s - w1 h)).  Grid: (tile column, tile row,
// wave function x spin).
template <bool kArray>
__global__ void __launch_bounds__(256) k_fock(OrbArgs one, const OrbArgs* __restrict__ recs) {
  __shared__ double tj[32][33], tk[32][33], red[4];
  const int nspin = kArray ? recs[0].nspin : one.nspin;
  const int w = blockIdx.z / nspin, s = blockIdx.z - w * nspin;
  const OrbArgs a = kArray ? recs[w] : one;
  const int n = a.nbf, i0 = blockIdx.y * 32, j0 = blockIdx.x * 32;
  const int tx = threadIdx.x & 31, ty = threadIdx.x >> 5;
  const double* K = a.K + (size_t)s * n * n;
  const double* R = a.R + (size_t)s * n * n;
  double* F = a.F + (size_t)s * n * n;
  const double cfac = nspin == 1 ? 2.0 : 1.0;
  for (int r = ty; r < 32; r += 8)
    if (j0 + r < n && i0 + tx < n) {
      tj[r][tx] = a.J[(size_t)(j0 + r) * n + i0 + tx];
      tk[r][tx] = K[(size_t)(j0 + r) * n + i0 + tx];
    }
  __syncthreads();
  double e2 = 0.0;
  for (int r = ty; r < 32; r += 8) {
    const int i = i0 + r, j = j0 + tx;
    if (i >= n || j >= n) continue;
    const size_t t = (size_t)i * n + j;
    const double f2 = cfac * (a.J[t] + tj[tx][r]) - (K[t] + tk[tx][r]);
    e2 += 0.5 * R[t] * f2;
    F[t] = cfac * a.H[t] + f2;  // w1 = cfac
  }
  e2 = block_sum(e2, red);
  if (threadIdx.x == 0)
    a.partial[((size_t)s * gridDim.y + blockIdx.y) * gridDim.x + blockIdx.x] = e2;
}

// Row p of Y_s = C F_s; p counts the spin's orbitals.
__device__ __forceinline__ void fock_row(const OrbArgs& a, Row r, int s, int p, RowScratch& lds) {
  const int tid = r.tid, nt = r.nt, n = a.nbf;
  double* w = lds.w;
  int* tgt = lds.tgt;
  const int off = s == 0 ? 0 : a.nunpd;
  const int k0 = a.orb_start[off + p], k1 = a.orb_start[off + p + 1];
  const double* F = a.F + (size_t)s * n * n;
  double* Y = a.Y[s] + (size_t)p * n;
  for (int kb = k0; kb < k1 || kb == k0; kb += kOrbEntries) {
    const int len = min(kOrbEntries, k1 - kb);
    r.sync();
    for (int k = tid; k < len; k += nt) {
      tgt[k] = a.ent[kb + k].tgt;
      w[k] = a.angn[tgt[k]] * a.coeff[kb + k];
    }
    r.sync();
    for (int v = tid; v < n; v += nt) {
      double y = kb == k0 ? 0.0 : Y[v];
      for (int k = 0; k < len; ++k) y += w[k] * F[(size_t)tgt[k] * n + v];
      Y[v] = y;
    }
  }
}

// Per spin V = P W, W = (Y C^T) P, into a.V; E2 from the Fock tiles.  LDS: two
// m x m matrices.
__device__ void gradient_middle(const OrbArgs& a, double* lds, double* red) {
  const int tid = threadIdx.x, n = a.nbf, ns = a.nsp;
  const int tiles = (n + 31) / 32, np = a.nspin * tiles * tiles;
  double e2 = 0.0;
  for (int e = tid; e < np; e += kOrbThreads) e2 += a.partial[e];
  e2 = block_sum(e2, red);
  if (tid == 0) a.scal[3] = e2;
  for (int s = 0; s < a.nspin; ++s) {
    const int off = s == 0 ? 0 : a.nunpd, m = s == 0 ? a.nalpha : a.ndocc;
    double *P = lds, *A = lds + m * m;
    const double* Y = a.Y[s];
    __syncthreads();  // the previous spin is done with the LDS
    for (int e = tid; e < m * m; e += kOrbThreads) P[e] = a.P[(size_t)s * ns * ns + e];
    for (int e = tid; e < m * m; e += kOrbThreads) {  // A = Y C^T
      const int p = e / m, q = e - p * m;
      double t = 0.0;
      for (int k = a.orb_start[off + q]; k < a.orb_start[off + q + 1]; ++k) {
        const int mu = a.ent[k].tgt;
        t += a.angn[mu] * a.coeff[k] * Y[(size_t)p * n + mu];
      }
      A[e] = t;
    }
    __syncthreads();
    double v[kOrbMax * kOrbMax / kOrbThreads];
#pragma unroll
    for (int x = 0; x < kOrbMax * kOrbMax / kOrbThreads; ++x) {  // P A
      const int e = tid + x * kOrbThreads;
      v[x] = 0.0;
      if (e < m * m)
        for (int r = 0; r < m; ++r) v[x] += P[(e / m) * m + r] * A[r * m + e % m];
    }
    __syncthreads();
#pragma unroll
    for (int x = 0; x < kOrbMax * kOrbMax / kOrbThreads; ++x)
      if (tid + x * kOrbThreads < m * m) A[tid + x * kOrbThreads] = v[x];
    __syncthreads();
    for (int e = tid; e < m * m; e += kOrbThreads) {  // V = (P A) P
      double t = 0.0;
      for (int r = 0; r < m; ++r) t += A[(e / m) * m + r] * P[r * m + e % m];
      a.V[s][e] = t;
    }
  }
}

// Row o of G = dE/dC, 2 (P_s Y_s - V_s T) summed over the spins that hold orbital
// o, and the gradient of its weights.  Row 0 also writes the zeros of the weights
// that belong to no occupied orbital.
__device__ __forceinline__ void gradient_row(const OrbArgs& a, Row r, double* grad, int o, RowScratch& lds) {
  const int tid = r.tid, nt = r.nt, n = a.nbf, ns = a.nsp;
  double* u = lds.w;
  for (int s = 0; s < a.nspin; ++s) {
    const int off = s == 0 ? 0 : a.nunpd, m = s == 0 ? a.nalpha : a.ndocc;
    const int p = o - off;
    const bool in = p >= 0 && p < m;  // the same in every thread
    r.sync();
    for (int q = tid; in && q < m; q += nt) {
      u[q] = a.P[(size_t)s * ns * ns + p * m + q];
      u[kOrbMax + q] = a.V[s][p * m + q];
    }
    r.sync();
    for (int v = tid; v < n; v += nt) {
      double g = 0.0;
      for (int q = 0; in && q < m; ++q)
        g += u[q] * a.Y[s][(size_t)q * n + v] - u[kOrbMax + q] * a.T[(size_t)(off + q) * n + v];
      double* G = a.G + (size_t)o * n + v;
      *G = (s == 0 ? 0.0 : *G) + 2.0 * g;
    }
  }
  r.sync();
  for (int k = a.orb_start[o] + tid; k < a.orb_start[o + 1]; k += nt) {
    const int mu = a.ent[k].tgt;
    grad[k] = a.angn[mu] * a.G[(size_t)o * n + mu];
  }
  if (o > 0) return;
  for (int k = tid; k < a.orb_start[0]; k += nt) grad[k] = 0.0;
  for (int k = a.orb_start[a.nsp] + tid; k < a.totlen; k += nt) grad[k] = 0.0;
}

template <bool kArray>
__global__ void __launch_bounds__(kOrbThreads) k_orbital_back(OrbArgs one, const OrbArgs* __restrict__ recs,
                                                              double* grad) {
  extern __shared__ double lds[];
  __shared__ double red[kOrbThreads / 64];
  __shared__ RowScratch row[kOrbThreads / 64];
  const OrbArgs a = record<kArray>(one, recs, blockIdx.x);
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  for (int s = 0; s < a.nspin; ++s)
    for (int p = wave; p < (s == 0 ? a.nalpha : a.ndocc); p += kOrbThreads / 64)
      fock_row(a, wave_row(), s, p, row[wave]);
  __syncthreads();
  gradient_middle(a, lds, red);
  __syncthreads();
  for (int o = wave; o < a.nsp; o += kOrbThreads / 64)
    gradient_row(a, wave_row(), kArray ? a.grad : grad, o, row[wave]);
}

// Grid (orbital, wave function, spin).
template <bool kArray>
__global__ void __launch_bounds__(256) k_fock_rows(OrbArgs one, const OrbArgs* __restrict__ recs) {
  __shared__ RowScratch row;
  const OrbArgs a = record<kArray>(one, recs, blockIdx.y);
  if ((int)blockIdx.x < (blockIdx.z == 0 ? a.nalpha : a.ndocc)) fock_row(a, block_row(), blockIdx.z, blockIdx.x, row);
}

template <bool kArray>
__global__ void __launch_bounds__(kOrbThreads) k_gradient_middle(OrbArgs one, const OrbArgs* __restrict__ recs) {
  extern __shared__ double lds[];
  __shared__ double red[kOrbThreads / 64];
  gradient_middle(record<kArray>(one, recs, blockIdx.x), lds, red);
}

// Grid (orbital, wave function).
template <bool kArray>
__global__ void __launch_bounds__(256) k_gradient_rows(OrbArgs one, const OrbArgs* __restrict__ recs, double* grad) {
  __shared__ RowScratch row;
  const OrbArgs a = record<kArray>(one, recs, blockIdx.y);
  gradient_row(a, block_row(), kArray ? a.grad : grad, blockIdx.x, row);
}

// E2 = the sum of the quartet kernels' partial sums (a fixed order), E.
__global__ void __launch_bounds__(kOrbThreads) k_energy_sum(const double* __restrict__ partial, long n, double enuc,
                                                            double* __restrict__ scal) {
  __shared__ double red[kOrbThreads / 64];
  double t[8] = {0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0};
  long i = threadIdx.x;
  for (; i + 7 * kOrbThreads < n; i += 8 * kOrbThreads)  // eight loads in flight
#pragma unroll
    for (int k = 0; k < 8; ++k) t[k] += partial[i + k * kOrbThreads];
  for (; i < n; i += kOrbThreads) t[0] += partial[i];
  const double e2 = block_sum(((t[0] + t[1]) + (t[2] + t[3])) + ((t[4] + t[5]) + (t[6] + t[7])), red);
  if (threadIdx.x == 0) {
    scal[1] = e2;
    scal[2] = scal[0] + e2 + enuc;
  }
}

}  // namespace

template <bool kArray>
static hipError_t front(hipStream_t st, const OrbArgs& one, const OrbArgs* recs, int nrec, const ZeroArgs& z) {
  if (one.nbf <= kOrbOneLaunch) {
    size_t most = 0;
    for (size_t n : z.n) most = std::max(most, n);
    const unsigned grid = (unsigned)nrec + (unsigned)std::min<size_t>(16, (most + kOrbThreads - 1) / kOrbThreads);
    hipLaunchKernelGGL(k_orbital_front<kArray>, dim3(grid), dim3(kOrbThreads), 0, st, one, recs, nrec, z);
    return hipGetLastError();
  }
  hipLaunchKernelGGL(k_orbital_rows<kArray>, dim3(one.nsp + kClearBlocks, nrec), dim3(256), 0, st, one, recs, z);
  hipLaunchKernelGGL(k_orbital_middle<kArray>, dim3(nrec), dim3(kOrbThreads), 0, st, one, recs);
  hipLaunchKernelGGL(k_density_rows<kArray>, dim3(one.nbf, nrec, one.nspin), dim3(256), 0, st, one, recs);
  return hipGetLastError();
}

template <bool kArray>
static hipError_t back(hipStream_t st, const OrbArgs& one, const OrbArgs* recs, int nrec, double* grad) {
  const unsigned tiles = (unsigned)(one.nbf + 31) / 32;
  const int m = std::max(one.nalpha, one.ndocc);
  const size_t lds = 2 * (size_t)m * m * sizeof(double);
  hipLaunchKernelGGL(k_fock<kArray>, dim3(tiles, tiles, (unsigned)(nrec * one.nspin)), dim3(256), 0, st, one, recs);
  if (one.nbf <= kOrbOneLaunch) {
    hipLaunchKernelGGL(k_orbital_back<kArray>, dim3(nrec), dim3(kOrbThreads), lds, st, one, recs, grad);
    return hipGetLastError();
  }
  hipLaunchKernelGGL(k_fock_rows<kArray>, dim3(m, nrec, one.nspin), dim3(256), 0, st, one, recs);
  hipLaunchKernelGGL(k_gradient_middle<kArray>, dim3(nrec), dim3(kOrbThreads), lds, st, one, recs);
  hipLaunchKernelGGL(k_gradient_rows<kArray>, dim3(one.nsp, nrec), dim3(256), 0, st, one, recs, grad);
  return hipGetLastError();
}

hipError_t launch_orbital_front(hipStream_t st, const OrbArgs& one, const OrbArgs* recs, int nrec, const ZeroArgs& z) {
  return recs ? front<true>(st, one, recs, nrec, z) : front<false>(st, one, recs, nrec, z);
}

hipError_t launch_orbital_back(hipStream_t st, const OrbArgs& one, const OrbArgs* recs, int nrec, double* grad) {
  return recs ? back<true>(st, one, recs, nrec, grad) : back<false>(st, one, recs, nrec, grad);
}

hipError_t launch_energy_sum(hipStream_t st, const double* partial, long n, double enuc, double* scal) {
  hipLaunchKernelGGL(k_energy_sum, dim3(1), dim3(kOrbThreads), 0, st, partial, n, enuc, scal);
  return hipGetLastError();
}

}  // namespace vsvb

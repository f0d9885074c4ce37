// Stored integrals: J and K of one geometry from a matrix of its two-electron
// integrals instead of quartet by quartet.
//
// A J/K pass contracts every quartet with every density as it is computed: per
// density six scattered sums and their atomics.  An energy pass that only stores
// its integrals is shorter than a J/K pass of one density and does not grow with
// the densities; the contractions are then dense products over a matrix that was
// written once.  What bounds them is reading that matrix (nbf^4 / 4 numbers), so
// they pay where the densities are many.  Function pairs of a shell pair lie a
// class apart (Pair::f0), so that the 64 bra pairs of a wavefront add to 64
// neighbours: side by side H12's (pp|ps) took 259 us instead of 53.
#include "vsvb_internal.h"

namespace vsvb {

namespace {

typedef double v4d __attribute__((ext_vector_type(4)));
typedef double d4u __attribute__((ext_vector_type(4), aligned(8)));

__device__ __forceinline__ int tri(int i, int j) { return i >= j ? i * (i + 1) / 2 + j : j * (j + 1) / 2 + i; }

struct ClassOffsets {
  int at[kNPairClass + 1];
};

// The functions of every entry of the function-pair list, and the entry of every
// pair of functions mu >= nu (t = mu (mu + 1) / 2 + nu).
__global__ void k_function_pairs(const Pair* __restrict__ pairs, ClassOffsets off, const Shell* __restrict__ shells,
                                 FnPair* __restrict__ fn, int* __restrict__ at) {
  const int p = blockIdx.x * blockDim.x + threadIdx.x;
  if (p >= off.at[kNPairClass]) return;
  int cl = 0;
  while (p >= off.at[cl + 1]) ++cl;
  const Pair P = pairs[p];
  const Shell A = shells[P.A], B = shells[P.B];
  int f = P.f0;
  for (int i = 0; i < ncart(A.l); ++i)
    for (int j = 0; j < ncart(B.l); ++j, f += off.at[cl + 1] - off.at[cl]) {
      fn[f] = FnPair{A.ao + i, B.ao + j, P.A == P.B};
      if (P.A != P.B || i >= j) at[tri(A.ao + i, B.ao + j)] = f;
    }
}

// M = T + T^T in place, a workgroup per 32 x 32 tile on or below the diagonal and
// its mirror image, through LDS so that both are read and written along rows.
__global__ void __launch_bounds__(256) k_sym_tiles(double* __restrict__ M, int n) {
  __shared__ double lo[32][33], up[32][33];
  const int bi = blockIdx.y, bj = blockIdx.x, tx = threadIdx.x & 31, ty = threadIdx.x >> 5;
  if (bj > bi) return;
  for (int r = ty; r < 32; r += 8) {
    const int i = bi * 32 + r, j = bj * 32 + tx, it = bj * 32 + r, jt = bi * 32 + tx;
    lo[r][tx] = i < n && j < n ? M[(size_t)i * n + j] : 0.0;
    up[r][tx] = it < n && jt < n ? M[(size_t)it * n + jt] : 0.0;
  }
  __syncthreads();
  for (int r = ty; r < 32; r += 8) {
    const int i = bi * 32 + r, j = bj * 32 + tx, it = bj * 32 + r, jt = bi * 32 + tx;
    if (i < n && j < n) M[(size_t)i * n + j] = lo[r][tx] + up[tx][r];
    if (bi != bj && it < n && jt < n) M[(size_t)it * n + jt] = up[r][tx] + lo[tx][r];
  }
}

// N[t][u] = M[at[t]][at[u]]: rows and columns by functions, for the exchange.  A
// workgroup takes a row; it is staged in LDS kStage numbers at a time, since a
// gather from memory fetches a line per number (C8H18's 3.9 GB: 6.8 ms so, 2.0
// through LDS), and a thread's numbers wait in registers until all are there.
constexpr int kRowThreads = 1024, kRowOwn = 24, kStage = 16384;

__global__ void __launch_bounds__(kRowThreads) k_by_functions(const double* __restrict__ M,
                                                              const int* __restrict__ at, int nf, int nt,
                                                              double* __restrict__ N) {
  extern __shared__ double part[];
  const int tid = threadIdx.x;
  const double* row = M + (size_t)at[blockIdx.x] * nf;
  double* out = N + (size_t)blockIdx.x * nt;
  for (int u0 = 0; u0 < nt; u0 += kRowThreads * kRowOwn) {
    int f[kRowOwn];
    double v[kRowOwn];
#pragma unroll
    for (int x = 0; x < kRowOwn; ++x) {
      const int u = u0 + x * kRowThreads + tid;
      f[x] = u < nt ? at[u] : -1;
    }
    for (int f0 = 0; f0 < nf; f0 += kStage) {
      const int len = min(kStage, nf - f0);
      __syncthreads();  // the previous part is read
      for (int k = tid; k < len; k += kRowThreads) part[k] = row[f0 + k];
      __syncthreads();
#pragma unroll
      for (int x = 0; x < kRowOwn; ++x)
        if (f[x] >= f0 && f[x] < f0 + len) v[x] = part[f[x] - f0];
    }
#pragma unroll
    for (int x = 0; x < kRowOwn; ++x)
      if (f[x] >= 0) out[u0 + x * kRowThreads + tid] = v[x];
  }
}

// Dp[w][t]: the Coulomb weight of a pair of functions, cfac sum_s D, twice off the
// diagonal.  Dt[b][d][x] = D_x[b][d], densities fastest, zero up to nd and xp.
__global__ void k_stored_densities(const double* __restrict__ dens, int n, int nwfn, int nspin, int nt, int nd, int xp,
                                   double* __restrict__ Dp, double* __restrict__ Dt) {
  const size_t nn = (size_t)n * n;
  const int b = blockIdx.x, X = nwfn * nspin;
  const double cfac = nspin == 1 ? 2.0 : 1.0;
  for (int e = threadIdx.x; e < nd * xp; e += blockDim.x) {
    const int d = e / xp, x = e - d * xp;
    Dt[(size_t)b * nd * xp + e] = d < n && x < X ? dens[x * nn + (size_t)b * n + d] : 0.0;
  }
  for (int e = threadIdx.x; e < nwfn * (b + 1); e += blockDim.x) {
    const int w = e / (b + 1), d = e - w * (b + 1);
    double s = 0.0;
    for (int k = 0; k < nspin; ++k) s += dens[(size_t)(w * nspin + k) * nn + (size_t)b * n + d];
    Dp[(size_t)w * nt + tri(b, d)] = (b == d ? 1.0 : 2.0) * cfac * s;
  }
}

// The accumulators hold half of the symmetric result (the Fock matrix adds the transpose).
__global__ void k_stored_coulomb(const double* __restrict__ Jp, int n, int nwfn, int nt, double* __restrict__ jacc) {
  const size_t nn = (size_t)n * n, tot = nwfn * nn;
  for (size_t e = blockIdx.x * (size_t)blockDim.x + threadIdx.x; e < tot; e += (size_t)gridDim.x * blockDim.x) {
    const size_t w = e / nn;
    const int r = (int)(e - w * nn);
    jacc[e] = 0.5 * Jp[w * nt + tri(r / n, r % n)];
  }
}

// K_x[a][c] = sum_bd (ab|cd) D_x[b][d], c <= a.  A workgroup takes one a, `bper` of
// the b and 256 of the c; a wavefront up to four tiles of 16 c and NT of 16
// densities: V_MFMA_F64_16X16X4F64 over blocks of 16 d, where lane (i, k) holds
// (ab|c_i d) of four consecutive d, so that the 16 x 16 block's lines are read whole
// at once: along d below the diagonal of (cd), along c above it.  Bounded by those
// loads, 8 GB of C8H18's matrix: 2.8 ms for 32 densities (5.0 with the d of a
// lane four apart).
constexpr int kTilesC = 4;

template <int NT>
__global__ void __launch_bounds__(256) k_stored_exchange(const double* __restrict__ N, int nt,
                                                         const double* __restrict__ Dt, int n, int nd, int xp, int X,
                                                         int bper, int ncg, double scale, double* __restrict__ kacc) {
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int li = lane & 15, lk = lane >> 4;
  const int a = n - 1 - (int)blockIdx.x;
  const int cg = (int)blockIdx.z % ncg, x0 = (int)blockIdx.z / ncg * 16 * NT;
  const int b0 = (int)blockIdx.y * bper, b1 = min(n, b0 + bper);
  int c0[kTilesC], c[kTilesC], tc[kTilesC];
  v4d acc[kTilesC][NT];
#pragma unroll
  for (int i = 0; i < kTilesC; ++i) {
    c0[i] = 16 * (cg * 4 * kTilesC + wave + 4 * i);
    c[i] = min(c0[i] + li, n - 1);
    tc[i] = c[i] * (c[i] + 1) / 2;
#pragma unroll
    for (int t = 0; t < NT; ++t) acc[i][t] = v4d{0.0, 0.0, 0.0, 0.0};
  }
  if (c0[0] > a) return;  // whole wavefront: its first tile is its lowest
  for (int b = b0; b < b1; ++b) {
    const double* row = N + (size_t)tri(a, b) * nt;
    const double* db = Dt + (size_t)b * nd * xp + x0 + li;
    for (int d0 = 0; d0 < nd; d0 += 16) {
      const int dl = d0 + 4 * lk;
      double y[NT][4];
      int d[4];
#pragma unroll
      for (int s = 0; s < 4; ++s) {
        d[s] = min(dl + s, n - 1);  // past the end: times zero
#pragma unroll
        for (int t = 0; t < NT; ++t) y[t][s] = db[(size_t)(dl + s) * xp + 16 * t];
      }
#pragma unroll
      for (int i = 0; i < kTilesC; ++i)
        if (c0[i] <= a) {  // the same in every lane
          double x[4];
          if (c0[i] >= d0 + 15) {
            const d4u q = *reinterpret_cast<const d4u*>(row + tc[i] + dl);
#pragma unroll
            for (int s = 0; s < 4; ++s) x[s] = q[s];
          } else {
#pragma unroll
            for (int s = 0; s < 4; ++s) x[s] = row[c[i] >= d[s] ? tc[i] + d[s] : d[s] * (d[s] + 1) / 2 + c[i]];
          }
#pragma unroll
          for (int s = 0; s < 4; ++s)
#pragma unroll
            for (int t = 0; t < NT; ++t)
              acc[i][t] = __builtin_amdgcn_mfma_f64_16x16x4f64(x[s], y[t][s], acc[i][t], 0, 0, 0);
        }
    }
  }
#pragma unroll
  for (int i = 0; i < kTilesC; ++i)
#pragma unroll
    for (int t = 0; t < NT; ++t)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int cc = c0[i] + lk + 4 * r, x = x0 + 16 * t + li;
        if (cc > a || x >= X) continue;
        double* K = kacc + (size_t)x * n * n;
        unsafeAtomicAdd(&K[(size_t)a * n + cc], scale * acc[i][t][r]);
        if (cc < a) unsafeAtomicAdd(&K[(size_t)cc * n + a], scale * acc[i][t][r]);
      }
}

}  // namespace

// Densities padded to what a launch of k_stored_exchange takes at once.
static int padded(int x) { return x > 16 ? (x + 31) / 32 * 32 : 16; }

void stored_setup(vsvb_context* c, StoredIntegrals& s, int nwfn, int nspin, size_t limit) {
  const size_t nf = (size_t)c->nfun, n = (size_t)c->nbf, nt = n * (n + 1) / 2;
  const size_t xp = padded(nwfn * nspin), nd = (n + 15) / 16 * 16;
  const size_t numbers = nf * nf + (nspin > 0 ? nt * nt + 2 * nwfn * nt + n * nd * xp : 0);
  // (many contexts leave room for the next: each takes a sixteenth of what is left)
  size_t free_bytes = 0, total_bytes = 0;
  hipError_t e = hipMemGetInfo(&free_bytes, &total_bytes);
  if (e == hipSuccess) limit = std::min(limit, free_bytes / 16);
  if (numbers * sizeof(double) > limit) return;
  e = s.fn.alloc(nf);
  if (e == hipSuccess) e = s.at.alloc(nt);
  if (nspin > 0) {
    if (e == hipSuccess) e = s.N.alloc(nt * nt);
    if (e == hipSuccess) e = s.Dp.alloc(nwfn * nt);
    if (e == hipSuccess) e = s.Jp.alloc(nwfn * nt);
    if (e == hipSuccess) e = s.Dt.alloc(n * nd * xp);
  }
  if (e == hipSuccess) e = s.M.alloc(nf * nf);
  if (e == hipSuccess) return;
  (void)hipGetLastError();  // the quartet-by-quartet pass runs instead
  s.M.release();
  s.N.release();
  s.Dp.release();
  s.Jp.release();
  s.Dt.release();
  s.at.release();
  s.fn.release();
}

int stored_integrals(vsvb_context* c, StoredIntegrals& s) {
  hipStream_t st = c->stream;
  const int nf = c->nfun;
  const unsigned tiles = (unsigned)(nf + 31) / 32;
  HIP_OK(launch_fill(st, s.M.p, (size_t)nf * nf, 0.0));
  const int rc = run_quartets(c, false, 0, nullptr, nullptr, nullptr, 0, s.M.p);
  if (rc) return rc;
  hipLaunchKernelGGL(k_sym_tiles, dim3(tiles, tiles), dim3(256), 0, st, s.M.p, nf);
  ClassOffsets off;
  std::copy(c->pair_off, c->pair_off + kNPairClass + 1, off.at);
  hipLaunchKernelGGL(k_function_pairs, dim3((c->npairs + 255) / 256), dim3(256), 0, st, c->d_pairs.p, off,
                     c->d_shells.p, s.fn.p, s.at.p);
  HIP_OK(hipGetLastError());
  return VSVB_OK;
}

int stored_jk(vsvb_context* c, StoredIntegrals& s, int nwfn, const double* dens, double* jacc, double* kacc) {
  hipStream_t st = c->stream;
  const int n = c->nbf, nt = n * (n + 1) / 2, nspin = c->nunpd > 0 ? 2 : 1;
  const int X = nwfn * nspin, xp = padded(X), nd = (n + 15) / 16 * 16;
  const int rc = stored_integrals(c, s);
  if (rc) return rc;
  hipLaunchKernelGGL(k_by_functions, dim3(nt), dim3(kRowThreads), std::min(c->nfun, kStage) * sizeof(double), st, s.M.p,
                     s.at.p, c->nfun, nt, s.N.p);
  hipLaunchKernelGGL(k_stored_densities, dim3(n), dim3(256), 0, st, dens, n, nwfn, nspin, nt, nd, xp, s.Dp.p, s.Dt.p);
  HIP_OK(hipGetLastError());
  HIP_OK(gemm(st, nwfn, nt, nt, 1.0, s.Dp.p, nt, false, s.N.p, nt, false, 0.0, s.Jp.p, nt));
  hipLaunchKernelGGL(k_stored_coulomb, dim3((unsigned)std::min<size_t>(4096, ((size_t)nwfn * n * n + 255) / 256)),
                     dim3(256), 0, st, s.Jp.p, n, nwfn, nt, jacc);
  HIP_OK(launch_fill(st, kacc, (size_t)X * n * n, 0.0));
  const int ncg = (n + 16 * 4 * kTilesC - 1) / (16 * 4 * kTilesC), split = std::max(1, std::min(n, 2048 / n));
  const int bper = (n + split - 1) / split, nb = (n + bper - 1) / bper;
  const double scale = nspin == 1 ? 1.0 : 0.5;
  if (X > 16)
    hipLaunchKernelGGL(k_stored_exchange<2>, dim3(n, nb, ncg * (xp / 32)), dim3(256), 0, st, s.N.p, nt, s.Dt.p, n,
                       nd, xp, X, bper, ncg, scale, kacc);
  else
    hipLaunchKernelGGL(k_stored_exchange<1>, dim3(n, nb, ncg), dim3(256), 0, st, s.N.p, nt, s.Dt.p, n, nd, xp, X, bper,
                       ncg, scale, kacc);
  HIP_OK(hipGetLastError());
  return VSVB_OK;
}

}  // namespace vsvb

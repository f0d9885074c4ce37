"""The device product's 64-row tiles (many rows; 48 and 64 columns per workgroup)
and its split-K tiles (long K, few tiles) against numpy through vsvb_debug_gemm:
edges of the tiles, of a K step and of a wavefront's share of K, every transpose
combination, and beta != 0.
Tolerance: 1e-13 of K * max|A| * max|B| (+ 2 max|C0|) per element."""
import itertools

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

# from 8e6 multiply-adds and 128 workgroups: 64-row tiles (columns 144, 50, 33, 64, 1100, 130), 32-row tiles
TILES = [(4097, 144, 40), (8200, 50, 33), (8129, 33, 31), (8192, 64, 16), (700, 1100, 17), (3001, 130, 65), (32, 8200, 40),
         (17, 8129, 70), (5, 8300, 200)]
# K >= 1024, or 8e6 multiply-adds in fewer workgroups: K split over a workgroup's wavefronts
DEEP = [(1, 144, 4096), (17, 5, 1024), (16, 16, 1025), (3, 2, 1087), (33, 1, 5000), (144, 144, 4096), (500, 130, 129)]


@pytest.fixture(scope="module")
def lib():
    from valence_amd import lib as L
    L.load()
    return L


@pytest.mark.parametrize("shape", TILES + DEEP)
def test_gemm_tiles_match_numpy(lib, shape):
    M, N, K = shape
    rng = np.random.default_rng(M * 1000 + N * 10 + K)
    a = rng.normal(size=(M, K)); b = rng.normal(size=(K, N)); c0 = rng.normal(size=(M, N))
    ref = a @ b
    scale = 1e-13 * K * np.abs(a).max() * np.abs(b).max()
    for ta, tb in itertools.product([False, True], [False, True]):
        A = a.T.copy() if ta else a
        B = b.T.copy() if tb else b
        err = np.abs(lib.device_gemm(A, B, ta, tb) - ref).max()
        errb = np.abs(lib.device_gemm(A, B, ta, tb, alpha=-0.5, beta=2.0, C0=c0) - (-0.5 * ref + 2.0 * c0)).max()
        print(f"M={M} N={N} K={K} ta={ta} tb={tb} max err {err:.2e} {errb:.2e} tol {scale:.2e}")
        assert err <= scale and errb <= scale + 2e-13 * np.abs(c0).max()

"""Shared launches and side streams against one launch per class on one stream, which
a forced chunk width (pair_chunk) selects: water, whose two cooperative classes run
beside the shared launch, methane, ethane in two spin densities and pentane, whose
larger classes have launches of their own.  Energies to 1e-12 relative, gradients to
1e-11 of their norm (another summation order), equal quartet counts; then a batch of
them against their own contexts.
"""
import numpy as np
import pytest

from valence_amd import workloads

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def lib():
    from valence_amd import lib as L
    L.load()
    return L


def _system(n, unpaired):
    if n == 0:
        return workloads.config0()
    base = workloads.config1()
    basis = {"C": (6.0, workloads._type_shells(base, 0)), "H": (1.0, workloads._type_shells(base, 1))}
    s = workloads.alkane_system(n, basis, np.random.default_rng(n))
    s.nunpd, s.ndocc = unpaired, s.ndocc - unpaired
    return s


def _close(e, g, e0, g0):
    assert abs(e - e0) <= 1e-12 * abs(e0)
    assert np.linalg.norm(g - g0) <= 1e-11 * np.linalg.norm(g0)


@pytest.mark.parametrize("n,unpaired", [(0, 0), (1, 0), (2, 2), (5, 0)])
def test_separate_launches_give_the_same(lib, n, unpaired):
    s = _system(n, unpaired)
    assert lib.launch_plan(s)[0][..., 7].any() and not lib.launch_plan(s, pair_chunk=1)[0][..., 7].any()
    with lib.Context(s, pair_chunk=1) as ref, lib.Context(s) as ctx:
        for scale in (1.0, 1.2, 1.0):
            x = s.coords * scale
            e0, q0 = ref.energy(coords=x), ref.counters()
            e1, q1 = ctx.energy(coords=x), ctx.counters()
            (g0, d0), (g1, d1) = ref.energy_grad(), ctx.energy_grad()
            print(f"n={n} nunpd={unpaired}: {e0:.12f} {e1:.12f} {g1:.12f}", flush=True)
            assert abs(e1 - e0) <= 1e-12 * abs(e0)
            _close(g1, d1, g0, d0)
            assert q0[0] == q1[0] and q0[2] == q1[2]


def test_batch_matches_separate_launches(lib):
    systems = [_system(0, 0), _system(1, 0), _system(2, 2), _system(1, 1)]
    want = []
    for s in systems:
        with lib.Context(s, pair_chunk=1) as ref:
            want.append(ref.energy_grad())
    for chunk in (0, 1):
        b = lib.Batch(systems, pair_chunk=chunk)
        for rep in range(3):
            e, g = b.run(want_grad=True)
            for k, (e0, g0) in enumerate(want):
                _close(e[k], g[k], e0, g0)
        b.close()

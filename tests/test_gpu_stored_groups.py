"""Batch groups of eight and more wave functions, whose J and K come from stored
integrals, against a context of its own for each: one and two spin densities, 8 to
33 densities (one block of 16, a part of 32, 32 and one more), bases below, at and
beyond multiples of 16 (25, 35, 60, 85, 210 AOs); a direct run, replays, and a
changed geometry.  Energies to 1e-10 Eh, gradients to 1e-10 of their norm (the sums
of another order, through the same inverse).
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


def _alkane(n, unpaired):
    base = workloads.config1()
    basis = {"C": (6.0, workloads._type_shells(base, 0)), "H": (1.0, workloads._type_shells(base, 1))}
    s = workloads.alkane_system(n, basis, np.random.default_rng(n))
    s.nunpd, s.ndocc = unpaired, s.ndocc - unpaired
    return s


@pytest.mark.parametrize("n,unpaired,members", [(0, 0, 33), (1, 0, 8), (1, 1, 8), (2, 2, 9), (3, 0, 20), (8, 0, 9)])
def test_group_of_many_matches_single_contexts(lib, n, unpaired, members):
    systems = []
    for k in range(members):
        s = _alkane(n, unpaired) if n else workloads.config0()
        s.coeff = s.coeff * (1.0 + 0.03 * k * np.sin(np.arange(s.totlen)))
        systems.append(s)
    b = lib.Batch(systems)
    for scale in (1.0, 1.03):
        for s in systems:
            s.coords = s.coords * scale
        if scale != 1.0:
            b.set_coords([s.coords for s in systems])
        want = []
        for s in systems:
            with lib.Context(s) as ctx:
                want.append(ctx.energy_grad())
        for rep in range(3):
            e, g = b.run(want_grad=True)
            for k, (e0, g0) in enumerate(want):
                assert abs(e[k] - e0) <= 1e-10, (rep, k, e[k], e0)
                assert np.linalg.norm(g[k] - g0) <= 1e-10 * np.linalg.norm(g0), (rep, k)

"""The shared launch of a small system's quartet classes against one launch per
class: pair_chunk=1 keeps whole pairs and separate launches.  Energies to 1e-12
relative, gradients to 1e-11 of their norm (rounding of another summation order),
at molecules whose classes are all shared (methane), partly shared (propane,
pentane) and in two spin densities; the same geometry again, and after changed
weights and profiling (which change the argument records or not).
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


@pytest.mark.parametrize("n,unpaired", [(1, 0), (1, 1), (3, 0), (3, 2), (5, 0)])
def test_shared_launch_matches_separate_launches(lib, n, unpaired):
    s = _alkane(n, unpaired)
    w = s.coeff * (1.0 + 0.1 * np.cos(np.arange(s.totlen)))
    with lib.Context(s, pair_chunk=1) as ref, lib.Context(s) as ctx:
        for k, (c, prof) in enumerate(((s.coeff, False), (w, False), (w, True), (s.coeff, True), (s.coeff, False))):
            ref.set_profiling(prof)
            ctx.set_profiling(prof)
            e0, (g0, d0) = ref.energy(c), ref.energy_grad(c)
            q0 = ref.counters()[0]
            e1, (g1, d1) = ctx.energy(c), ctx.energy_grad(c)
            print(f"C{n} nunpd={unpaired} step {k}: {e0:.12f} {e1:.12f} {g1:.12f}")
            assert abs(e1 - e0) <= 1e-12 * abs(e0) and abs(g1 - g0) <= 1e-12 * abs(g0)
            assert np.linalg.norm(d1 - d0) <= 1e-11 * np.linalg.norm(d0)
            assert ctx.counters()[0] == q0


def test_shared_launch_in_a_replayed_batch(lib):
    """Batches of small molecules: direct run, graph replays, new geometries."""
    systems = [_alkane(1, 0), _alkane(2, 0), _alkane(1, 1), workloads.config0()]
    b = lib.Batch(systems)
    for scale in (1.0, 1.02):
        for k, s in enumerate(systems):
            s.coords = s.coords * scale
        if scale != 1.0:
            b.set_coords([s.coords for s in systems])
        for rep in range(3):
            e, g = b.run(want_grad=True)
            for k, s in enumerate(systems):
                with lib.Context(s, pair_chunk=1) as ctx:
                    e1, g1 = ctx.energy_grad()
                assert abs(e[k] - e1) <= 1e-12 * abs(e1), (scale, rep, k)
                assert np.linalg.norm(g[k] - g1) <= 1e-11 * np.linalg.norm(g1)
    b.close()

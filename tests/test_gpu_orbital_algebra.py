"""The orbital algebra along each orbital's own entries against the dense path
(grid_inverse_min=1 takes it): the one-launch form (up to 64 AOs), the launches of
a workgroup per row (above), 61 orbitals (close to the 64 its LDS holds) and 65
(dense in both), one and two spin densities, an empty beta block, an orbital that
lists an AO twice, and members of a batch group in one launch.  Energies to 1e-10
Eh, gradients to 1e-10 of their norm: rounding through the same inverse.
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


def _alkane(n, unpaired=0):
    base = workloads.config1()
    basis = {"C": (6.0, workloads._type_shells(base, 0)), "H": (1.0, workloads._type_shells(base, 1))}
    s = workloads.alkane_system(n, basis, np.random.default_rng(n))
    s.nunpd, s.ndocc = unpaired, s.ndocc - unpaired
    return s


def _hydrogen_triplet():
    """Two unpaired orbitals and no doubly occupied one."""
    s = workloads.config0()
    basis = {"H": (1.0, workloads._type_shells(s, 1))}
    rng = np.random.default_rng(3)
    orbs = [([k], workloads._rand_orbital(rng, basis, ["H", "H"], [k])) for k in range(2)]
    return workloads.assemble(["H", "H"], np.array([[0.0, 0, 0], [0, 0, 0.8]]), basis, orbs, nunpd=2)


def _twice():
    """Every orbital's second entry repeats its first AO."""
    s = workloads.config0()
    s.xpset = s.xpset.copy()
    for p in range(s.nspatial):
        s.xpset[s.orb_start[p] + 1] = s.xpset[s.orb_start[p]]
    return s


CASES = {"water": workloads.config0, "twice": _twice, "h2_triplet": _hydrogen_triplet, "ethane": lambda: _alkane(2),
         "ethane_spin": lambda: _alkane(2, 2), "propane_spin": lambda: _alkane(3, 1), "octane": workloads.config1,
         "octane_spin": lambda: _alkane(8, 2), "c15": lambda: _alkane(15), "c16": lambda: _alkane(16)}


@pytest.mark.parametrize("name", sorted(CASES))
def test_entry_lists_match_dense_products(lib, name):
    s = CASES[name]()
    w = s.coeff * (1.0 + 0.1 * np.cos(np.arange(s.totlen)))
    with lib.Context(s, grid_inverse_min=1) as ref, lib.Context(s) as ctx:
        for c in (s.coeff, w):
            e0, (g0, d0) = ref.energy(c), ref.energy_grad(c)
            e1, (g1, d1) = ctx.energy(c), ctx.energy_grad(c)
            print(f"{name}: {e0:.12f} {e1:.12f} {g1:.12f} |dg| {np.linalg.norm(d1 - d0):.2e}")
            assert abs(e1 - e0) <= 1e-10 and abs(g1 - g0) <= 1e-10
            assert np.linalg.norm(d1 - d0) <= 1e-10 * np.linalg.norm(d0)


def test_group_members_match_single_contexts(lib):
    """Two groups of three wave functions each (35 and 210 AOs are both sides of
    the one-launch rule), run directly, captured and replayed."""
    systems = []
    for make in (lambda: _alkane(1, 1), workloads.config1):
        for k in range(3):
            s = make()
            s.coeff = s.coeff * (1.0 + 0.05 * k * np.sin(np.arange(s.totlen)))
            systems.append(s)
    want = []
    for s in systems:
        with lib.Context(s, grid_inverse_min=1) as ctx:
            want.append(ctx.energy_grad())
    b = lib.Batch(systems)
    for rep in range(3):
        e, g = b.run(want_grad=True)
        for k, (e0, g0) in enumerate(want):
            assert abs(e[k] - e0) <= 1e-10
            assert np.linalg.norm(g[k] - g0) <= 1e-10 * np.linalg.norm(g0)

"""Spin-coupled wave functions whose integrals are stored once for all orbital
pair densities, against the closed-shell path: a singlet pair of one orbital taken
twice is that orbital doubly occupied, so the energies agree and the gradients of
the two copies add up to the closed-shell orbital's.  Water (every class up to
(dd|dd)), methane, propane, butane, hexane (above the limit on the matrix:
contracted quartet by quartet), H2 (below the fewest densities), with a changed
geometry.  Energies to 1e-10 Eh, gradients to 1e-9 of their
norm (two different chains of small inverses and products).
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


def _alkane(n):
    base = workloads.config1()
    basis = {"C": (6.0, workloads._type_shells(base, 0)), "H": (1.0, workloads._type_shells(base, 1))}
    return workloads.alkane_system(n, basis, np.random.default_rng(n))


def _hydrogen():
    basis = {"H": (1.0, workloads._type_shells(workloads.config0(), 1))}
    orb = ([0, 1], workloads._rand_orbital(np.random.default_rng(3), basis, ["H", "H"], [0, 1]))
    return workloads.assemble(["H", "H"], np.array([[0.0, 0, 0], [0, 0, 0.8]]), basis, [orb])


def _doubled(s, npair):
    """s with its first npair orbitals as spin-coupled pairs of one orbital twice."""
    orbs = []
    for p in range(s.nspatial):
        atoms = list(s.orb_atoms[p, :s.orb_natom[p]])
        orbs += [(atoms, s.coeff[s.orb_start[p]:s.orb_start[p + 1]].copy())] * (2 if p < npair else 1)
    elems = [f"X{t}" for t in s.atom_type]
    basis = {f"X{t}": (float(s.nuc_charge[t]), workloads._type_shells(s, t)) for t in range(len(s.nuc_charge))}
    xyz = s.coords / workloads.ANGSTROM_TO_BOHR
    pairs = [(2 * k + 1, 2 * k + 2) for k in range(npair)]
    return workloads.assemble(elems, xyz, basis, orbs, npair=npair, pair_sc=pairs)


CASES = {"water": (workloads.config0, 2), "methane": (lambda: _alkane(1), 3), "propane": (lambda: _alkane(3), 2),
         "butane": (lambda: _alkane(4), 1), "hexane": (lambda: _alkane(6), 1), "hydrogen": (_hydrogen, 1)}


@pytest.mark.parametrize("name", sorted(CASES))
def test_doubled_orbitals_match_closed_shell(lib, name):
    make, npair = CASES[name]
    s = make()
    t = _doubled(s, npair)
    cut = s.orb_start[npair]
    with lib.Context(s) as ref, lib.Context(t) as ctx:
        for scale in (1.0, 1.1):
            e0 = ref.energy(coords=s.coords * scale)
            e1 = ctx.energy(coords=s.coords * scale)
            _, g0 = ref.energy_grad()
            e2, g1 = ctx.energy_grad()
            folded = np.concatenate([g1[2 * s.orb_start[p]:2 * s.orb_start[p] + s.orb_start[p + 1] - s.orb_start[p]]
                                     + g1[s.orb_start[p] + s.orb_start[p + 1]:2 * s.orb_start[p + 1]]
                                     for p in range(npair)] + [g1[2 * cut:]])
            print(f"{name}: {e0:.12f} {e1:.12f} {e2:.12f} "
                  f"|dg| {np.linalg.norm(folded - g0):.2e} of {np.linalg.norm(g0):.2e}")
            assert abs(e1 - e0) <= 1e-10 and abs(e2 - e0) <= 1e-10
            assert np.linalg.norm(folded - g0) <= 1e-9 * np.linalg.norm(g0)

"""Segments of long primitive lists in units of several kets: one deeply contracted
atom ahead of a long chain of one-primitive shells, in energy mode and in both J/K
orientations, with units handed out by the fixed rule and claimed.  The counts of
evaluated and of skipped quartets are those of whole pairs, one ket per unit, and add
up to the unique quartets; energies to 1e-12 relative, gradients to 1e-11 of their
norm (another summation order).
"""
import numpy as np
import pytest

from shell_systems import deep_shell_chain

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def lib():
    from valence_amd import lib as L
    L.load()
    return L


@pytest.mark.parametrize("natom,nprim,ls", [(110, 40, (0,)), (180, 40, (0,)), (130, 12, (1,)), (90, 12, (0, 1))])
def test_counts_of_segments_in_chunks(lib, natom, nprim, ls):
    s = deep_shell_chain(natom, nprim, ls)
    plan = lib.launch_plan(s)[0]
    paired = [(m, q, plan[m, q, 1:7].astype(int).tolist()) for m in range(2) for q in range(21)
              if plan[m, q, 1:3].any() and plan[m, q, 5] > 1 and not plan[m, q, 0]]
    print(f"{natom} atoms, {nprim} primitives, l {ls}: {paired}", flush=True)
    assert {m for m, _, _ in paired} == {0, 1}
    npair = natom * len(ls) * (natom * len(ls) + 1) // 2
    unique = npair * (npair + 1) // 2
    got = []
    for chunk in (1, 0):
        with lib.Context(s, pair_chunk=chunk) as ctx:
            e, ce = ctx.energy(), ctx.counters()
            (eg, g), cg = ctx.energy_grad(), ctx.counters()
        print(f"  pair_chunk={chunk}: {e:.12f} {eg:.12f} {ce[0]:.0f}+{ce[2]:.0f} {cg[0]:.0f}+{cg[2]:.0f} of {unique}",
              flush=True)
        got.append((e, eg, g, ce, cg))
    (e0, eg0, g0, ce0, cg0), (e1, eg1, g1, ce1, cg1) = got
    assert abs(e1 - e0) <= 1e-12 * abs(e0) and abs(eg1 - eg0) <= 1e-12 * abs(eg0)
    assert np.linalg.norm(g1 - g0) <= 1e-11 * np.linalg.norm(g0)
    for a, b in ((ce1, ce0), (cg1, cg0)):
        assert a[0] == b[0] and a[2] == b[2] > 0
        assert a[0] + a[2] == unique

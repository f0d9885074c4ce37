"""Bases without some angular momenta, of few and of contracted shells: the energy
against the oracle to 1e-9 Eh, and the energy of the J/K pass to 1e-10 Eh of it, at three geometries; at
the widest no primitive pair of two atoms passes the screen.
Eight d shells, and one of six primitives, have more workgroups of the cooperative
kernel than any other class.
"""
import numpy as np
import pytest

import oracle
from shell_systems import shell_system

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def lib():
    from valence_amd import lib as L
    L.load()
    return L


@pytest.mark.parametrize("ls,natom,nprim", [((2,), 8, 1), ((2,), 1, 6), ((2,), 3, 2), ((1, 2), 4, 1), ((0, 2), 4, 1),
                                            ((1,), 6, 3), ((0,), 9, 2)])
def test_energy_matches_oracle(lib, ls, natom, nprim):
    s = shell_system(ls, natom, nprim)
    _, used, held = lib.launch_plan(s)
    print(f"l {ls}, {natom} atoms, {nprim} primitives: {used} of {held} partial sums", flush=True)
    assert used <= held
    with lib.Context(s) as ctx:
        for scale in (1.0, 1.5, 12.0):
            at = s.copy()
            at.coords = s.coords * scale
            ref = oracle.energy(at).energy
            e = ctx.energy(coords=at.coords)
            eg, g = ctx.energy_grad()
            print(f"  x{scale}: {e:.12f} J/K {eg:.12f} oracle {ref:.12f}", flush=True)
            assert abs(e - ref) <= 1e-9
            assert abs(eg - e) <= 1e-10 and np.all(np.isfinite(g))

"""Work lists of pair segments (small systems) against whole pairs.

A context picks, per quartet class, shell pairs or segments of their primitive
lists; pair_chunk=1 keeps whole pairs.  Both evaluate the same contracted
quartets: equal evaluated and skipped counts, energies and gradients within the
rounding of a sum taken in another order (1e-12 relative, 1e-11 of the
gradient's norm), for a closed-shell, a high-spin and a spin-coupled wave
function, and again after the geometry, and with it the lists, has changed.
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


def _high_spin():
    s = workloads.alkane_system(2, {"C": (6.0, workloads._type_shells(workloads.config1(), 0)),
                                    "H": (1.0, workloads._type_shells(workloads.config1(), 1))},
                                np.random.default_rng(7))
    s.nunpd, s.ndocc = 2, s.ndocc - 2
    return s


SYSTEMS = {"water": workloads.config0, "ethane_high_spin": _high_spin, "chain12": workloads.config2,
           "octane": workloads.config1}


@pytest.mark.parametrize("name", sorted(SYSTEMS))
def test_segments_match_whole_pairs(lib, name):
    s = SYSTEMS[name]()
    far = s.coords * 1.3  # fewer primitive pairs survive: other lists
    ref = {}
    for chunk in (1, 0):
        with lib.Context(s, pair_chunk=chunk) as ctx:
            for key, x in (("near", s.coords), ("far", far), ("near again", s.coords)):
                e = ctx.energy(s.coeff, x)
                ce = ctx.counters()
                eg, g = ctx.energy_grad(s.coeff, x)
                cg = ctx.counters()
                print(f"{name} {key} pair_chunk={chunk}: {e:.12f} {eg:.12f} {ce[0]:.0f}+{ce[2]:.0f}")
                if chunk == 1:
                    ref[key] = (e, eg, g, ce, cg)
                    continue
                r = ref[key]
                assert abs(e - r[0]) <= 1e-12 * abs(r[0]) and abs(eg - r[1]) <= 1e-12 * abs(r[1])
                assert np.linalg.norm(g - r[2]) <= 1e-11 * np.linalg.norm(r[2])
                for a, b in ((ce, r[3]), (cg, r[4])):
                    assert a[0] == b[0] and a[2] == b[2]

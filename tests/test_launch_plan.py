"""Launch plans on the host (vsvb_debug_plan), without a GPU.

Every workgroup of an energy writes four partial sums per part of its class, so
the buffer a context allocates has to hold what any geometry's launches write:
over the bases of every subset of {s, p, d}, few and many shells, contracted or
not, on devices of few and many compute units.
"""
import itertools

import pytest

from shell_systems import shell_system
from valence_amd import lib, workloads

SUBSETS = [c for n in (1, 2, 3) for c in itertools.combinations(range(3), n)]


@pytest.mark.parametrize("ls", SUBSETS, ids=lambda ls: "".join("spd"[l] for l in ls))
def test_partial_sums_fit_their_buffer(ls):
    for natom, nprim, ncu in itertools.product((1, 2, 7, 8, 30, 90), (1, 6), (1, 32, 256, 304)):
        _, used, held = lib.launch_plan(shell_system(ls, natom, nprim), ncu)
        assert used <= held, (natom, nprim, ncu, used, held)


def test_partial_sums_of_the_workloads_fit():
    for make in (workloads.config0, workloads.config1, workloads.config2, workloads.config4):
        _, used, held = lib.launch_plan(make())
        assert 0 < used <= held


def test_environment_does_not_change_a_plan(monkeypatch):
    """Plans follow the system alone: no environment variable selects their work lists."""
    s = workloads.config0()
    want = lib.launch_plan(s)[0]
    for value in ("0,0", "1,1", "2,2"):
        monkeypatch.setenv("VSVB_LV", value)
        assert (lib.launch_plan(s)[0] == want).all(), value


@pytest.mark.parametrize("make,shares", [(workloads.config0, True), (workloads.config1, False)])
def test_forced_chunks_keep_whole_pairs_and_separate_launches(make, shares):
    """pair_chunk > 0: shell pairs as work lists, a launch per class; by default some
    classes of these molecules take segments, and water's share a launch."""
    s = make()
    default = lib.launch_plan(s)[0]
    assert default[..., 1:3].any() and (default[..., 7].any() or not shares)
    for chunk in (1, 2, 64):
        forced = lib.launch_plan(s, pair_chunk=chunk)[0]
        assert not forced[..., 1:3].any() and not forced[..., 7].any()

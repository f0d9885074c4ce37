"""Quartet counts of a batch: those of a direct run and of every replay are the sums
over the wave functions' own contexts (energy + gradient), exactly; profiling on and
off, and at other coordinates.
"""
import numpy as np
import pytest

from valence_amd import workloads

pytestmark = pytest.mark.gpu


def test_replayed_counts_are_the_contexts_sums():
    from valence_amd import lib
    base = workloads.config1()
    basis = {"C": (6.0, workloads._type_shells(base, 0)), "H": (1.0, workloads._type_shells(base, 1))}
    systems = [workloads.config0(), workloads.alkane_system(1, basis, np.random.default_rng(1)), base]
    b = lib.Batch(systems)
    for scale, profile in ((1.0, False), (1.1, True), (1.1, False)):
        b.set_profiling(profile)
        b.set_coords([s.coords * scale for s in systems])
        want = np.zeros((21, 3))
        for s in systems:
            with lib.Context(s) as ctx:
                ctx.energy_grad(coords=s.coords * scale)
                want += ctx.class_stats()[:, 1:4]
        assert want.sum() > 0
        for rep in range(4):
            b.run(want_grad=True)
            got = b.class_stats()
            print(f"scale {scale} profile {profile} run {rep} graph {b.uses_graph()}: {got[:, 1:4].sum(0)}", flush=True)
            assert np.all(got[:, 1:4] == want)
            if profile:
                assert np.all(got[want[:, 0] > 0, 0] > 0.0)
        assert b.uses_graph()
    b.close()

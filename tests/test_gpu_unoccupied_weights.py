"""Weights of orbitals beyond the occupied ones (norbs > the electrons need) have no
part in the energy: their gradient is zero in every entry point, whatever the memory
held before, and the other weights' gradient is that of the system without them, to
1e-10 of its norm.  Water (one launch per orbital stage), C5H12 (a workgroup per
row), one and two spin densities, against the dense path too.
"""
import numpy as np
import pytest
import torch

from valence_amd import autograd, workloads

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


def _cases(name, unpaired):
    """The full system, the same with its last two orbitals empty, and without those two."""
    full = workloads.config0() if name == "water" else _alkane(5)
    full.nunpd, full.ndocc = unpaired, full.ndocc - unpaired
    s = full.copy()
    s.ndocc -= 2
    t = s.copy()
    cut = int(s.orb_start[s.nspatial])
    t.orb_natom, t.orb_atoms = s.orb_natom[:s.nspatial], s.orb_atoms[:s.nspatial]
    t.orb_start, t.xpset, t.coeff = s.orb_start[:s.nspatial + 1], s.xpset[:cut], s.coeff[:cut]
    return full, s, t, cut


@pytest.mark.parametrize("name,unpaired", [("water", 0), ("water", 1), ("pentane", 0), ("pentane", 2)])
def test_unoccupied_weights_have_no_gradient(lib, name, unpaired):
    full, s, t, cut = _cases(name, unpaired)
    assert 0 < cut < s.totlen
    with lib.Context(t) as ctx:
        e0, g0 = ctx.energy_grad()

    def check(entry, e, g):
        print(f"{name} nunpd={unpaired} {entry}: {e - e0:.1e} unoccupied {np.abs(g[cut:]).max():.3e}", flush=True)
        assert abs(e - e0) <= 1e-10
        assert np.all(g[cut:] == 0.0)
        assert np.linalg.norm(g[:cut] - g0) <= 1e-10 * np.linalg.norm(g0)

    for gim in (0, 1):
        with lib.Context(full, grid_inverse_min=gim) as ctx:  # its gradient stays in the freed memory
            ctx.energy_grad()
        with lib.Context(s, grid_inverse_min=gim) as ctx:
            check(f"context, grid_inverse_min={gim}", *ctx.energy_grad())
    lib.energy_grad_static(full)
    check("static", *lib.energy_grad_static(s))

    with lib.Context(s) as ctx:
        c = torch.tensor(s.coeff, dtype=torch.float64, device="cuda")
        e = torch.zeros(1, dtype=torch.float64, device="cuda")
        g = torch.full_like(c, float("nan"))
        ctx.energy_grad_device(c.data_ptr(), e.data_ptr(), g.data_ptr(), torch.cuda.current_stream().cuda_stream)
        check("device", float(e), g.cpu().numpy())
        c.requires_grad_(True)
        e = autograd.energy(ctx, c)
        e.backward()
        check("torch", float(e.detach()), c.grad.cpu().numpy())

    b = lib.Batch([full, full])
    b.run(want_grad=True)
    b.close()
    for members in (1, 2, 8):
        b = lib.Batch([s] * members)
        for rep in range(2):
            e, g = b.run(want_grad=True)
            for k in range(members):
                check(f"batch of {members}, run {rep}", e[k], g[k])
        b.close()

"""Closed-shell systems whose basis holds chosen angular momenta only."""
import numpy as np

from valence_amd import workloads


def shell_system(ls, natom, nprim=1, norb=2, seed=5):
    """natom atoms of charge 2 on a distorted grid (1.2 A), on each a shell of nprim primitives per
    angular momentum in ls; norb doubly occupied orbitals over two atoms each."""
    rng = np.random.default_rng(seed)
    shells = [(l, np.sort(np.exp(rng.uniform(np.log(0.3), np.log(3.0 if nprim == 1 else 30.0), nprim)))[::-1],
               rng.uniform(0.3, 1.0, nprim)) for l in ls]
    basis = {"X": (2.0, shells)}
    elems = ["X"] * natom
    side = int(np.ceil(natom ** (1 / 3)))
    xyz = 1.2 * np.array([[k % side, k // side % side, k // side ** 2] for k in range(natom)], float)
    xyz += rng.normal(0.0, 0.05, xyz.shape)
    atoms = [sorted({k % natom, (k + 1) % natom}) for k in range(norb)]
    orbs = [(a, workloads._rand_orbital(rng, basis, elems, a)) for a in atoms]
    return workloads.assemble(elems, xyz, basis, orbs)


def deep_shell_chain(natom, nprim, ls):
    """A chain of one-primitive shells, 1.6 A apart, behind one atom whose shells have nprim primitives: its
    pairs' long primitive lists are cut into segments, and the many others fill units of several kets."""
    rng = np.random.default_rng(11)
    basis = {"X": (2.0, [(l, np.array([0.9 - 0.2 * l]), np.ones(1)) for l in ls]),
             "Y": (4.0, [(l, np.sort(np.exp(rng.uniform(np.log(0.2), np.log(500.0), nprim)))[::-1],
                          rng.uniform(0.1, 1.0, nprim)) for l in ls])}
    elems = ["Y"] + ["X"] * (natom - 1)
    xyz = np.zeros((natom, 3))
    xyz[:, 0] = 1.6 * np.arange(natom)
    xyz += rng.normal(0.0, 0.05, xyz.shape)
    orbs = [(a, workloads._rand_orbital(rng, basis, elems, a)) for a in ([0, 1], [2, 3], [60, 61])]
    return workloads.assemble(elems, xyz, basis, orbs)

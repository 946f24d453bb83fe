"""Forces on j slots that two clusters share a group for (mixed form): the FP32
sum of each cluster's tile is converted to fixed point by itself, so a force is
the exact sum of the two.  Atoms of even clusters and atoms of odd clusters act
on the atoms of the last clusters (no others interact), by LJ and one kind at a
time: the forces with both kinds are the sums of the forces with each."""
import numpy as np
import pytest

import fenzi

pytestmark = pytest.mark.gpu

EDGE, L = 14, 30.8  # 2,744 atoms on a jittered lattice: above the size of entry lists


def _system(ctx, xyz, types, eps):
    n = len(xyz)
    topo = dict(n_atoms=n, n_types=4, charge=np.zeros(n), mass=np.full(n, 12.0), type=types.astype(np.int32),
                lj_eps=eps.ravel(), lj_sig2=np.full(16, 6.25), lj14_eps=np.zeros(16), lj14_sig2=np.ones(16))
    for f, w in (("bond", 2), ("angle", 3), ("dihedral", 4), ("improper", 4), ("constraint", 2)):
        topo["n_%ss" % f] = 0
        topo["%s_atoms" % f] = np.zeros(0, np.int32)
    for f in ("bond_k", "bond_r0", "angle_k", "angle_theta0", "ub_k", "ub_s0", "dihedral_k", "dihedral_delta",
              "improper_k", "improper_psi0", "constraint_length"):
        topo[f] = np.zeros(0)
    topo["dihedral_n"] = np.zeros(0, np.int32)
    params = dict(box=(L, L, L), cutoff=10.0, cuton=8.0, pairlist=11.0, beta=0.32, K=(32, 32, 32), dt_ps=0.001,
                  shake_tol=1e-8)
    return fenzi.System(ctx, topo, params, fenzi.MIXED, xyz=xyz)


def test_forces_of_two_clusters_add_exactly(ctx):
    rng = np.random.default_rng(12)
    g = np.stack(np.meshgrid(*[np.arange(EDGE)] * 3, indexing="ij"), -1).reshape(-1, 3) * (L / EDGE)
    xyz = g + rng.uniform(-0.3, 0.3, g.shape)
    n = len(xyz)
    s = _system(ctx, xyz, np.zeros(n), np.zeros((4, 4)))
    slots = s.cluster_layout()[2]
    cluster = np.empty(n, int)
    cluster[slots[slots >= 0]] = np.flatnonzero(slots >= 0) // 8
    last = cluster >= cluster.max() - 40  # nothing acts on a cluster after these
    types = np.where(last, 3, 1 + cluster % 2)
    f = {}
    for kinds in ((1, 2), (1,), (2,)):
        eps = np.zeros((4, 4))
        for k in kinds:
            eps[k, 3] = eps[3, k] = 0.15
        t = _system(ctx, xyz, types, eps)
        f[kinds] = t.forces()[0][last]
        t.close()
    assert (np.abs(f[(1,)]) > 1e-3).mean() > 0.9 and (np.abs(f[(2,)]) > 1e-3).mean() > 0.9
    # multiples of 2^-32 below 2^20: exact in FP64
    assert np.abs(f[(1, 2)]).max() < 2.0 ** 20
    assert np.array_equal(f[(1, 2)], f[(1,)] + f[(2,)])

"""A pair list of groups that outgrows its capacity: the build leaves the list
unwritten whichever of its blocks see the overflow flag first, and the call
grows, replays and ends bitwise where a run without the overflow ends.  The
largest case has more blocks of the group build than the device holds at once,
so that blocks start after the flag is up."""
import numpy as np
import pytest

import fenzi
import fz_synth

pytestmark = pytest.mark.gpu


def _water(n, L, seed):
    topo, xyz = fz_synth.make_system(0, n, (L, L, L), seed=seed, jitter=0.1)
    K = fz_synth.smooth235(int(np.ceil(L)))
    return topo, xyz, dict(box=(L, L, L), cutoff=10.0, cuton=8.0, pairlist=10.8, beta=0.32, K=(K, K, K),
                           dt_ps=0.001, shake_tol=1e-8)


@pytest.mark.parametrize("n,L", [(1400, 34.8), (25000, 91.0)])
def test_group_list_overflow_is_replayed_bitwise(ctx, n, L):
    topo, xyz, params = _water(n, L, seed=n)
    a, b = (fenzi.System(ctx, topo, params, fenzi.MIXED, xyz=xyz) for _ in range(2))
    for s in (a, b):
        s.reassign_velocities(400.0, 5, 0)
        s.step(4)
    pairs, _ = b.cluster_pairs()
    b.set_neighbor_capacity(len(pairs) // 2, 0)  # the list held does not fit: overflows at once
    b.set_neighbor_capacity(len(pairs), 0)  # it fits, a longer one does not
    assert b.info()["device_bytes"] < a.info()["device_bytes"]
    for _ in range(3):
        a.step(10)
        b.step(10)
        assert np.array_equal(a.get_fixed(), b.get_fixed())
        assert np.array_equal(a.get_state()[1], b.get_state()[1])
        assert a.energies()["list_builds"] == b.energies()["list_builds"]
        assert np.array_equal(a.cluster_pairs()[0], b.cluster_pairs()[0])


def test_evaluation_of_a_batch_with_an_overflowing_member(ctx):
    """fz_set_state's own evaluation overflows one member's list, among others'."""
    members = []
    for k, n in enumerate((1400, 1500, 1600)):
        topo, xyz, params = _water(n, 36.0, seed=60 + k)
        members.append(fenzi.System(ctx, topo, params, fenzi.MIXED, xyz=xyz))
    x = [s.get_state()[0] for s in members]
    v = [s.get_state()[1] for s in members]
    f = [s.forces()[0] for s in members]
    members[1].set_neighbor_capacity(len(members[1].cluster_pairs()[0]) // 2, 0)
    for s, x_, v_, f_ in zip(members, x, v, f):
        s.set_state(x_, v_)
        assert np.array_equal(s.forces()[0], f_)


def _groups(pairs, masks):
    """Groups of the list: per pair of clusters the j slots of both, of the first
    only and of the second only, eight to a group."""
    I, J = pairs[:, 0].astype(np.int64), pairs[:, 1].astype(np.int64)
    slots = masks.view(np.uint8).reshape(-1, 8) != 0
    key, at = np.unique((I >> 1) * (J.max() + 1) + J, return_inverse=True)
    near = np.zeros((2, len(key), 8), bool)
    near[I & 1, at] = slots
    s = key // (J.max() + 1)
    return int(sum(np.ceil(np.bincount(s, n.sum(1)) / 8.0).sum()
                   for n in (near[0] & near[1], near[0] & ~near[1], near[1] & ~near[0])))


def test_more_groups_than_half_the_entries(ctx):
    """Blobs of eight atoms, one to a column, those of neighbouring columns half a box
    apart: no j slot is near two clusters and every entry is a group.  The entries fit
    their capacity exactly, the groups do not fit the room that goes with it."""
    side, L = 16, (48.0, 48.0, 44.0)
    rng = np.random.default_rng(5)
    cx, cy = np.meshgrid(np.arange(side), np.arange(side), indexing="ij")
    centre = np.stack([3.0 * cx + 1.5, 3.0 * cy + 1.5, 10.0 + 22.0 * (cx % 2)], -1).reshape(-1, 1, 3)
    corner = np.stack(np.meshgrid([-0.5, 0.5], [-0.5, 0.5], [-0.5, 0.5], indexing="ij"), -1).reshape(1, 8, 3)
    xyz = (centre + corner + rng.uniform(-0.1, 0.1, (side * side, 8, 3))).reshape(-1, 3)
    n, z = len(xyz), np.zeros
    topo = dict(n_atoms=n, n_types=1, charge=np.tile([0.1, -0.1], n // 2), mass=np.full(n, 12.0), type=z(n, np.int32),
                lj_eps=z(1), lj_sig2=np.ones(1), lj14_eps=z(1), lj14_sig2=np.ones(1), dihedral_n=z(0, np.int32))
    for f in ("bond", "angle", "dihedral", "improper", "constraint"):
        topo["n_%ss" % f], topo["%s_atoms" % f] = 0, z(0, np.int32)
    for f in ("bond_k", "bond_r0", "angle_k", "angle_theta0", "ub_k", "ub_s0", "dihedral_k", "dihedral_delta",
              "improper_k", "improper_psi0", "constraint_length"):
        topo[f] = z(0)
    s = fenzi.System(ctx, topo, dict(box=L, cutoff=10.0, cuton=8.0, pairlist=11.0, beta=0.3125, K=(48, 48, 45),
                                     column_grid=(side, side)), fenzi.FP64, xyz=xyz)
    f0, e0 = s.forces()
    pairs, masks = s.cluster_pairs()
    clusters = len(s.cluster_layout()[2]) // 8
    assert clusters == side * side
    room = clusters + 8
    assert _groups(pairs, masks) > len(pairs) // 2 + 3 * ((room + 1) // 2)
    s.set_neighbor_capacity(len(pairs), room)
    f, e = s.forces()
    now, masks_now = s.cluster_pairs()
    order = lambda p, m: sorted(zip(p[:, 0].tolist(), p[:, 1].tolist(), m.tolist()))
    assert order(now, masks_now) == order(pairs, masks)
    assert e["list_builds"] == e0["list_builds"] and e["pairs_within_cutoff"] == e0["pairs_within_cutoff"]
    assert np.sqrt(((f - f0) ** 2).sum() / (f0 ** 2).sum()) < 1e-12  # the order of FP64 atomics
    s.close()


def test_device_memory_of_a_list(ctx):
    """Groups' room is made for the lists there are, not for the worst case (45.3 MB
    here, against 39.6 for a benchmark system of this size with plain entry lists)."""
    L = 41.6
    topo, _ = fz_synth.make_system(0, 2400, (L, L, L), seed=3)
    s = fenzi.System(ctx, topo, dict(box=(L, L, L), cutoff=9.0, cuton=7.0, pairlist=10.5, beta=0.34, K=(45, 45, 45)),
                     fenzi.FP64)
    assert s.info()["device_bytes"] < 42e6
    s.close()

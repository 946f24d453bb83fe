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

"""Forces through the device-side conversion (slot lookup, three sums, fixed-point
scale), and positions and velocities read together after an evaluation whose brick
records used the same scratch memory."""
import numpy as np
import pytest

import fenzi
import fz_synth

pytestmark = pytest.mark.gpu


def _water(n, L, K):
    topo, xyz = fz_synth.make_system(0, n, (L, L, L), seed=n, jitter=0.1)
    return topo, xyz, dict(box=(L, L, L), cutoff=9.0, cuton=7.0, pairlist=10.2, beta=0.34, K=(K, K, K), dt_ps=0.001,
                           shake_tol=1e-10)


@pytest.mark.parametrize("n,L,K", [(1, 21.0, 24), (300, 21.0, 24), (1500, 35.6, 36), (8200, 62.7, 64)])
def test_mixed_forces_are_the_fixed_point_sums(ctx, n, L, K):
    topo, xyz, params = _water(n, L, K)
    a, b = (fenzi.System(ctx, topo, params, fenzi.MIXED, xyz=xyz) for _ in range(2))
    b.step(3)  # another list's slots first
    b.set_state(xyz)
    f, g = a.forces()[0], b.forces()[0]
    assert np.array_equal(f, g)
    assert np.array_equal(f * 2.0 ** 32, np.rint(f * 2.0 ** 32)) and np.abs(f).max() < 2.0 ** 20
    a.close()
    b.close()


@pytest.mark.parametrize("prec", [fenzi.FP64, fenzi.MIXED])
def test_state_read_after_a_brick_evaluation(ctx, prec):
    topo, xyz, params = _water(8200, 62.7, 64)  # 24,600 atoms: the grid path spreads by bricks
    s = fenzi.System(ctx, topo, params, prec)
    assert s.set_launch(pme_path=fenzi.PME_GRID)["pme_path"] == fenzi.PME_GRID
    rng = np.random.default_rng(2)
    v = rng.normal(0.0, 3.0, xyz.shape)
    s.set_state(xyz, v)
    u = s.get_fixed()
    f0, e0 = s.forces()
    x, w = s.get_state()
    box = np.array(params["box"])
    back = u.astype(float) * (box * 2.0 ** -64)
    back -= np.where(back >= 0.5 * box, box, 0.0)
    assert np.array_equal(x, back) and np.array_equal(w, v)
    assert np.array_equal(s.get_fixed(), u)
    f1, e1 = s.forces()  # the scratch holds the state read: the next evaluation does not see it
    if prec == fenzi.MIXED:
        assert np.array_equal(f0, f1)
    assert e0["pairs_within_cutoff"] == e1["pairs_within_cutoff"] and e0["pme"] == pytest.approx(e1["pme"], rel=1e-12)
    s.close()

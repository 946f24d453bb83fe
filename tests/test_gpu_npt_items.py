"""Under a barostat the pair list may be allocated again at another box than the
system was created with; how its sums are cut into work items must stay.  The
system's estimated tiles lie just below the size from which items are longer,
and the box shrinks past it before one copy's list is allocated again."""
import numpy as np
import pytest

import fenzi
import fz_synth

pytestmark = pytest.mark.gpu


def test_list_allocated_again_in_a_smaller_box_keeps_the_sums(ctx):
    n, rc = 3133, 10.0
    pairs30 = 0.5 * (3 * n) ** 2 * (4.0 / 3.0 * np.pi * rc ** 3) / 30.0  # tiles = this / volume
    L = (pairs30 / (65536.0 * (1.0 - 1e-6))) ** (1.0 / 3.0)
    topo, xyz = fz_synth.make_system(0, n, (L, L, L), seed=8, jitter=0.1)
    params = dict(box=(L, L, L), cutoff=rc, cuton=8.0, pairlist=11.0, beta=0.3125, K=(48, 48, 48), dt_ps=0.001,
                  shake_tol=1e-8)
    a, b = (fenzi.System(ctx, topo, params, fenzi.MIXED, xyz=xyz) for _ in range(2))
    for s in (a, b):
        s.reassign_velocities(300.0, 4, 0)
        s.set_barostat(2e4, 1e-4)
        s.step(40)
        assert s.barostat()["volume"] < L ** 3 * (1.0 - 1e-5)
    pairs, _ = b.cluster_pairs()
    b.set_neighbor_capacity(2 * len(pairs), 0)
    for _ in range(2):
        for s in (a, b):
            s.step(10)
        assert np.array_equal(a.get_fixed(), b.get_fixed())
        assert np.array_equal(a.get_state()[1], b.get_state()[1])

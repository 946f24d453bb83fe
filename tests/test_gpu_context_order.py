"""A context may be destroyed before the systems and batches made with it (the
interpreter ends a cycle of objects in any order): they keep what they need."""
import numpy as np
import pytest

import fenzi
import systems

pytestmark = pytest.mark.gpu


def test_systems_and_batches_outlive_their_context():
    topo, xyz, params = systems.water_box()
    ctx = fenzi.Context(0)
    a, b = (fenzi.System(ctx, topo, params, fenzi.MIXED, xyz=xyz) for _ in range(2))
    batch = fenzi.Batch(ctx, [b])
    ctx.close()
    np.arange(64).tolist()  # the freed words are taken again
    other = [fenzi.Context(0) for _ in range(4)]
    a.step(5)
    batch.step(5)
    assert np.array_equal(a.get_fixed(), b.get_fixed())
    batch.close()
    a.close()
    b.close()
    for c in other:
        c.close()

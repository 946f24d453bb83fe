"""A build that needs more clusters than there is room for is left out and
repeated after the arrays have grown.  What the evaluation runs after it must
not use its cluster count (slot copies) nor the slots of the list before (COM
restraint): they may lie past the arrays of now."""
import numpy as np
import pytest

import fenzi
import systems

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("prec", [fenzi.FP64, fenzi.MIXED])
@pytest.mark.parametrize("n_waters,L", [(300, 26.0), (1700, 40.0)])
def test_evaluation_short_of_clusters_grows_them(ctx, prec, n_waters, L):
    topo, xyz, params = systems.slab(n_chains=2, n_waters=n_waters, L=L, seed=3, K=(40, 40, 40))
    n = topo["n_atoms"]
    s = fenzi.System(ctx, topo, params, prec, xyz=xyz)
    g = np.full(n, -1, np.int32)
    g[:38], g[n - 60:] = 0, 1  # the last slots of the list among them
    s.set_com_restraint(g, (1.0, 2.0, 3.0), 0.5)
    f0, e0 = s.forces()
    clusters = len(s.cluster_layout()[2]) // 8
    least = n // 8 + 1
    assert least < clusters and (8 * least) % 256  # fewer than the list has, no whole block of slots
    s.set_neighbor_capacity(0, least)
    f, e = s.forces()
    assert len(s.cluster_layout()[2]) // 8 == clusters
    if prec == fenzi.MIXED:
        assert np.array_equal(f, f0)
    else:
        assert systems.rel_rms(f, f0) < 1e-12  # the order of FP64 atomics
    assert e["pairs_within_cutoff"] == e0["pairs_within_cutoff"]
    s.close()

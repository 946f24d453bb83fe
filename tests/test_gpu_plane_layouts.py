"""The plane kernels on planes whose padded lines would not fit a compute unit's
160 KiB of LDS (the unpadded layout), in both forms, against the grid passes."""
import numpy as np
import pytest

import fenzi
import fz_synth
import systems

pytestmark = pytest.mark.gpu

# plane points x K2 planes: at least a plane per 256 points of one
CASES = [(fenzi.MIXED, (96, 96, 40)), (fenzi.MIXED, (100, 100, 40)), (fenzi.MIXED, (90, 108, 45)),
         (fenzi.FP64, (64, 75, 20)), (fenzi.FP64, (72, 60, 20)), (fenzi.FP64, (60, 80, 24))]


@pytest.mark.parametrize("prec,K", CASES)
def test_unpadded_planes_match_the_grid_passes(ctx, prec, K):
    box = (30.0, 31.0, 24.0)
    topo, xyz = fz_synth.make_system(2, 500, box, seed=sum(K), jitter=0.1)
    params = dict(box=box, cutoff=9.0, cuton=7.0, pairlist=10.2, beta=0.34, K=K, dt_ps=0.001, shake_tol=1e-10)
    csz = 8 if prec == fenzi.MIXED else 16
    assert (2 * K[0] * K[1] + K[0] + K[1]) * csz <= 163840  # a plane fits
    # its padded lines do not: a first pass of eight points or less in the mixed form, of four in FP64
    assert 2 * K[0] * K[1] * (9 / 8 if prec == fenzi.MIXED else 5 / 4) * csz > 163840
    got = {}
    for path in (fenzi.PME_AUTO, fenzi.PME_GRID):
        s = fenzi.System(ctx, topo, params, prec, xyz=xyz)
        used = s.set_launch(pme_path=path)["pme_path"]
        assert used == (fenzi.PME_PLANES if path == fenzi.PME_AUTO else fenzi.PME_GRID)
        got[path] = s.forces()
        s.close()
    (f, e), (fg, eg) = got[fenzi.PME_AUTO], got[fenzi.PME_GRID]
    if prec == fenzi.MIXED:
        assert np.array_equal(f, fg) and e["pme"] == eg["pme"]
    else:  # the order of FP64 sums differs
        assert systems.rel_rms(f, fg) < 1e-12 and abs(e["pme"] - eg["pme"]) <= 1e-12 * abs(eg["pme"]) + 2.0 ** -27

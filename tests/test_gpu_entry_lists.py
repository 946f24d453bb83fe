"""Entry lists of small systems in the mixed form (pair sums in list order).

The recorded trajectory (golden/mixed_small.npz: forces of the initial frame,
fixed-point positions and velocities after 20 moves of the minimiser and 80
steps of 2 fs) is the one this library gave when every system kept an entry
list and one wave ran a chunk of 32 entries: a system of about 1,000 atoms
multiplies a difference in the order of FP32 sums some eightfold in 40 steps,
so its frames agree with those of earlier versions only if the sums do, to the
bit.  Either side of the size limit is compared with the oracle, and a batch
of both kinds with the members alone."""
import os

import numpy as np
import pytest

import fenzi
import fz_synth
import oracle
import systems

pytestmark = pytest.mark.gpu

GOLDEN = os.path.join(os.path.dirname(os.path.abspath(__file__)), "golden", "mixed_small.npz")


def test_trajectory_of_a_small_system_is_the_recorded_one(ctx):
    topo, xyz = fz_synth.make_system(4, 293, (24.0, 24.0, 24.0), seed=7)
    params = dict(box=(24.0, 24.0, 24.0), cutoff=10.0, cuton=8.0, pairlist=11.5, beta=0.3125, K=(24, 24, 24),
                  dt_ps=0.002, shake_tol=1e-8)
    ref = np.load(GOLDEN)
    s = fenzi.System(ctx, topo, params, fenzi.MIXED, xyz=xyz)
    assert np.array_equal(s.forces()[0], ref["forces"])
    s.minimize(20, 0.05)
    s.reassign_velocities(300.0, 3, 0)
    for n in (1, 39, 40):
        s.step(n)
    assert np.array_equal(s.get_fixed(), ref["u"])
    assert np.array_equal(s.get_state()[1], ref["v"])


def _water(n, L, rc=10.0):
    topo, xyz = fz_synth.make_system(0, n, (L, L, L), seed=5 + n, jitter=0.1)
    K = fz_synth.smooth235(int(np.ceil(L)))
    return topo, xyz, dict(box=(L, L, L), cutoff=rc, cuton=rc - 2.0, pairlist=rc + 1.2, beta=0.32, K=(K, K, K),
                           dt_ps=0.001, shake_tol=1e-10)


# pair tiles estimated from the density: 0 .. 15,900 keep entries, 17,200 groups
SIZES = {"one_entry": (2, 21.0), "a_chunk": (16, 21.0), "below": (770, 28.6), "above": (800, 28.6)}


@pytest.mark.parametrize("name", sorted(SIZES))
def test_forces_vs_oracle_either_side_of_the_limit(ctx, name):
    topo, xyz, params = _water(*SIZES[name])
    orc = oracle.Oracle(topo, params)
    u = orc.to_fixed(xyz)
    f_ref, _, _ = orc.forces(u)
    s = fenzi.System(ctx, topo, params, fenzi.MIXED)
    s.set_fixed(u)
    f, e = s.forces()
    assert systems.rel_rms(f, f_ref) < 1e-5  # the mixed form's tolerance
    assert systems.pair_count_ok(e["pairs_within_cutoff"], orc, u, params["cutoff"], True)
    s.close()


def test_batch_of_both_kinds_matches_its_members_alone(ctx):
    names = ["above", "below", "a_chunk", "above", "one_entry"]
    alone, members = [], []
    for k, n in enumerate(names):
        topo, xyz, params = _water(*SIZES[n])
        for group in (alone, members):
            s = fenzi.System(ctx, topo, params, fenzi.MIXED, xyz=xyz)
            s.reassign_velocities(300.0, 20 + k, 0)
            group.append(s)
    b = fenzi.Batch(ctx, members)
    for n in (1, 30):
        b.step(n)
        for a, m in zip(alone, members):
            a.step(n)
            assert np.array_equal(a.get_fixed(), m.get_fixed())
            assert np.array_equal(a.get_state()[1], m.get_state()[1])
            assert a.energies()["potential"] == m.energies()["potential"]
    b.close()


def test_batch_with_a_wave_per_chunk_matches_its_members_alone(ctx):
    """Many chunks in one launch (about 800 estimated per member, from 4,096 on a wave
    each), an odd and a tiny list among them."""
    alone, members = [], []
    for k, n in enumerate(["below"] * 6 + ["a_chunk", "one_entry"]):
        topo, xyz, params = _water(*SIZES[n])
        for group in (alone, members):
            s = fenzi.System(ctx, topo, params, fenzi.MIXED, xyz=xyz)
            s.reassign_velocities(300.0, 40 + k, 0)
            group.append(s)
    b = fenzi.Batch(ctx, members)
    b.step(30)
    for a, m in zip(alone, members):
        a.step(30)
        assert np.array_equal(a.get_fixed(), m.get_fixed())
        assert np.array_equal(a.get_state()[1], m.get_state()[1])
        ea, em = a.energies(), m.energies()
        for k in ("potential", "vdw", "elec", "pairs_within_cutoff", "pair_tiles", "list_builds"):
            assert ea[k] == em[k], k
    b.minimize(2, 0.02)  # the other energy levels
    for a, m in zip(alone, members):
        a.minimize(2, 0.02)
        assert np.array_equal(a.get_fixed(), m.get_fixed())
        assert a.energies()["potential"] == m.energies()["potential"]
    b.close()

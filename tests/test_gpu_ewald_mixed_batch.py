"""Batches in which some systems have the real-space Ewald polynomials and one has
not (beta times cutoff above 3.5): every member's reported energies are those it
has alone, whatever the others are.  Charges 300 times the usual ones, so that a
term's last bits reach the energies' 2^-28 kcal/mol."""
import numpy as np
import pytest

import fenzi
import systems

pytestmark = pytest.mark.gpu


def _members(ctx, prec):
    got = []
    # 4.0 has no polynomials; 3.2 has; the last is large enough for pair groups in both forms
    for k, (n_waters, L, K, beta) in enumerate(((300, 24.0, 24, 0.32), (280, 24.0, 24, 0.40), (1500, 37.0, 40, 0.32))):
        topo, xyz, params = systems.slab(n_chains=3, n_waters=n_waters, L=L, seed=70 + k, K=(K, K, K))
        topo = dict(topo, charge=300.0 * np.asarray(topo["charge"]))
        got.append(fenzi.System(ctx, topo, dict(params, beta=beta), prec, xyz=xyz))
    return got


@pytest.mark.parametrize("prec", [fenzi.FP64, fenzi.MIXED])
def test_member_energies_do_not_depend_on_the_batch(ctx, prec):
    members = _members(ctx, prec)
    alone = [s.forces()[1] for s in members]
    b = fenzi.Batch(ctx, members)
    b.minimize(0, 0.02)  # the evaluation alone
    for e, s in zip(alone, members):
        now = s.energies()
        for k in ("vdw", "elec"):
            assert e[k] == now[k], k
    b.close()

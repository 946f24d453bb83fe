"""The FP64 form's real-space Ewald energy of one pair, relative to itself, from
short range to the cutoff: the charges make it 1e9 kcal/mol, of which the
accumulators' 2^-28 steps are 4e-18 (their range is 3.4e10)."""
import math

import numpy as np
import pytest

import fenzi

pytestmark = pytest.mark.gpu

CC, L, RC = 332.0716, 32.0, 10.0


def _pair(ctx, beta, q):
    z = np.zeros
    topo = dict(n_atoms=2, n_types=1, charge=np.array([q, -q]), mass=np.full(2, 12.0), type=z(2, np.int32),
                lj_eps=z(1), lj_sig2=np.ones(1), lj14_eps=z(1), lj14_sig2=np.ones(1), dihedral_n=z(0, np.int32))
    for f, w in (("bond", 2), ("angle", 3), ("dihedral", 4), ("improper", 4), ("constraint", 2)):
        topo["n_%ss" % f], topo["%s_atoms" % f] = 0, z(0, np.int32)
    for f in ("bond_k", "bond_r0", "angle_k", "angle_theta0", "ub_k", "ub_s0", "dihedral_k", "dihedral_delta",
              "improper_k", "improper_psi0", "constraint_length"):
        topo[f] = z(0)
    return fenzi.System(ctx, topo, dict(box=(L, L, L), cutoff=RC, cuton=8.0, pairlist=11.0, beta=beta, K=(32, 32, 32)))


@pytest.mark.parametrize("beta", [0.05, 0.2, 0.3125, 0.35])
@pytest.mark.parametrize("r", [0.9, 2.7, 5.3, 8.1, 9.4, 9.99])
def test_pair_energy_keeps_its_relative_accuracy(ctx, beta, r):
    q = math.sqrt(1e9 * r / (CC * math.erfc(beta * r)))
    s = _pair(ctx, beta, q)
    u = np.zeros((2, 3), np.uint64)
    u[1, 0] = int(r / L * 2.0 ** 64)
    s.set_fixed(u)
    e = s.forces()[1]["elec"]
    x = int(u[1, 0]) * (L / 2.0 ** 64)
    ref = -CC * q * q * math.erfc(beta * x) / x
    # the argument's rounding counts 2 z^2 times on either side (z^2 <= 12.25, 1e-16), the
    # other factors a few times 1e-16; 2^-29 the energy's own steps
    assert abs(e - ref) <= 1e-14 * abs(ref) + 2.0 ** -29
    s.close()

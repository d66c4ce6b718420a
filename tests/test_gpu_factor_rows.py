"""The time-invariant factorisations on meshes around their chunks of 64 rows
and lines, against the oracle, with the tolerance that the oracle's own
reorderings give (as the other engine tests)."""

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

from oracle.engine import HestonOracle, HestonParams
from tests.parity import grid_tolerance, alternates

SIZES = [(4, 4), (5, 64), (64, 65), (65, 63), (66, 128), (129, 129), (130, 5), (194, 66)]


@pytest.mark.parametrize("barrier", [False, True])
@pytest.mark.parametrize("scheme, theta", [("douglas", 0.5), ("hundsdorferverwer", 0.7)])
def test_factors_match_oracle(gpu, scheme, theta, barrier):
    import fd_adi_amd
    P, S, V, O = [], [], [], []
    for k, (nS, nv) in enumerate(SIZES):
        x, y = np.arange(nS) / (nS - 1.0), np.arange(nv) / (nv - 1.0)
        S.append(400.0 * (0.3 * x + 0.7 * x ** 2))
        V.append(0.5 * (0.2 * y + 0.8 * y ** 2))
        P.append(dict(r=0.03, kappa=1.5, theta=0.06, sigma=0.25, rho=-0.5, barrier=barrier))
        O.append(HestonOracle(HestonParams(strike=100, r=0.03, v0=0.06, kappa=1.5, theta=0.06,
                                           sigma=0.25, rho=-0.5,
                                           barrier=S[-1][-1] if barrier else None), S[-1], V[-1]))
    dts = [0.01] * len(SIZES)
    hb = fd_adi_amd.HestonBatch(P, S, V, dts)
    hb.set_state([o.payoff() for o in O])
    hb.configure(scheme, theta)
    hb.step(4)
    for k, (got, o) in enumerate(zip(hb.get_state(), O)):
        solve = lambda e: getattr(e, "solve_" + scheme)(4, 0.01, o.payoff(), theta=theta)
        want = solve(o)
        tol, _ = grid_tolerance(want, [solve(a) for a in alternates(o)])
        err = float(np.max(np.abs(got - want)))
        assert err <= tol, (SIZES[k], err, tol)

"""Line solves around the solver's chunks of 64 rows, its groups of eight
lines and the longest line kept on chip (384 rows), along both axes, with
residuals, Dirichlet rows and folded boundary rows, against the oracle.

The systems are I - 0.01 A of the Heston operators on gentle meshes.  Both
sides eliminate without pivoting in FP64: about 8 roundings of 1.1e-16 a row
forward and back, damped along the line, on well-conditioned rows: 1e-12 of
the largest value leaves three decades."""

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

from oracle.engine import HestonOracle, HestonParams


@pytest.mark.parametrize("nS, nv", [(4, 4), (5, 7), (63, 8), (64, 9), (65, 16), (66, 17),
                                    (129, 65), (8, 64), (9, 66), (384, 5), (385, 6), (449, 12),
                                    (7, 384), (6, 386), (450, 450)])
@pytest.mark.parametrize("barrier", [None, 400.0])
def test_solve_matches_oracle(gpu, nS, nv, barrier):
    from fd_adi_amd.FiniteDifferenceEngineGPU import HestonFiniteDifferenceEngine
    from fd_adi_amd.Option import HestonOption, HestonBarrierOption
    kw = dict(spot=100, strike=100, interest_rate=0.03, variance=0.04, tenor=1.0,
              mean_reversion=1.0, mean_variance=0.12, vol_of_variance=0.3, correlation=-0.4)
    opt = HestonBarrierOption(top=(False, barrier), **kw) if barrier else HestonOption(**kw)
    x, y = np.arange(nS) / (nS - 1.0), np.arange(nv) / (nv - 1.0)
    G = HestonFiniteDifferenceEngine(opt, spots=(barrier or 500.0) * (0.3 * x + 0.7 * x ** 2),
                                     vars=0.2 * y + 0.8 * y ** 2, force_exact=False)
    O = HestonOracle(HestonParams(spot=100, strike=100, r=0.03, v0=0.04, T=1.0, kappa=1.0,
                                  theta=0.12, sigma=0.3, rho=-0.4, barrier=barrier),
                     G.spots, G.vars)
    G.set_zero_derivative()
    G.scale_and_combine_operators()
    V = np.random.default_rng(nS).random(G.shape) * 10
    for k in (0, 1):
        L = G.operators[k].mul_scalar_from_host(-0.01).add(1, inplace=True)
        want = (O.operators[k] * -0.01).add(1).solve(V)
        tol = 1e-12 * np.max(np.abs(want))
        assert np.max(np.abs(L.solve(V) - want)) <= tol
        if L.is_foldable():
            L.diagonalize()
            assert np.max(np.abs(L.solve(V) - want)) <= tol
            L.undiagonalize()

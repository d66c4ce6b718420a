"""y += A x and y -= A x in one launch: bit for bit the product followed by
the elementwise sum, for both axes (plain, folded, with and without residual)
and the cross derivative, up to work-groups' remainders."""

import numpy as np
import numpy.testing as npt
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nS, nv", [(20, 12), (16, 16), (33, 31)])
def test_apply_add_equals_apply_and_sum(gpu, nS, nv):
    from fd_adi_amd.FiniteDifferenceEngineGPU import HestonFiniteDifferenceEngine
    from fd_adi_amd.Option import HestonOption
    from fd_adi_amd.SizedArrayPtr import SizedArrayPtr
    opt = HestonOption(spot=100, strike=100, interest_rate=0.03, variance=0.04, tenor=1.0,
                       mean_reversion=1.0, mean_variance=0.12, vol_of_variance=0.3,
                       correlation=0.4)
    G = HestonFiniteDifferenceEngine(opt, nspots=nS, nvols=nv, spot_max=500.0, var_max=1.0)
    G.set_zero_derivative()
    G.scale_and_combine_operators()
    rng = np.random.default_rng(nS)
    x, y = rng.random(G.shape) * 10, rng.random(G.shape) * 10
    X = SizedArrayPtr(x)

    def check(L):
        Ax = L.apply(x)
        for minus, want in ((False, y + Ax), (True, y - Ax)):
            Y = SizedArrayPtr(y)
            L.apply_add_(X, Y, minus)
            npt.assert_array_equal(Y.to_numpy(), want)
        Y = SizedArrayPtr(y)
        L.apply_to_(X, Y)
        npt.assert_array_equal(Y.to_numpy(), Ax)
        with pytest.raises(ValueError):
            L.apply_add_(X, X)
        with pytest.raises(ValueError):
            L.apply_add_(X, SizedArrayPtr(np.zeros(x.size + 1)))

    for L in G.operators.values():
        check(L)
        L.enable_residual(False)
        check(L)
        if L.is_foldable():
            L.diagonalize()
            check(L)

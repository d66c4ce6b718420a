"""Predictions against the NumPy network with the kernels' bf16 roundings, for
each of the three row blocks of the inference kernel (32, 64 and 48 rows) and
feature counts up to the largest.

Both sides round the input, four activations and the weights to bf16; where their
fp32 sums straddle a rounding, an activation differs by a unit of 2^-8.  Five
such layers bound the difference by 2e-2 in the norm over the rows."""

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

from oracle import mlp_ref as R


@pytest.mark.parametrize("n, nin", [(1, 8), (33, 1), (8192, 13), (8193, 16), (16384, 8), (16385, 8),
                                    (30001, 16)])
def test_prices_match_the_numpy_network(gpu, n, nin):
    from fd_adi_amd.surrogate import MLP, init_params
    lo, hi = -np.ones(nin), 2 * np.ones(nin)
    p = init_params(3, nin)
    P = np.random.default_rng(n).uniform(-1, 2, (n, nin))
    m = MLP(lo, hi, 1.5, 2.0, params=p, max_rows=128)
    got = (m.predict(P) - 1.5) / 2.0
    rows = np.unique(np.r_[0:min(n, 150), max(0, n - 150):n])
    want = R.forward(p.astype(np.float64), R.features(P[rows], lo, hi), bf16=True)[0]
    rel = np.linalg.norm(got[rows] - want) / np.linalg.norm(want)
    print("n = %d, %d features: %.2e" % (n, nin, rel))
    assert rel < 2e-2

"""The network on blocks of 32 and 64 rows: prices and gradients at row
counts on both sides of a block's edge and of the change from 32-row to
64-row blocks.  A row's price does not depend on the rows around it, bit for
bit; gradients are held to the NumPy reference with the 12 bf16 roundings an
element passes at most (4 activations, 4 derivatives, 4 back-propagated
gradients, each 2^-9 relative: 2.3e-2) as tolerance."""

import numpy as np
import numpy.testing as npt
import pytest

pytestmark = pytest.mark.gpu

from oracle import mlp_ref as R


@pytest.fixture(scope="module")
def net(gpu):
    from fd_adi_amd import surrogate as S
    m = S.MLP(S.BOX_LO, S.BOX_HI, 1.5, 2.0, seed=3, max_rows=1024)
    P = S.draw_params(16500, 4)
    return m, P, m.predict(P[:8192])


@pytest.mark.parametrize("n", [1, 15, 17, 31, 33, 64, 8191, 8193, 8257, 16500])
def test_prices_do_not_depend_on_the_batch(net, n):
    m, P, want = net
    got = m.predict(P[:n])
    k = min(n, 8192)
    npt.assert_array_equal(got[:k], want[:k])
    # the rows beyond the first 8192, against a batch of 32-row blocks
    if n > 8192:
        npt.assert_array_equal(got[8192:], np.concatenate(
            [m.predict(P[a:min(a + 5000, n)]) for a in range(8192, n, 5000)]))


@pytest.mark.parametrize("rows", [1, 31, 33, 127, 129, 640])
def test_gradients_at_ragged_batches(gpu, rows):
    from fd_adi_amd.SizedArrayPtr import SizedArrayPtr
    from fd_adi_amd.surrogate import MLP, init_params
    rng = np.random.default_rng(rows)
    lo, hi = -np.ones(8), 2 * np.ones(8)
    p = init_params(3, 8)
    P = rng.uniform(-1, 2, (700, 8))
    t = np.sin(P.sum(axis=1))
    idx = rng.permutation(700)[:rows].astype(np.int32)
    m = MLP(lo, hi, 0.0, 1.0, params=p, max_rows=1024)
    dP, dT = SizedArrayPtr(P), SizedArrayPtr(t)
    m.grad(dP, dT, None, 640)  # leaves its rows in the buffers
    pad = np.zeros((rows + 1) // 2 * 2, dtype=np.int32)
    pad[:rows] = idx
    loss = m.grad(dP, dT, SizedArrayPtr(pad.view(np.float64).copy()), rows)
    g = m.grads().astype(np.float64)
    ref_loss, ref = R.loss_and_grad(p.astype(np.float64), R.features(P[idx], lo, hi), t[idx],
                                    bf16=True)
    npt.assert_allclose(loss, ref_loss, rtol=2.3e-2)
    offs, o4, ob4, _ = R.layout()
    for a, b in ([(ow, ob) for ow, ob in offs] + [(ob, ob + R.N_H) for _, ob in offs]
                 + [(o4, ob4)]):
        rel = np.linalg.norm(g[a:b] - ref[a:b]) / np.linalg.norm(ref[a:b])
        assert rel < 2.3e-2, (a, b, rel)

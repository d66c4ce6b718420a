"""Prices written into the memory of the features they come from: bit for bit
those written elsewhere, at the start, inside and at the end of the rows, in one
part and in several, with and without allocation."""

import ctypes

import numpy as np
import numpy.testing as npt
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("name, n", [("fdadi_mlp_predict", 1), ("fdadi_mlp_predict", 33),
                                     ("fdadi_mlp_predict", 5128), ("fdadi_mlp_predict", 5129),
                                     ("fdadi_mlp_predict", 40000),
                                     ("fdadi_mlp_predict_noalloc", 4096)])
def test_prices_in_the_features_memory(gpu, name, n):
    from fd_adi_amd import _lib, surrogate as S
    from fd_adi_amd.SizedArrayPtr import SizedArrayPtr
    m = S.MLP(S.BOX_LO, S.BOX_HI, 1.5, 2.0, seed=3, max_rows=128)
    P = S.draw_params(n, 5)
    want = m.predict(P)
    # a part's prices must not fall on later parts' rows: the start alone there
    for at in (0,) if n > 5128 else (0, 3, 4 * n, 7 * n):
        buf = SizedArrayPtr(np.concatenate([P.ravel(), np.zeros(8)]))
        out = ctypes.c_void_p(buf.p.value + 8 * at)
        _lib.call(name, m._h, buf.p, n, out, m.stream)
        npt.assert_array_equal(buf.to_numpy()[at:at + n], want)

"""Line solves whose pivots lie at the ends of the exponent range: 1 / p
overflows to an infinity of p's sign below 2^-1024 and is itself subnormal
above 2^1022, as the IEEE division has it.

The pivot stands on the last row of a diagonal line, so x there is
(1 / p) d with d = +-1: one rounding of the quotient, held to two units of
2^-52 (relative) or of 2^-1074 (subnormal results)."""

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

TINY = 5e-324
PIVOTS = [TINY, 1e-320, 1e-310, 2.0 ** -1025, 2.0 ** -1024,
          2.0 ** -1024 + TINY, 2.0 ** -1024 + 2.0 ** -1054, 2.0 ** -1024 + 2.0 ** -1046, 2.0 ** -1023, 1.5 * 2.0 ** -1023,
          2.0 ** -1022, 1e-300, 0.3, 1.0, 3e7, 1e300, 2.0 ** 1021, 1.7 * 2.0 ** 1021, 2.0 ** 1022,
          1e308, np.finfo(float).max, np.inf, 0.0, np.nan]


@pytest.mark.parametrize("n", [3, 65, 450])  # within a chunk, across chunks, kept in scratch
def test_pivots_at_the_ends_of_the_range(gpu, n):
    from fd_adi_amd.BandedOperatorGPU import BandedOperator, HostBandedOperator
    piv = np.array(PIVOTS + [-p for p in PIVOTS])
    blocks = piv.size
    mid = np.ones((blocks, n))
    mid[:, -1] = piv
    data = np.zeros((3, blocks * n))
    data[1] = mid.ravel()
    L = BandedOperator(HostBandedOperator(data, (1, 0, -1), None, axis=1, blocks=blocks))
    d = np.where(np.arange(blocks) % 3 == 0, -1.0, 1.0)
    V = np.ones((blocks, n))
    V[:, -1] = d
    got = L.solve(V)[:, -1]
    with np.errstate(all="ignore"):
        want = (1.0 / piv) * d
    finite = np.isfinite(want)
    print(np.c_[piv, want, got])
    np.testing.assert_array_equal(got[~finite], want[~finite])
    err = np.abs(got[finite] - want[finite])
    assert np.all(err <= np.maximum(2 * 2.0 ** -52 * np.abs(want[finite]), 2 * TINY))
    np.testing.assert_array_equal(np.signbit(got[finite]), np.signbit(want[finite]))

"""The semi-analytic price on both sides of what its short form takes: small
sigma (the short form starts at 1e-3), mean reversion below sigma rho / 2 (the
drift's real part changes sign), no mean reversion, no variance, strikes far
out, against the same quadrature in 80-bit arithmetic with the complex
functions of the formula as it is written.

Each node's exponent is a difference magnified by kappa theta / sigma^2, so 100
roundings of 2.2e-16 of (1 + kappa theta / sigma^2) on the spot bound the
error, and 1e-9 below that."""

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

#        S0,  K,   r,    v0,   T,    kappa, theta, sigma,   rho
ROWS = [[100, 100, 0.05, 0.04, 1.0, 2.0, 0.04, 0.999e-3, -0.5],
        [100, 100, 0.05, 0.04, 1.0, 2.0, 0.04, 1.001e-3, -0.5],
        [100, 100, 0.05, 0.04, 1.0, 2.0, 0.04, 1e-2, 0.5],
        [100, 90, 0.0, 0.04, 2.0, 0.2, 0.04, 1.5, 0.9],
        [100, 90, 0.0, 0.04, 2.0, 0.3375, 0.04, 0.75, 0.9],
        [100, 110, 0.03, 0.04, 0.5, 0.0, 0.04, 0.6, -0.9],
        [100, 110, 0.03, 0.04, 0.5, 1.0, 0.0, 0.6, 0.3],
        [100, 110, 0.03, 0.0, 0.5, 1.0, 0.09, 0.6, 0.0],
        [100, 30, 0.03, 0.04, 5.0, 5.0, 0.16, 1.0, -0.9],
        [100, 300, 0.03, 0.04, 0.1, 0.5, 0.01, 0.1, -0.9],
        [100, 100, 0.01, 0.01, 0.01, 5.0, 0.16, 1.0, -0.999],
        [1e-3, 1.1e-3, 0.01, 0.09, 1.0, 1.0, 0.09, 30.0, -0.2]]


def reference(X):
    from fd_adi_amd.pricing import gauss_legendre
    L = np.longdouble
    S, K, r, v0, T, kappa, theta, sigma, rho = X.astype(L).T[:, :, None]
    x1, w1 = (a.astype(L) for a in gauss_legendre(512))
    x2, w2 = (a.astype(L) for a in gauss_legendre(64))
    c = np.sqrt(1 - rho * rho) * (v0 + kappa * theta * T) / sigma
    a = np.clip(20 / c, 10, 20000)
    t = (x2 + 1) / 2
    u = np.concatenate([a * (x1 + 1) / 2, a / t], 1)
    w = np.concatenate([a * w1 / 2, a * w2 / 2 / t ** 2], 1)
    s2, q = sigma * sigma, u * u + L(0.25)
    xi = (kappa - sigma * rho / 2) - 1j * (sigma * rho * u)
    d = np.sqrt(xi * xi + s2 * q)
    xm = np.where(xi.real > 0, -s2 * q / (xi + d), xi - d)
    g, e = xm / np.where(xi.real > 0, xi + d, -s2 * q / xm), np.exp(-d * T)
    A = kappa * theta / s2 * (xm * T - 2 * np.log((1 - g * e) / (1 - g)))
    z = A + v0 / s2 * xm * (1 - e) / (1 - g * e) + 1j * u * (np.log(S / K) + r * T)
    integral = (w * (np.exp(z) / q).real).sum(1, keepdims=True)
    pi = 4 * np.arctan(L(1))
    return (S - np.sqrt(S * K) * np.exp(-r * T / 2) / pi * integral)[:, 0].astype(float)


def test_edges_match_extended_precision(gpu):
    from fd_adi_amd.pricing import heston_call
    X = np.array(ROWS, dtype=float)
    S, K, r, v0, T, kappa, theta, sigma, rho = X.T
    got = heston_call(S, K, r, v0, T, kappa, theta, sigma, rho)
    tol = (1e-9 + 100 * 2.2e-16 * (1 + kappa * theta / sigma ** 2)) * S
    err = np.abs(got - reference(X))
    print(np.c_[got, err, tol])
    assert np.all(err <= tol)


def test_bad_rows_are_nan(gpu):
    from fd_adi_amd.pricing import heston_call
    X = np.array([ROWS[2]] * 9, dtype=float)
    X[np.arange(9), np.arange(9)] = np.nan
    S, K, r, v0, T, kappa, theta, sigma, rho = X.T
    assert np.all(np.isnan(heston_call(S, K, r, v0, T, kappa, theta, sigma, rho)))

"""Spot sweeps on 8-column tiles of 16 rows, whose LDS lets one work-group of 256
threads run per CU: more tiles than CUs, up to and beyond two per work-group.

Options are also solved alone on four-column tiles, with the bound on the
rounding between the two that follows from some 10 roundings in each of 24
line solves (3e-14 of the largest value; 1e-12 of it is allowed)."""

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

RTOL = 1e-12


@pytest.mark.parametrize("scheme, theta", [("cs", 0.5), ("hv", 0.7), ("implicit", 1.0)])
@pytest.mark.parametrize("n", [1, 86, 171])  # 3 tiles an option: 3, 258 and 513
def test_tiles_beyond_the_work_groups(gpu, n, scheme, theta):
    import fd_adi_amd
    rng = np.random.default_rng(n)
    P, S, V, U = [], [], [], []
    for k in range(n):
        nS, nv = int(rng.integers(257, 513)), int(rng.integers(17, 25))
        x, y = np.arange(nS) / (nS - 1.0), np.arange(nv) / (nv - 1.0)
        S.append(400.0 * (0.3 * x + 0.7 * x ** 2))
        V.append(0.5 * (0.2 * y + 0.8 * y ** 2))
        U.append(np.maximum(S[-1][:, None] - 100.0, 0.0) + 0.0 * V[-1][None, :])
        P.append(dict(r=0.03, kappa=1.5, theta=0.06, sigma=0.25, rho=-0.5))

    def solve(pick, shape):
        hb = fd_adi_amd.HestonBatch([P[k] for k in pick], [S[k] for k in pick],
                                    [V[k] for k in pick], [0.01] * len(pick))
        hb.set_state([U[k] for k in pick])
        hb.configure(scheme, theta)
        hb.set_shape(0, *shape)
        hb.step(6)
        return hb.get_state()

    got = solve(range(n), (256, 8))
    for k in sorted({0, n // 2, n - 1}):
        want = solve([k], (0, 4))[0]
        assert np.all(np.isfinite(want))
        assert np.max(np.abs(got[k] - want)) <= RTOL * np.max(np.abs(want)), k

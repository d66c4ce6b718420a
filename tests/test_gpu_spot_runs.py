"""Spot sweeps whose work-groups take tile after tile: more tiles than the GPU
holds at once, options of different grids following one another on one
work-group, chunks shorter than their slots, grids narrower than a tile.

Each option is also solved alone on four-column tiles (one tile per
work-group, another chunking).  Both solve the same discrete system by the
same elimination in FP64; they differ in how the chunk maps are composed, a
few rounding errors per line solve, which the stable solves here do not
amplify: 4 solves a step, 6 steps, about 10 roundings of 1.1e-16 each on
values up to the grid's maximum bound the difference by 3e-14 of it.  The
bound taken is 1e-12 of it.
"""

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

RTOL = 1e-12


def _options(sizes, barrier_every=7):
    rng = np.random.default_rng(11)
    params, S, V = [], [], []
    for k, (nS, nv) in enumerate(sizes):
        K = rng.uniform(80.0, 120.0)
        x = np.arange(nS) / float(nS - 1)
        top = 2 * K if k % barrier_every == 0 else 5 * K
        S.append(top * (0.3 * x + 0.7 * x ** 2))
        V.append(0.5 * (np.arange(nv) / float(nv - 1)) ** 2)
        params.append(dict(r=rng.uniform(0.0, 0.08), kappa=rng.uniform(1.0, 2.0),
                           theta=rng.uniform(0.05, 0.12), sigma=rng.uniform(0.1, 0.3),
                           rho=rng.uniform(-0.8, 0.3), barrier=k % barrier_every == 0))
    return params, S, V


def _solve(params, S, V, scheme, theta, shape):
    from fd_adi_amd import HestonBatch
    hb = HestonBatch(params, S, V, [0.01] * len(S))
    hb.set_state([np.maximum(s[:, None] - 100.0, 0.0) + 0.0 * v[None, :] for s, v in zip(S, V)])
    hb.configure(scheme, theta)
    if shape is not None:
        hb.set_shape(0, *shape)
    hb.step(6)
    return hb.get_state()


@pytest.mark.parametrize("shape, nS", [((256, 16), (17, 256)), ((512, 16), (260, 500)),
                                       ((512, 32), (33, 250)), ((256, 8), (65, 200)),
                                       ((-1, 16), (40, 400))])
@pytest.mark.parametrize("scheme, theta", [("cs", 0.5), ("hv", 0.6), ("mcs", 0.5),
                                           ("douglas", 0.7), ("implicit", 1.0)])
def test_many_tiles_match_one_by_one(gpu, shape, nS, scheme, theta):
    rng = np.random.default_rng(3)
    lo = 32 if shape[1] == 32 else 4
    nv = [lo, lo + 1, shape[1], shape[1] + 1, 2 * shape[1] - 1, 4 * shape[1]]
    # over 1,100 tiles: every work-group of the largest grid (512) takes two or three
    n = max(6, -(-1100 * shape[1] // 35))
    sizes = [(int(rng.integers(nS[0], nS[1] + 1)), nv[k] if k < len(nv)
              else int(rng.integers(lo, 70))) for k in range(n)]
    params, S, V = _options(sizes)
    got = _solve(params, S, V, scheme, theta, shape)
    pick = list(range(8)) + [n // 2, n - 3, n - 2, n - 1]
    for k in pick:
        want = _solve([params[k]], [S[k]], [V[k]], scheme, theta, None)[0]
        assert np.all(np.isfinite(want))
        err = float(np.max(np.abs(got[k] - want)))
        assert err <= RTOL * float(np.max(np.abs(want))), (k, sizes[k], err)

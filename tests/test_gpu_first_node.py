"""A spot mesh whose first node is above zero but squares to zero: its variance
line is an ordinary one, not the S = 0 line whose operator keeps only -r/2.
Against the oracle on one-tile (four columns) and wide spot tiles, from a state
that is not zero on that line, with the tolerance that the oracle's own
reorderings give (as the other engine tests)."""

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

from oracle.engine import HestonOracle, HestonParams
from tests.parity import grid_tolerance, alternates


@pytest.mark.parametrize("first", [0.0, 1e-170, 1e-3])
@pytest.mark.parametrize("shape", [(0, 4), (256, 8), (512, 32)])
@pytest.mark.parametrize("scheme, theta", [("douglas", 0.5), ("hundsdorferverwer", 0.7),
                                           ("craigsneyd", 0.5)])
def test_first_node_matches_oracle(gpu, scheme, theta, shape, first):
    import fd_adi_amd
    x, y = np.arange(70) / 69.0, np.arange(40) / 39.0
    S, V = 400.0 * (0.3 * x + 0.7 * x ** 2), 0.5 * (0.2 * y + 0.8 * y ** 2)
    S[0] = first
    o = HestonOracle(HestonParams(strike=100, r=0.03, v0=0.06, kappa=1.5, theta=0.06, sigma=0.25,
                                  rho=-0.5), S, V)
    U = 1.0 + np.maximum(S[:, None] - 100.0, 0.0) + np.sin(5.0 * y)[None, :]
    hb = fd_adi_amd.HestonBatch([dict(r=0.03, kappa=1.5, theta=0.06, sigma=0.25, rho=-0.5)], [S],
                                [V], [0.01])
    hb.set_state([U])
    hb.configure({"hundsdorferverwer": "hv", "craigsneyd": "cs"}.get(scheme, scheme), theta)
    hb.set_shape(0, *shape)
    hb.step(3)
    solve = lambda e: getattr(e, "solve_" + scheme)(3, 0.01, U, theta=theta)
    want = solve(o)
    tol, _ = grid_tolerance(want, [solve(a) for a in alternates(o)])
    err = np.abs(hb.get_state()[0] - want)
    assert float(np.max(err)) <= tol, (float(np.max(err)), np.unravel_index(np.argmax(err), err.shape), tol)

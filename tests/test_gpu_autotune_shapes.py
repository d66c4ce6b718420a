"""The launch-shape tuner where some shapes that set_shape takes cannot run:
8-column tiles of 513 to 1,024 spot nodes exceed the LDS in every scheme's
stages but the implicit one's.  It leaves those out, keeps the state, and puts
state and shapes back if a step fails for another reason."""

import numpy as np
import numpy.testing as npt
import pytest

pytestmark = pytest.mark.gpu


def _batch(nS, nv=12):
    import fd_adi_amd
    x, y = np.arange(nS) / (nS - 1.0), np.arange(nv) / (nv - 1.0)
    S, V = 400.0 * (0.3 * x + 0.7 * x ** 2), 0.5 * (0.2 * y + 0.8 * y ** 2)
    par = dict(r=0.03, kappa=1.5, theta=0.06, sigma=0.25, rho=-0.5)
    hb = fd_adi_amd.HestonBatch([par] * 2, [S] * 2, [V] * 2, [0.01] * 2)
    U = np.maximum(S[:, None] - 100.0, 0.0) + np.sin(5.0 * y)[None, :]
    hb.set_state([U, 2.0 * U])
    return hb


@pytest.mark.parametrize("scheme", ["cs", "douglas", "implicit"])
@pytest.mark.parametrize("nS", [513, 600, 1024])
def test_autotune_leaves_out_shapes_that_cannot_run(gpu, nS, scheme):
    hb, ref = _batch(nS), _batch(nS)
    before = hb.get_packed()
    hb.configure(scheme, 0.5)
    shapes = hb.autotune(steps=1)
    npt.assert_array_equal(hb.get_packed(), before)
    assert hb.get_shape(0) == shapes[0] and hb.get_shape(1)[0] == shapes[1][0]
    ref.configure(scheme, 0.5)
    hb.step(3), ref.step(3)
    want = ref.get_packed()
    assert np.max(np.abs(hb.get_packed() - want)) <= 1e-12 * np.max(np.abs(want))


def test_autotune_puts_state_and_shapes_back(gpu, monkeypatch):
    hb = _batch(70)
    hb.configure("cs", 0.5)
    hb.set_shape(0, 256, 16)
    hb.set_shape(1, 8)
    before, calls, step = hb.get_packed(), [], hb.step_timed

    def failing(n):
        calls.append(n)
        if len(calls) == 6:
            raise RuntimeError("stopped")
        return step(n)

    monkeypatch.setattr(hb, "step_timed", failing)
    with pytest.raises(RuntimeError, match="stopped"):
        hb.autotune(steps=1)
    npt.assert_array_equal(hb.get_packed(), before)
    assert hb.get_shape(0) == (256, 16) and hb.get_shape(1)[0] == 8

"""fdadi_mlp_predict_noalloc under HIP graph capture, in the mode that refuses
allocations to the capturing thread: kernel nodes alone, and replays on new
features, with eager work in between, give the prices of a direct prediction bit
for bit (which the other tests hold to the NumPy network)."""

import ctypes

import numpy as np
import numpy.testing as npt
import pytest

pytestmark = pytest.mark.gpu

THREAD_LOCAL = 1  # hipStreamCaptureModeThreadLocal
KERNEL = 0        # hipGraphNodeTypeKernel


@pytest.mark.parametrize("n, in_place, kernels", [(1, False, 1), (700, False, 1), (4096, False, 1),
                                                  (4096, True, 2)])
def test_captured_prediction(gpu, n, in_place, kernels):
    from fd_adi_amd import _lib, surrogate as S
    from fd_adi_amd.SizedArrayPtr import SizedArrayPtr
    hip = ctypes.CDLL("libamdhip64.so.7")

    def check(status):
        assert status == 0, status

    m = S.MLP(S.BOX_LO, S.BOX_HI, 1.5, 2.0, seed=3, max_rows=256)
    s, graph, run = m.stream, ctypes.c_void_p(), ctypes.c_void_p()
    s = s if isinstance(s, ctypes.c_void_p) else ctypes.c_void_p(s)
    dP, dout = SizedArrayPtr(S.draw_params(n, 1)), SizedArrayPtr().alloc(n)
    out = dP if in_place else dout
    _lib.sync()
    check(hip.hipStreamBeginCapture(s, THREAD_LOCAL))
    try:
        _lib.call("fdadi_mlp_predict_noalloc", m._h, dP.p, n, out.p, s)
    finally:
        ended = hip.hipStreamEndCapture(s, ctypes.byref(graph))
    check(ended)
    count = ctypes.c_size_t()
    check(hip.hipGraphGetNodes(graph, None, ctypes.byref(count)))
    nodes = (ctypes.c_void_p * count.value)()
    check(hip.hipGraphGetNodes(graph, nodes, ctypes.byref(count)))
    kinds = []
    for node in nodes:
        kind = ctypes.c_int()
        check(hip.hipGraphNodeGetType(ctypes.c_void_p(node), ctypes.byref(kind)))
        kinds.append(kind.value)
    assert kinds == [KERNEL] * kernels
    check(hip.hipGraphInstantiate(ctypes.byref(run), graph, None, None, ctypes.c_size_t(0)))
    try:
        for seed in (2, 3, 4):
            P = S.draw_params(n, seed)
            want = m.predict(P)  # eager work between the replays
            dP.copy_from(SizedArrayPtr(P))
            _lib.sync()
            check(hip.hipGraphLaunch(run, s))
            check(hip.hipStreamSynchronize(s))
            npt.assert_array_equal(out.to_numpy().ravel()[:n], want)
    finally:
        check(hip.hipGraphExecDestroy(run))
        check(hip.hipGraphDestroy(graph))

"""nlm_batch_dev recorded into a caller's graph as the first call of its plan: lengths that are
not powers of two, and Chi3GNLSE at N = 8192, which run as plain launches that allocate
nothing.  Every replay, with eager calls in between, gives the same result, which agrees with
the eager one; recorded after an eager call it equals it."""
import ctypes as C

import numpy as np
import pytest

from cases import small_case
from conftest import rel_l2
from test_gpu_gnlse_buffers import gnlse

pytestmark = pytest.mark.gpu


def check(rc):
    assert rc == 0, rc


@pytest.mark.parametrize("name,N", [("Chi2PDC", 600), ("Chi3", 96), ("Chi2PDC", 30), ("Chi2SHG", 300),
                                    ("Chi3GNLSE", 8192)])
def test_first_call_under_capture(nlm, name, N):
    from multimodenonlinearoptics_amd import capi
    print("capture %s N=%d" % (name, N), flush=True)
    L, H, rows = capi.lib(), capi.hip(), 5
    m = gnlse(nlm, N, 12) if name == "Chi3GNLSE" else getattr(nlm, name)(**small_case(name, nlm, N=N, nZ=40, seed=1)[1])
    if name in ("Chi2PDC", "Chi3"):
        m.runPumpSimulation()
    h, mode = C.c_void_p(m.planHandle()), (C.c_int32 * 1)(0)
    check(H.hipDeviceSynchronize())
    r = np.random.default_rng(N)
    X = capi.DeviceArray(0.1 * (r.standard_normal((rows, N)) + 1j * r.standard_normal((rows, N))))
    Y, Z = capi.DeviceArray(shape=(rows, N)), capi.DeviceArray(shape=(rows, N))
    s = C.c_void_p()
    check(H.hipStreamCreate(C.byref(s)))
    capi.check(L.nlm_plan_set_stream(h, s))

    def call(out):
        capi.check(L.nlm_batch_dev(h, X.ptr, rows, N, 1, 0, 1, mode, out.ptr))

    def record():
        graph, ex = C.c_void_p(), C.c_void_p()
        check(H.hipStreamBeginCapture(s, C.c_int(1)))
        try:
            call(Y)
        finally:
            rc = H.hipStreamEndCapture(s, C.byref(graph))
        check(rc)
        check(H.hipGraphInstantiate(C.byref(ex), graph, None, None, C.c_size_t(0)))
        check(H.hipGraphDestroy(graph))
        return ex

    def replay(ex):
        check(H.hipGraphLaunch(ex, s))
        check(H.hipStreamSynchronize(s))
        return Y.numpy()

    first = record()
    a = replay(first)
    call(Z)
    check(H.hipStreamSynchronize(s))
    eager = Z.numpy()
    assert np.isfinite(eager).all() and rel_l2(a, eager) < 1e-10
    for _ in range(3):
        assert np.array_equal(replay(first), a)
        call(Z)
        check(H.hipStreamSynchronize(s))
        assert np.array_equal(Z.numpy(), eager)
    if N != 8192:  # whose eager calls run staged
        later = record()
        for _ in range(3):
            assert np.array_equal(replay(later), eager)
        check(H.hipGraphExecDestroy(later))
    check(H.hipGraphExecDestroy(first))
    capi.check(L.nlm_plan_set_stream(h, None))
    check(H.hipStreamDestroy(s))

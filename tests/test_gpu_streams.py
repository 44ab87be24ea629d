"""Asynchronous batches of one plan on two streams: the second call, queued while the first
runs, uses the same scratch of the plan (staged Chi3GNLSE state, step table of any-length
media) and has to wait for it.  Outputs equal those of the calls one after the other."""
import ctypes as C

import numpy as np
import pytest

from cases import small_case

pytestmark = pytest.mark.gpu


class Stream:
    def __init__(self):
        from multimodenonlinearoptics_amd import capi
        self.hip, self.ptr = capi.hip(), C.c_void_p()
        assert self.hip.hipStreamCreate(C.byref(self.ptr)) == 0

    def sync(self):
        assert self.hip.hipStreamSynchronize(self.ptr) == 0

    def __del__(self):
        self.hip.hipStreamDestroy(self.ptr)


def gnlse(nlm, N, nZ):
    return nlm.Chi3GNLSE(relativeLength=2e-4 * (nZ - 1), nlLength=1 / 9, selfSteepLength=100.0, fr=0.18, fb=0.21,
                         tau1=0.0122, tau2=0.032, tau3=0.096, beta2=-1.0, tMax=50.0 * N / 16384, tPrecision=N,
                         nZSteps=nZ)


@pytest.mark.parametrize("N,rows", [(8192, (4, 4)), (8192, (3, 9)), (16384, (2, 2)), (600, (40, 40))])
def test_stream_change_between_calls(nlm, N, rows):
    from multimodenonlinearoptics_amd import capi
    print("stream change N=%d rows=%s" % (N, rows), flush=True)
    L = capi.lib()
    m = gnlse(nlm, N, 40) if N > 600 else nlm.Chi2PDC(**small_case("Chi2PDC", nlm, N=N, nZ=60, seed=1)[1])
    if N == 600:
        m.runPumpSimulation()
    h, mode = C.c_void_p(m.planHandle()), (C.c_int32 * 1)(0)
    r = np.random.default_rng(N)
    X = [capi.DeviceArray(0.1 * (r.standard_normal((k, N)) + 1j * r.standard_normal((k, N)))) for k in rows]
    Y = [capi.DeviceArray(shape=(k, N)) for k in rows]
    streams = [Stream(), Stream()]

    def call(i, k):
        capi.check(L.nlm_plan_set_stream(h, streams[k].ptr))
        capi.check(L.nlm_batch_dev(h, X[i].ptr, rows[i], N, 1, 0, 1, mode, Y[i].ptr))

    want = []
    for i in range(2):
        call(i, 0)
        streams[0].sync()
        want.append(Y[i].numpy())
    for _ in range(4):
        for i in range(2):
            call(i, i)
        for s in streams:
            s.sync()
        for i in range(2):
            assert np.array_equal(Y[i].numpy(), want[i])
    capi.check(L.nlm_plan_set_stream(h, None))

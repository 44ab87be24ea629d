"""Asynchronous staged Chi3GNLSE batches of one plan, one after the other on its stream: each
into a buffer of its own, with another number of rows, or in the other domain.  The graph of
the z loop serves every buffer, and is not taken down while a call before still replays it.
Outputs equal those of the calls with a synchronization after each."""
import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def gnlse(nlm, N, nZ):
    return nlm.Chi3GNLSE(relativeLength=2e-4 * (nZ - 1), nlLength=1 / 9, selfSteepLength=100.0, fr=0.18, fb=0.21,
                         tau1=0.0122, tau2=0.032, tau3=0.096, beta2=-1.0, tMax=50.0 * N / 16384, tPrecision=N,
                         nZSteps=nZ)


@pytest.mark.parametrize("N,nZ", [(8192, 34), (16384, 5)])
def test_calls_in_a_row(nlm, N, nZ):
    from multimodenonlinearoptics_amd import capi
    print("calls in a row N=%d" % N, flush=True)
    L = capi.lib()
    m = gnlse(nlm, N, nZ)
    h, mode = C.c_void_p(m.planHandle()), (C.c_int32 * 1)(0)
    r = np.random.default_rng(N)
    # (rows, time domain) of each call: a new buffer, more rows, fewer, the frequency domain
    calls = [(2, 1), (2, 1), (5, 1), (2, 1), (2, 0), (2, 1)]
    X = [capi.DeviceArray(0.1 * (r.standard_normal((k, N)) + 1j * r.standard_normal((k, N)))) for k, _ in calls]

    def run(wait):
        Y = [capi.DeviceArray(shape=(k, N)) for k, _ in calls]
        for x, y, (rows, in_time) in zip(X, Y, calls):
            capi.check(L.nlm_batch_dev(h, x.ptr, rows, N, in_time, 0, 1, mode, y.ptr))
            if wait:
                capi.check(L.nlm_plan_sync(h))
        capi.check(L.nlm_plan_sync(h))
        return [y.numpy() for y in Y]

    alone = [gnlse(nlm, N, nZ).batchSignalSimulation(x.host, inTimeDomain=bool(t)) for x, (_, t) in zip(X, calls)]
    for _ in range(3):
        for wait in (True, False):
            for y, a in zip(run(wait), alone):
                assert np.array_equal(y, a)

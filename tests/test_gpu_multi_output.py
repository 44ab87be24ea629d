"""MultiBatch.output from a second thread while the batch is launched again: results that are
read once a launch has been waited for are that launch's, not a copy of the ones before."""
import ctypes as C
import threading

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def test_output_of_the_last_launch(nlm):
    from multimodenonlinearoptics_amd import capi
    N = 64
    # Chi3's pump rows come from the medium's grid: its peak power decides the result
    m = nlm.Chi3(relativeLength=1.0, nlLength=1.0, beta2=-1.0, tMax=10, tPrecision=N, nZSteps=20)
    tau = np.asarray(m.tau)
    pumps = [a / np.cosh(tau) + 0j for a in (0.5, 1.0)]
    b = nlm.MultiBatch([m], [np.exp(-tau ** 2) + 0j], inTimeDomain=True, autotune=False)

    def launch(k):
        m.setPump(pumps[k])
        m.runPumpSimulation()
        capi.check(capi.lib().nlm_plan_sync(C.c_void_p(m.planHandle())))
        b.launch()
        b.sync()
        return b.output(0)

    want = [launch(0), launch(1)]
    assert not np.array_equal(want[0], want[1])
    done = threading.Event()

    def read():
        while not done.is_set():
            b.output(0)

    readers = [threading.Thread(target=read) for _ in range(3)]
    for t in readers:
        t.start()
    try:
        for i in range(100):
            assert np.array_equal(launch(i % 2), want[i % 2]), i
    finally:
        done.set()
        for t in readers:
            t.join()

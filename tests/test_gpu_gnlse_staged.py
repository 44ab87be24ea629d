"""The staged Chi3GNLSE kernels (nlm_big.hip) over their splits N = P x M and row groups:
every P of 1..16, rows below, at and beyond a multiple of eight (fields are placed eight at
a time), one step, a segment of one step, and a Raman response that is not the spectrum of a
real one, whose convolution takes complex exchanges.  Batches of N = 8192, which run staged,
against the oracle.  Tolerance: the engine's relative L2 of 1e-10."""
import ctypes as C

import numpy as np
import pytest

import gnlse_torch as GT
from conftest import rel_l2
from test_gnlse_torch_reference import sech_inputs, small_kwargs

pytestmark = pytest.mark.gpu
TOL = 1e-10


def case(oracle, N, nZ, rows, in_time):
    kw = small_kwargs(N, nZ, 0.001 * nZ if N <= 2048 else 0.0004 * nZ)
    kw["tMax"] = 10.0 if N <= 2048 else 40.0
    X = sech_inputs(N, rows, N + nZ, kw["tMax"])
    ref = oracle.Chi3GNLSE(**kw)
    return kw, X if in_time else np.fft.fft(X, axis=1), GT.GnlseTables(kw, ref.omega, ref.ramanResponse)


@pytest.mark.parametrize("N,nZ,rows,in_time,ckpt", [
    (32, 6, 8, True, 2), (512, 5, 9, False, 1), (1024, 8, 17, True, 3), (2048, 2, 5, True, 0), (4096, 5, 9, False, 4),
    (8192, 4, 10, True, 1), (16384, 3, 9, True, 2), (32768, 3, 2, True, 1)])
def test_splits(nlm, oracle, N, nZ, rows, in_time, ckpt):
    print("staged N=%d nZ=%d rows=%d" % (N, nZ, rows), flush=True)
    kw, X, t = case(oracle, N, nZ, rows, in_time)
    w, c = GT.loss_weights(rows, N, N + 1)
    Yref, gref = GT.reference_gradient(X, t, in_time, w, c)
    dev = nlm.Chi3GNLSE(**kw)
    Y = dev.batchForward(X, inTimeDomain=in_time, ckptEvery=ckpt)
    assert rel_l2(Y, Yref) < TOL
    assert rel_l2(dev.batchAdjoint(GT.grad_out(Y, w, c)), gref) < TOL


@pytest.mark.parametrize("rows,nZ,in_time", [(1, 4, True), (9, 35, False), (8, 2, True), (256, 2, True), (257, 2, True)])
def test_batch_8192(nlm, oracle, rows, nZ, in_time):
    print("batch N=8192 rows=%d nZ=%d" % (rows, nZ), flush=True)
    kw, X, _ = case(oracle, 8192, nZ, rows, in_time)
    got = nlm.Chi3GNLSE(**kw).batchSignalSimulation(X, inTimeDomain=in_time)
    ref = oracle.Chi3GNLSE(**kw).batchSignalSimulation(X, inTimeDomain=in_time, nThreads=min(rows, 8))
    assert rel_l2(got, ref) < TOL


@pytest.mark.parametrize("N,rows,in_time", [(64, 3, True), (1024, 9, False), (4096, 2, True)])
def test_complex_response(nlm, oracle, N, rows, in_time):
    """A plan made directly, with a response whose spectrum is not Hermitian."""
    import torch
    from multimodenonlinearoptics_amd import capi
    print("complex response N=%d" % N, flush=True)
    nZ = 6
    kw, X, t = case(oracle, N, nZ, rows, in_time)
    t.raman = t.raman * torch.exp(0.3j * torch.linspace(-1, 1, N, dtype=torch.float64))
    w, c = GT.loss_weights(rows, N, N + 1)
    Yref, gref = GT.reference_gradient(X, t, in_time, w, c)
    L = capi.lib()
    L.nlm_batch_forward.argtypes = [C.c_void_p, C.c_void_p, C.c_int, C.c_int, C.c_int, C.c_void_p]
    L.nlm_batch_adjoint.argtypes = [C.c_void_p, C.c_void_p, C.c_void_p]
    host = [np.ascontiguousarray(x.numpy(), dtype=np.complex128)
            for x in (t.disp, t.half_in, t.half_out, t.raman, t.filt)]
    coef, const = np.ones((nZ, 3), np.complex128), np.zeros(1, np.complex128)
    ptr = lambda a: a.ctypes.data  # noqa: E731
    desc = capi.PlanDesc(14, N, nZ, ptr(host[0]), ptr(host[1]), ptr(host[2]), ptr(coef), ptr(const), ptr(host[3]),
                         ptr(host[4]))
    plan = C.c_void_p()
    capi.check(L.nlm_plan_create(C.byref(desc), C.byref(plan)))
    try:
        x, Y, g = np.ascontiguousarray(X), np.empty((rows, N), np.complex128), np.empty((rows, N), np.complex128)
        capi.check(L.nlm_batch_forward(plan, ptr(x), rows, int(in_time), 2, ptr(Y)))
        assert rel_l2(Y, Yref) < TOL
        go = np.ascontiguousarray(GT.grad_out(Y, w, c))
        capi.check(L.nlm_batch_adjoint(plan, ptr(go), ptr(g)))
        assert rel_l2(g, gref) < TOL
    finally:
        L.nlm_plan_destroy(plan)

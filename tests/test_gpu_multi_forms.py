"""The forms that a heterogeneous batch's classes take with less memory than everything staged
would need, which stageLimit sets: pump rows generated in the kernel ("inline"), one-mode media
fed from their pump grids ("field"), and a limit that holds only the largest class.  Every
instance against the oracle at the engine's rel. L2 of 1e-10."""
import ctypes as C

import numpy as np
import pytest

from cases import ALL, make, random_inputs, small_case
from conftest import rel_l2

pytestmark = pytest.mark.gpu
TOL = 1e-10
# single linear pump: one mode takes a step table, several the staged rows
LINEAR = ("Chi2PDC", "Chi2SFG", "Chi2AFC", "Chi2SFGPDC", "Chi2SFGII", "Chi2PDCII", "Chi2SFGXPM")


def batch(nlm, oracle, cases, **kw):
    """(batch, run) over cases of (solver, N, nZ), checked against the oracle."""
    media, ref, xs = [], [], []
    for j, (name, N, nZ) in enumerate(cases):
        media.append(make(nlm, name, small_case(name, nlm, N=N, nZ=nZ, seed=100 + j, poled=nZ > 16)[1]))
        ref.append(make(oracle, name, small_case(name, oracle, N=N, nZ=nZ, seed=100 + j, poled=nZ > 16)[1]))
        xs.append(random_inputs(name, N, 1, seed=200 + j)[0])
    b = nlm.MultiBatch(media, xs, inTimeDomain=True, autotune=False, **kw)
    b.run()
    for i, (r, x, c) in enumerate(zip(ref, xs, cases)):
        err = rel_l2(b.output(i), r.batchSignalSimulation(x[None, :], inTimeDomain=True)[0])
        print("instance", c, "%.1e" % err, flush=True)
        assert err < TOL, (c, err)
    return b


def forms(b):
    """{(class model id, N): form}"""
    return {(c[0], 1 << c[1]): f for c, f in zip(b.classes(), b.forms())}


@pytest.mark.parametrize("limit", [-1, 0])
def test_large_pdc_class(nlm, oracle, limit):
    """Chi2PDC at N = 4096 over chunks of 16 steps (the last one partial) or, generated in the
    kernel, over the exact phase every 64 rows."""
    b = batch(nlm, oracle, [("Chi2PDC", 4096, nZ) for nZ in (3, 70, 150)] + [("Chi2SHG", 4096, 20)], stageLimit=limit)
    f = forms(b)
    assert f[(1, 4096)] == (("table", 2 * (3 + 70 + 150) * 4096 * 16) if limit else ("inline", 0))
    assert f[(9, 4096)] == ("modes", 0)


@pytest.mark.parametrize("limit", [-1, 0])
def test_every_solver(nlm, oracle, limit):
    b = batch(nlm, oracle, [(name, N, nZ) for name in ALL for N, nZ in ((32, 21), (128, 37))], stageLimit=limit)
    assert sum(s for _, s in b.forms()) > 0 if limit else all(s == 0 for _, s in b.forms())
    f = forms(b)
    for N in (32, 128):
        assert f[(0, N)][0] == ("table" if limit else "field")   # Chi3, from its pump grid
        assert f[(1, N)][0] == ("table" if limit else "inline")  # Chi2PDC
        for model in (2, 4, 5, 6, 8):                            # multi-mode media with a linear pump
            assert f[(model, N)][0] == ("modes" if limit else "inline")


@pytest.mark.parametrize("N,nZ", [(512, 20), (2048, 8), (4096, 6)])
def test_generated_rows_of_larger_media(nlm, oracle, N, nZ):
    b = batch(nlm, oracle, [(name, N, nZ) for name in LINEAR], stageLimit=0)
    assert all(f == ("inline", 0) for f in b.forms())


def test_limit_holds_the_largest_class(nlm, oracle):
    cases = [("Chi2PDC", 1024, 10), ("Chi2PDC", 256, 40)]
    need = 2 * 10 * 1024 * 16
    f = forms(batch(nlm, oracle, cases, stageLimit=need))
    assert f == {(1, 1024): ("table", need), (1, 256): ("inline", 0)}
    f = forms(batch(nlm, oracle, cases, stageLimit=need - 1))
    assert f[(1, 1024)] == ("inline", 0)


def test_staging_that_cannot_be_had(nlm):
    """More than the card has: the largest class falls back to generated rows, the small one is
    staged within what is left, and the results are those of that choice made at once."""
    N, nZ = 4096, 20000
    small = dict(relativeLength=1.0, nlLength=1.0, beta2=0.1, beta2s=-0.2, tMax=20, tPrecision=256, nZSteps=50)
    big = dict(small, tPrecision=N, nZSteps=nZ)
    count = 400 * 10 ** 9 // (2 * nZ * N * 16)
    media = [nlm.Chi2PDC(**big) for _ in range(count)] + [nlm.Chi2PDC(**small)]
    r = np.random.default_rng(0)
    xs = [r.standard_normal(m.omega.size) + 0j for m in media]
    got = []
    for limit in (1 << 60, 1 << 30):
        b = nlm.MultiBatch(media, xs, inTimeDomain=True, autotune=False, stageLimit=limit)
        assert forms(b) == {(1, N): ("inline", 0), (1, 256): ("table", 2 * 50 * 256 * 16)}
        print("created, limit", limit, "ms", b.run(), flush=True)
        got.append([b.output(i) for i in (0, count - 1, count)])
    for a, c in zip(*got):
        assert np.isfinite(a).all() and np.array_equal(a, c)


class Item(C.Structure):
    _fields_ = [("plan", C.c_void_p), ("input", C.c_void_p), ("cols", C.c_int32), ("in_time", C.c_int32),
                ("input_mode", C.c_int32), ("n_out", C.c_int32), ("outputs", C.c_int32 * 4), ("envelope", C.c_void_p),
                ("disp_pump", C.c_void_p), ("dzp", C.c_double), ("strength", C.c_void_p)]


@pytest.mark.parametrize("limit,form", [(-1, 3), (0, 0)])
def test_pump_grids_of_pdc_media(nlm, limit, form):
    """Chi2PDC media without an envelope, through the C interface: step tables made of their pump
    grids, or the grids read in the kernel; lengths of 1 step, one chunk and a partial one."""
    from multimodenonlinearoptics_amd import capi
    L = capi.lib()
    L.nlm_multi_create_staged.argtypes = [C.c_int, C.c_void_p, C.c_int, C.c_int64, C.c_void_p]
    L.nlm_multi_output.argtypes = [C.c_void_p, C.c_int, C.c_void_p]
    media, xs, items = [], [], []
    for j, (N, nZ) in enumerate([(32, 2), (64, 17), (64, 40), (1024, 19), (4096, 5)]):
        m = nlm.Chi2PDC(**small_case("Chi2PDC", nlm, N=N, nZ=nZ, seed=j, poled=False)[1])
        m.runPumpSimulation()
        media.append(m)
        xs.append(random_inputs("Chi2PDC", N, 1, seed=j)[0])
        it = Item(m.planHandle(), xs[-1].ctypes.data, N, 1, 0, 1)
        items.append(it)
        capi.check(L.nlm_plan_sync(C.c_void_p(m.planHandle())))
    arr, b = (Item * len(items))(*items), C.c_void_p()
    capi.check(L.nlm_multi_create_staged(len(items), arr, 0, limit, C.byref(b)))
    try:
        for c in range(L.nlm_multi_classes(b)):
            f = C.c_int32()
            capi.check(L.nlm_multi_form(b, c, C.byref(f), None))
            assert f.value == form
        capi.check(L.nlm_multi_launch(b))
        capi.check(L.nlm_multi_sync(b, None))
        for i, (m, x) in enumerate(zip(media, xs)):
            out = np.empty(x.size, np.complex128)
            capi.check(L.nlm_multi_output(b, i, out.ctypes.data))
            assert rel_l2(out, m.batchSignalSimulation(x[None, :], inTimeDomain=True)[0]) < 1e-12, i
    finally:
        L.nlm_multi_destroy(b)

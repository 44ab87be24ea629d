"""The step-table kernel with eight points per lane below N = 256, which runs once the fields
fill more than 256 of its waves (fewer take four points per lane): 4 to 64 fields in a wave,
the last wave with one.  Against the oracle at the engine's rel. L2 of 1e-10, and against the
same rows in a batch of four points per lane."""
import numpy as np
import pytest

from cases import make, random_inputs, small_case
from conftest import rel_l2

pytestmark = pytest.mark.gpu
TOL = 1e-10


@pytest.mark.parametrize("name,N,rows", [("Chi2PDC", 8, 16385), ("Chi3", 16, 8193), ("Chi2PDC", 32, 4097),
                                         ("Chi3", 64, 2049), ("Chi2PDC", 128, 1025)])
def test_just_past_the_four_point_form(nlm, oracle, name, N, rows):
    print("eight points %s N=%d rows=%d" % (name, N, rows), flush=True)
    nZ = 5
    dev, ref = (make(mod, name, small_case(name, mod, N=N, nZ=nZ, seed=5, poled=False)[1]) for mod in (nlm, oracle))
    X = random_inputs(name, N, rows, seed=N, nch=1)
    for in_time in (True, False):
        got = dev.batchSignalSimulation(X, inTimeDomain=in_time, runPump=True)
        few = dev.batchSignalSimulation(X[-9:], inTimeDomain=in_time, runPump=True)
        assert rel_l2(got[-9:], few) < 1e-13
        pick = np.unique(np.r_[0:70, rows // 2, rows - 70:rows])
        want = ref.batchSignalSimulation(X[pick], inTimeDomain=in_time, runPump=True)
        for k, i in enumerate(pick):
            assert rel_l2(got[i], want[k]) < TOL, i


@pytest.mark.parametrize("name,N,rows", [("Chi2PDC", 32, 4097), ("Chi3", 128, 1025)])
def test_grids(nlm, name, N, rows):
    """z-resolved grids of the same rows in both forms."""
    m = make(nlm, name, small_case(name, nlm, N=N, nZ=4, seed=6, poled=False)[1])
    X = random_inputs(name, N, rows, seed=N, nch=1)
    m.runPumpSimulation()
    many, few = m.batchSignalGrids(X, inTimeDomain=True), m.batchSignalGrids(X[-5:], inTimeDomain=True)
    for a, b in zip(many, few):
        a, b = np.asarray(a).reshape(rows, -1)[-5:], np.asarray(b).reshape(5, -1)
        assert np.isfinite(a).all() and rel_l2(a, b) < 1e-13

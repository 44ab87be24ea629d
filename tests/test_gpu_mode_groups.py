"""The multi-mode split step with one lane group per mode (nlm_modes.hpp) against the
oracle at the engine's rel. L2 1e-10: several fields per wave, groups of less than a
wave with spare lanes (three modes), groups of several waves, more than 512 lanes
(128 registers, compact twiddle tables), and the sizes just beyond, which keep all
modes in the same lanes."""
import numpy as np
import pytest

from cases import DEPLETED, NMODES, make, random_inputs, small_case
from conftest import rel_l2

pytestmark = pytest.mark.gpu
TOL = 1e-10


def both(nlm, oracle, name, N, nZ):
    return [make(mod, name, small_case(name, mod, N=N, nZ=nZ, seed=7, poled=nZ > 20)[1]) for mod in (nlm, oracle)]


@pytest.mark.parametrize("name,N", [
    ("Chi2SHG", 8), ("Chi2SHG", 32), ("Chi2SHG", 512), ("Chi2SHG", 2048), ("Chi2SHG", 4096), ("Chi2SHG", 8192),
    ("Chi2DSFG", 8), ("Chi2DSFG", 64), ("Chi2DSFG", 256), ("Chi2DSFG", 1024), ("Chi2DSFG", 2048), ("Chi2DSFG", 4096),
    ("Chi2SFGII", 16), ("Chi2SFGII", 128), ("Chi2SFGII", 1024), ("Chi2SFGII", 2048), ("Chi2SHGOPA", 256),
    ("Chi2SFGOPA", 64), ("Chi2SFGOPA", 4096), ("Chi2PDCII", 1024), ("Chi2PDCII", 4096)])
def test_batch(nlm, oracle, name, N):
    rows, nZ = 5, 40 if N <= 512 else 8
    print("batch %s N=%d" % (name, N), flush=True)
    dev, ref = both(nlm, oracle, name, N, nZ)
    extra = {} if name in DEPLETED else {"runPump": True}
    for in_time, nch in ((True, 1), (False, NMODES[name])):
        X = random_inputs(name, N, rows, seed=N, nch=nch)
        got = dev.batchSignalSimulation(X, inTimeDomain=in_time, **extra)
        assert rel_l2(got, ref.batchSignalSimulation(X, inTimeDomain=in_time, **extra)) < TOL


@pytest.mark.parametrize("name,N", [("Chi2SHG", 64), ("Chi2DSFG", 512), ("Chi2SFGII", 32), ("Chi2PDCII", 4096)])
def test_grids(nlm, oracle, name, N):
    print("grids %s N=%d" % (name, N), flush=True)
    dev, ref = both(nlm, oracle, name, N, 30 if N <= 512 else 6)
    X = random_inputs(name, N, 1, seed=N, nch=1)[0]
    for m in (dev, ref):
        if name not in DEPLETED:
            m.runPumpSimulation()
        m.runSignalSimulation(X)
    for q in range(NMODES[name]):
        assert rel_l2(dev.signalTimes(q), ref.signalTimes(q)) < TOL
        assert rel_l2(dev.signalFreqs(q), ref.signalFreqs(q)) < TOL


@pytest.mark.parametrize("name,N", [("Chi2PDCII", 16), ("Chi2SFGII", 64), ("Chi2SFGPDC", 256)])
def test_greens(nlm, oracle, name, N):
    print("greens %s N=%d" % (name, N), flush=True)
    dev, ref = both(nlm, oracle, name, N, 25)
    got, exp = dev.computeGreensFunction(), ref.computeGreensFunction()
    assert rel_l2(np.hstack(got), np.hstack(exp)) < TOL

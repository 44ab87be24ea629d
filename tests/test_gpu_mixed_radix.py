"""The in-register mixed-radix kernels (nlm_mix.hpp) at the edges of their plans,
against the oracle at the engine's rel. L2 1e-10: every first radix, several fields per
wave with a last workgroup that is not full, one to four signal modes, one wave and
several per field, 0 to 3 middle stages, LDS beyond 64 KB, and the lengths just
outside (no square factor, a prime factor above 7) that the general kernel runs."""
import numpy as np
import pytest

from cases import DEPLETED, make, random_inputs, small_case
from conftest import rel_l2

pytestmark = pytest.mark.gpu
TOL = 1e-10


def both(nlm, oracle, name, N, nZ, poled=True):
    out = []
    for mod in (nlm, oracle):
        _, kw = small_case(name, mod, N=N, nZ=nZ, seed=N, poled=poled)
        out.append(make(mod, name, kw))
    return out


@pytest.mark.parametrize("name,N", [
    ("Chi2PDC", 12), ("Chi2PDC", 18), ("Chi3", 48), ("Chi2PDC", 100), ("Chi2PDC", 150), ("Chi3", 384),
    ("Chi2PDC", 486), ("Chi2PDC", 588), ("Chi2PDC", 648), ("Chi2PDC", 1350), ("Chi2PDC", 2400), ("Chi3", 4000),
    ("Chi2PDC", 98), ("Chi2PDC", 210), ("Chi2PDCII", 48), ("Chi2PDCII", 150), ("Chi2SHG", 300), ("Chi2SHG", 1500),
    ("Chi2SFG", 486), ("Chi2SFGOPA", 100), ("Chi2SFGXPM", 90), ("Chi2SFGPDC", 250), ("Chi2AFC", 72),
    ("Chi2DSFG", 60), ("Chi2DSFG", 250), ("Chi2SFGII", 36), ("Chi2SFGII", 200), ("Chi2SHGOPA", 150),
    ("Chi2SHGOPA", 400), ("Chi3GNLSE", 48), ("Chi3GNLSE", 150), ("Chi3GNLSE", 384), ("Chi3GNLSE", 1500)])
def test_batch(nlm, oracle, name, N):
    rows, nZ = 7, 30
    print("batch %s N=%d" % (name, N), flush=True)
    dev, ref = both(nlm, oracle, name, N, nZ)
    X = random_inputs(name, N, rows, seed=N, nch=1)
    extra = {} if name in DEPLETED else {"runPump": True}
    for in_time in (True, False):
        got = dev.batchSignalSimulation(X, inTimeDomain=in_time, **extra)
        assert rel_l2(got, ref.batchSignalSimulation(X, inTimeDomain=in_time, **extra)) < TOL


@pytest.mark.parametrize("name,N", [("Chi3", 60), ("Chi2PDCII", 100), ("Chi2SHG", 144), ("Chi2DSFG", 500)])
def test_grids(nlm, oracle, name, N):
    print("grids %s N=%d" % (name, N), flush=True)
    dev, ref = both(nlm, oracle, name, N, 30)
    X = random_inputs(name, N, 1, seed=N, nch=1)[0]
    for m in (dev, ref):
        if name not in DEPLETED:
            m.runPumpSimulation()
        m.runSignalSimulation(X)
    if name not in DEPLETED:
        assert rel_l2(dev.pumpTime, ref.pumpTime) < TOL and rel_l2(dev.pumpFreq, ref.pumpFreq) < TOL
    modes = {"Chi3": 1, "Chi2DSFG": 3}.get(name, 2)
    for q in range(modes):
        assert rel_l2(dev.signalTimes(q), ref.signalTimes(q)) < TOL
        assert rel_l2(dev.signalFreqs(q), ref.signalFreqs(q)) < TOL


@pytest.mark.parametrize("name,N", [("Chi2PDC", 20), ("Chi2PDC", 300), ("Chi2PDCII", 90), ("Chi2SFGII", 60)])
def test_greens_and_the_general_kernel(nlm, oracle, name, N):
    print("greens %s N=%d" % (name, N), flush=True)
    dev, ref = both(nlm, oracle, name, N, 30)
    C, S = dev.computeGreensFunction()
    Co, So = ref.computeGreensFunction()
    both_of = lambda a, b: np.hstack([a, b])  # noqa: E731
    assert rel_l2(both_of(C, S), both_of(Co, So)) < TOL
    if name == "Chi2PDC":
        dev.setStepTable(False)  # the per-field DiffEq: the general kernel
        assert rel_l2(both_of(*dev.computeGreensFunction()), both_of(C, S)) < TOL


def test_one_and_two_steps(nlm, oracle):
    for nZ in (2, 3):
        dev, ref = both(nlm, oracle, "Chi2SHG", 60, nZ, poled=False)
        X = random_inputs("Chi2SHG", 60, 3, seed=nZ, nch=1)
        assert rel_l2(dev.batchSignalSimulation(X), ref.batchSignalSimulation(X)) < TOL

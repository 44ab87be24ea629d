"""The step-table propagation with four points per lane (nlm_quad.hpp), taken by launches of
few fields up to N = 256, against the oracle at the engine's rel. L2 1e-10: both parities of
log2 N, fields that fill a wave and leave part of it empty, and the shortest media, whose
rows are fetched two steps ahead; beyond 256 waves of the other form that one runs."""
import numpy as np
import pytest

from cases import make, random_inputs, small_case
from conftest import rel_l2

pytestmark = pytest.mark.gpu
TOL = 1e-10


def both(nlm, oracle, name, N, nZ):
    return [make(mod, name, small_case(name, mod, N=N, nZ=nZ, seed=5, poled=nZ > 20)[1]) for mod in (nlm, oracle)]


@pytest.mark.parametrize("name,N,rows,nZ", [
    ("Chi2PDC", 8, 33, 30), ("Chi2PDC", 16, 1, 2), ("Chi3", 16, 17, 3), ("Chi2PDC", 32, 9, 4), ("Chi2PDC", 64, 5, 25),
    ("Chi3", 64, 4, 2), ("Chi2PDC", 128, 3, 30), ("Chi3", 128, 2, 5), ("Chi2PDC", 256, 1, 3), ("Chi2PDC", 256, 7, 40),
    ("Chi2PDC", 256, 512, 3), ("Chi2PDC", 256, 513, 3)])
def test_batch(nlm, oracle, name, N, rows, nZ):
    print("batch %s N=%d rows=%d nZ=%d" % (name, N, rows, nZ), flush=True)
    dev, ref = both(nlm, oracle, name, N, nZ)
    X = random_inputs(name, N, rows, seed=N, nch=1)
    for in_time in (True, False):
        got = dev.batchSignalSimulation(X, inTimeDomain=in_time, runPump=True)
        assert rel_l2(got, ref.batchSignalSimulation(X, inTimeDomain=in_time, runPump=True)) < TOL


@pytest.mark.parametrize("name,N,nZ", [("Chi2PDC", 8, 25), ("Chi3", 32, 2), ("Chi2PDC", 64, 3), ("Chi3", 128, 30),
                                       ("Chi2PDC", 256, 24)])
def test_grids_and_greens(nlm, oracle, name, N, nZ):
    print("grids %s N=%d nZ=%d" % (name, N, nZ), flush=True)
    dev, ref = both(nlm, oracle, name, N, nZ)
    x = random_inputs(name, N, 1, seed=N, nch=1)[0]
    for m in (dev, ref):
        m.runPumpSimulation()
        m.runSignalSimulation(x)
    assert rel_l2(dev.signalTimes(0), ref.signalTimes(0)) < TOL
    assert rel_l2(dev.signalFreqs(0), ref.signalFreqs(0)) < TOL
    assert rel_l2(np.hstack(dev.computeGreensFunction()), np.hstack(ref.computeGreensFunction())) < TOL


@pytest.mark.parametrize("N,nZ,ckpt", [(32, 9, 3), (128, 20, 4), (256, 7, 1)])
def test_checkpoints(nlm, N, nZ, ckpt):
    """The adjoint rebuilds its states from the forward's checkpoints: directional derivative of
    the device's own Green's function, central differences at 1e-6 (second order, error ~1e-9)."""
    import torch
    from multimodenonlinearoptics_amd.autograd import GreensFunction
    m = make(nlm, "Chi2PDC", small_case("Chi2PDC", nlm, N=N, nZ=nZ, seed=5, poled=False)[1])
    r = np.random.default_rng(N)
    w = r.standard_normal((N, N)) + 1j * r.standard_normal((N, N))
    env = 0.3 * (r.standard_normal(N) + 1j * r.standard_normal(N))
    pol = np.array(r.uniform(0.5, 1.0, nZ))

    def loss(e, g=False):
        te = torch.tensor(e, requires_grad=g)
        C, S = GreensFunction.apply(m, te, torch.tensor(pol))
        v = (torch.as_tensor(w).to(S.device) * S).real.sum()
        return (v, te) if g else float(v)

    v, te = loss(env, True)
    v.backward()
    d = r.standard_normal(N) + 1j * r.standard_normal(N)
    d /= np.linalg.norm(d)
    h = 1e-6
    fd = (loss(env + h * d) - loss(env - h * d)) / (2 * h)
    an = float(np.real(np.vdot(te.grad.numpy(), d)))
    assert abs(fd - an) <= 1e-6 * np.linalg.norm(te.grad.numpy())

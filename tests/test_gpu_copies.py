"""Copies between the device and host memory (nlm_copy.hip): results of less than one
1 MB piece, of several and of a ragged last one, from several threads at once; and
the autograd functions on device tensors against the same on host tensors."""
import os
import subprocess
import sys
import threading

import numpy as np
import pytest

from cases import small_case

pytestmark = pytest.mark.gpu
ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.mark.parametrize("rows", [1, 32, 33, 383, 384, 1151])
def test_batch_results_of_every_size(nlm, rows):
    """N = 512: 8 KB a row; up to 32 rows are gathered, from 384 the copy goes in pieces."""
    N = 512
    m = nlm.Chi2PDC(**small_case("Chi2PDC", nlm, N=N, nZ=30, seed=1)[1])
    r = np.random.default_rng(rows)
    X = r.standard_normal((rows, N)) + 1j * r.standard_normal((rows, N))
    Y = m.batchSignalSimulation(X, inTimeDomain=True)
    for i in {0, rows // 2, rows - 1}:
        assert np.array_equal(Y[i], m.batchSignalSimulation(X[i:i + 1], inTimeDomain=True)[0])


def test_concurrent_callers(nlm):
    """Each thread's medium gives what it gives alone (Green's matrices of 4 MB)."""
    media = [nlm.Chi2PDC(**small_case("Chi2PDC", nlm, N=512, nZ=20 + k, seed=k, poled=False)[1]) for k in range(4)]
    alone = [m.computeGreensFunction() for m in media]
    got = [[] for _ in media]

    def work(k):
        for _ in range(3):
            got[k].append(media[k].computeGreensFunction())

    threads = [threading.Thread(target=work, args=(k,)) for k in range(len(media))]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    for k, (C, S) in enumerate(alone):
        assert len(got[k]) == 3
        for Ck, Sk in got[k]:
            assert np.array_equal(C, Ck) and np.array_equal(S, Sk)


SCRIPT = """
import sys
sys.path[:0] = [%(root)r, %(root)r + "/tests"]
import numpy as np, torch
import multimodenonlinearoptics_amd as pkg
from multimodenonlinearoptics_amd.autograd import BatchSignal, GreensFunction
torch.zeros(1, device="cuda")
nlm = pkg.nonlinearmedium
r = np.random.default_rng(0)
N, nZ = 128, 25
m = nlm.Chi2PDC(relativeLength=1, nlLength=1, beta2=0.3, beta2s=-0.2, beta1=0.5, tMax=20, tPrecision=N, nZSteps=nZ)
env = np.exp(-np.asarray(m.tau) ** 2 / 2).astype(complex)
pol = r.uniform(-1, 1, nZ)
w = torch.tensor(r.standard_normal((2, N, N)) + 1j * r.standard_normal((2, N, N)))
probe = torch.zeros(4, dtype=torch.complex128, device="cuda")
print("direct", m.onDevice([probe.data_ptr()]), m.onDevice([pol.ctypes.data]))
def greens(dev, form):
    e, p = torch.tensor(env, device=dev, requires_grad=True), torch.tensor(pol, device=dev, requires_grad=True)
    C, S = GreensFunction.apply(m, e, p)
    a, b = w[0].to(dev), w[1].to(dev)
    # a gradient that is a lazy conjugate, a transpose, an expanded scalar, or none at all
    L = {"plain": lambda: (C * a).real.sum() + (S * b).real.sum(), "conj": lambda: (C.conj() * a).real.sum(),
         "transposed": lambda: (S.transpose(0, 1) @ a).real.sum(), "expanded": lambda: S.real.sum()}[form]()
    return [t.detach().cpu().numpy() for t in (C, S, *torch.autograd.grad(L, (e, p)))]
for form in ("plain", "conj", "transposed", "expanded"):
    for x, y in zip(greens("cuda", form), greens("cpu", form)):
        assert np.allclose(x, y, rtol=0, atol=1e-12 * np.abs(y).max()), form
g = nlm.Chi3GNLSE(relativeLength=0.02, nlLength=1 / 9, selfSteepLength=100, fr=0.18, fb=0.21, tau1=0.0122,
                  tau2=0.032, tau3=0.096, beta2=-1, tMax=5, tPrecision=512, nZSteps=15)
x0 = r.standard_normal((3, 512)) + 1j * r.standard_normal((3, 512))
def batch(dev, lazy):
    x = torch.tensor(x0, device=dev, requires_grad=True)
    y = BatchSignal.apply(g, x.conj() if lazy else x, True)
    return [t.detach().resolve_conj().cpu().numpy() for t in (y, *torch.autograd.grad((y.abs() ** 2).sum(), x))]
for lazy in (False, True):
    for x, y in zip(batch("cuda", lazy), batch("cpu", lazy)):
        assert np.allclose(x, y, rtol=0, atol=1e-12 * np.abs(y).max()), lazy
print("device tensors agree with host tensors")
"""


def test_device_tensors_agree_with_host_tensors():
    """In a process of its own, where torch is loaded first and both share one HIP runtime."""
    p = subprocess.run([sys.executable, "-c", SCRIPT % {"root": ROOT}], stdout=subprocess.PIPE, stderr=subprocess.STDOUT,
                       text=True, timeout=110)
    print(p.stdout)
    assert p.returncode == 0, p.stdout[-2000:]
    assert "direct True False" in p.stdout and "agree" in p.stdout

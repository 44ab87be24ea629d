"""The self-phase modulated pump on both sides of the phase pi/4 per row, where its sine and
cosine change from the short polynomials to the library's: waves that are below it, above
it, and split between their lanes' points; one wave and several, and the mixed-radix rows.
Seven rows only, as phases above 1 amplify a rounding error by about 1 + 2 phase per row:
5^6 x 1e-15 stays below the tolerance."""
import numpy as np
import pytest

from conftest import rel_l2

pytestmark = pytest.mark.gpu
TOL = 1e-10


@pytest.mark.parametrize("N", [8, 16, 32, 64, 128, 256, 512, 1024, 4096, 90, 600])
@pytest.mark.parametrize("phase", [0.05, 0.785, 2.0])
def test_pump_rows(nlm, oracle, N, phase):
    print("pump N=%d phase=%g" % (N, phase), flush=True)
    ms = []
    for mod in (nlm, oracle):  # six steps of 1/6 over the unit peak intensity
        m = mod.Chi3(relativeLength=1.0, nlLength=1.0 / (6 * phase), beta2=-0.8, beta3=0.1,
                     pulseType=mod.PulseType.Sech, tPrecision=N, tMax=8.0, nZSteps=4)
        m.runPumpSimulation()
        ms.append(m)
    dev, ref = ms
    assert rel_l2(np.asarray(dev.pumpTime), np.asarray(ref.pumpTime)) < TOL
    assert rel_l2(np.asarray(dev.pumpFreq), np.asarray(ref.pumpFreq)) < TOL

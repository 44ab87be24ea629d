"""nlm_greens_noalloc at lengths that are not powers of two: the same bits as nlm_greens where
the step table fits its scratch array, and agreement at rel. L2 1e-10 where it does not."""
import numpy as np
import pytest

from cases import small_case
from conftest import rel_l2
from test_zz_no_alloc import _both

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("name,N,nZ,modes", [("Chi2PDC", 600, 40, 1), ("Chi3", 96, 25, 1), ("Chi2PDC", 30, 20, 1),
                                             ("Chi2PDC", 10, 3, 1), ("Chi2SFG", 100, 20, 2)])
def test_equals_greens(nlm, oracle, name, N, nZ, modes):
    print("no-alloc %s N=%d" % (name, N), flush=True)
    kw = small_case(name, nlm, N=N, nZ=nZ, seed=3, poled=nZ > 16)[1]
    Ch, Sh, Cn, Sn = _both(getattr(nlm, name)(**kw), n_modes=modes)
    assert np.array_equal(Cn, Ch) and np.array_equal(Sn, Sh)
    Co, So = getattr(oracle, name)(**small_case(name, oracle, N=N, nZ=nZ, seed=3, poled=nZ > 16)[1]).computeGreensFunction()
    assert rel_l2(np.hstack([Cn, Sn]), np.hstack([Co, So])) < 1e-10


def test_table_beyond_the_scratch(nlm):
    N, nZ = 96, 50000  # 154 MB of table, 128 MiB of scratch
    m = nlm.Chi2PDC(relativeLength=1.0, nlLength=1.0, beta2=0.3, beta2s=-0.2, tMax=10, tPrecision=N, nZSteps=nZ)
    Ch, Sh, Cn, Sn = _both(m)
    assert rel_l2(np.hstack([Cn, Sn]), np.hstack([Ch, Sh])) < 1e-10

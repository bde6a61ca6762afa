"""The canonical sweep does not depend on how a state's scale is spread over its
tensors (FP64): a walker with one site times 2^-500 and its left neighbour times 2^500
is the same state, to the last bit of every product.  The squares of such a site are
near the end of the range of a double.  Bars as in the tests of the sweep's shapes:
1e-10 in the energy, 1e-12 in the orthonormality of every site."""
import numpy as np
import pytest

from mpsqmc_amd import mps as M
from mpsqmc_amd import systems
from mpsqmc_amd.engine import Engine

from .common import random_trial, rel

pytestmark = [pytest.mark.gpu, pytest.mark.usefixtures("require_gpu")]


# registers with 8 and 4 lanes a column, panels, memory
@pytest.mark.parametrize("L,D", [(8, 8), (12, 32), (13, 48), (14, 65), (17, 130)])
def test_scale_between_sites(L, D):
    s = systems.chain(L)
    tvd, tdata = random_trial(L, D, L + D)
    vd, data = random_trial(L, D, 3 * L + D)
    walkers = [data]
    for k in (L // 2, L - 2):
        T = [M.site_tensor(vd, data, q) for q in range(L)]
        T[k] = T[k] * 2.0 ** -500
        T[k - 1] = T[k - 1] * 2.0 ** 500
        walkers.append(M.from_site_tensors(T)[1])
    eng = Engine(s, tvd, tdata, n_desired=3, capacity=12, max_bond=D, precision="fp64", seed=2)
    eng.load_walkers([vd] * 3, walkers)
    eng.prepare()
    sc = eng.scalars()
    assert rel(sc["EL"][1:], np.full(2, sc["EL"][0])) < 1e-10
    assert rel(sc["O"][1:], np.full(2, sc["O"][0])) < 1e-10
    for i in range(3):
        wvd, wdata = eng.walker(i)
        for k in range(1, L):
            A = M.site_tensor(wvd, wdata, k)
            assert np.abs(np.einsum("slr,smr->lm", A, A) - np.eye(A.shape[1])).max() < 1e-12
    eng.close()

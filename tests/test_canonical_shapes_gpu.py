"""The canonical sweep's LQ at the edges of its three forms: in registers up to a
128 x 64 site (8 lanes a column up to 64 x 32, else 4), by panels of 32 columns up
to 256 x 128, in memory above.  Energy,
overlap and the right-orthonormality of every site against the oracle and plain
numpy; bars 1e-10 as for the other FP64 quantities (LQ errors are a few ulps a
site, the bar leaves four orders of magnitude)."""
import numpy as np
import pytest

from mpsqmc_amd import mps as M
from mpsqmc_amd import systems
from mpsqmc_amd.engine import Engine

from .common import oracle_population, random_trial, rel

pytestmark = [pytest.mark.gpu, pytest.mark.usefixtures("require_gpu")]


@pytest.mark.parametrize("L,D", [(3, 2), (6, 3), (11, 31), (12, 32), (12, 33), (13, 63), (13, 64), (14, 65),
                                 (15, 97), (16, 128), (17, 130)])
def test_prepare_shapes_fp64(L, D):
    s = systems.chain(L, periodic=4 < L < 14)
    tvd, tdata = random_trial(L, D, L + D)
    n = 3
    orc = oracle_population(s, tvd, tdata)
    eng = Engine(s, tvd, tdata, n_desired=n, capacity=4 * n, max_bond=D, precision="fp64", seed=2)
    walkers = [random_trial(L, max(1, D - i), 50 + i) for i in range(n)]
    one = np.ones(n)
    orc.set_walkers([w[0] for w in walkers], [w[1] for w in walkers], one, one, 0 * one)
    eng.load_walkers([w[0] for w in walkers], [w[1] for w in walkers], one, one, 0 * one)
    E = eng.prepare()
    EP, _, EL = orc.energy(1, dofluct=False)
    assert abs(E - EP) <= 1e-10 * abs(EP)
    assert rel(eng.scalars()["EL"], EL) < 1e-10
    for i in range(n):
        vd, data = eng.walker(i)
        for k in range(1, L):
            A = M.site_tensor(vd, data, k)
            assert np.abs(np.einsum("slr,smr->lm", A, A) - np.eye(A.shape[1])).max() < 1e-12
    eng.close()

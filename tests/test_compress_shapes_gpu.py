"""Recompression at the edges of its shapes: odd bonds, bonds above the size whose
work matrices fit the LDS (64), targets above the rank, a target of 1 and 2, and
chains short enough that the two-site matrix has fewer columns than its inner
bond.  Against the oracle's CompressState; bars as in the FP64 compression test
(1e-10 relative: both sides work in FP64 and the states are well conditioned)."""
import numpy as np
import pytest

import oracle
from mpsqmc_amd import mps as M
from mpsqmc_amd import systems
from mpsqmc_amd.engine import Engine

from .common import random_gauge, random_trial

pytestmark = [pytest.mark.gpu, pytest.mark.usefixtures("require_gpu")]


@pytest.mark.parametrize("L,D,targets", [(3, 2, [1, 2, 5]), (7, 5, [1, 2, 3, 4, 5]), (11, 23, [7, 11, 22, 23]),
                                         (13, 33, [2, 16, 17, 33]), (13, 64, [31, 63]), (14, 66, [5, 33, 65])])
def test_compress_shapes_fp64(L, D, targets):
    s = systems.chain(L)
    tvd, tdata = random_trial(L, D, 3 + L)
    gvd, gdata = random_gauge(tvd, tdata, 4 + L)
    n = len(targets)
    eng = Engine(s, tvd, tdata, n_desired=n, capacity=4 * n, max_bond=D, precision="fp64", seed=1)
    eng.load_copies(gvd, gdata, n)
    eng.compress_walkers(targets)
    O = eng.scalars()["O"]
    for i, t in enumerate(targets):
        ovd, odata, _ = oracle.compress(L, 2, gvd, gdata, t)
        _, odata = oracle.left_normalize(L, 2, ovd, odata)
        oO = abs(oracle.inner(L, 2, tvd, tdata, ovd, odata))
        vd, data = eng.walker(i)
        assert np.array_equal(vd, ovd), (t, vd, ovd)
        assert abs(O[i] - oO) <= 1e-10 * oO
        # sites 1.. are right-orthonormal: the norm is the first site's
        assert abs(np.linalg.norm(M.site_tensor(vd, data, 0)) - 1.0) < 1e-12
        a, b = M.to_dense(vd, data), M.to_dense(ovd, odata)
        a, b = a * np.sign(a[np.argmax(np.abs(a))]), b * np.sign(b[np.argmax(np.abs(a))])
        assert np.allclose(a, b, atol=1e-10)
    eng.close()

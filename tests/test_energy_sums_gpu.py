"""Energies of several couplings that end on one site (FP32 engines): every coupling is
summed, times its J, in FP64.

The trial's tensors are small integers and the walkers basis states (padded to wide
bonds), so every FP32 product and partial sum of a coupling is an exact integer; the
energy sum_c J_c <trial|S_i . S_j|n> = sum_c J_c (+-psi(n) / 4 + psi(n with i, j
exchanged) / 2) then carries FP64 rounding only, whatever the J.  Bar: fewer than 100
terms of a few roundings of 1.1e-16 each, 1e-13 of the sum of their magnitudes."""
import numpy as np
import pytest

from mpsqmc_amd import mps as M
from mpsqmc_amd import systems
from mpsqmc_amd.engine import Engine

from .test_engine_gpu import _run_parity

pytestmark = [pytest.mark.gpu, pytest.mark.usefixtures("require_gpu")]


def _profile(L, D):
    return np.array([min(D, 2 ** min(k, L - k)) for k in range(L + 1)], dtype=np.int32)


# products chained in 16- and in 32-column strips, and unchained (bonds above 64)
@pytest.mark.parametrize("L,D", [(9, 8), (12, 40), (14, 72)])
def test_couplings_of_any_size_and_sign(L, D):
    rng = np.random.default_rng(100 * L + D)
    J = rng.choice([-1.0, 1.0], L * (L - 1) // 2) * 10.0 ** rng.uniform(-3, 3, L * (L - 1) // 2)
    J[rng.uniform(size=J.size) < 0.4] = 0.0
    s = systems.System(L, J)
    vd = _profile(L, D)
    # about three entries +-1 in a column: no partial sum comes near 2^24
    T = []
    for k in range(L):
        f = min(1.0, 3.0 / vd[k])
        T.append(rng.choice([-1.0, 0.0, 1.0], size=(2, vd[k], vd[k + 1]), p=[f / 2, 1 - f, f / 2]))

    def psi(n, T=T):
        v = np.ones(1)
        for k in range(L):
            v = v @ T[k][n[k]]
        return v[0]

    configs = rng.integers(0, 2, size=(6, L))
    assert max(psi(n, [np.abs(t) for t in T]) for n in configs) < 2 ** 22
    walkers = []
    for n in configs:
        W = [np.zeros((2, vd[k], vd[k + 1])) for k in range(L)]
        for k in range(L):
            W[k][n[k], 0, 0] = 1.0
        walkers.append(M.from_site_tensors(W))
    tvd, tdata = M.from_site_tensors(T)
    one = np.ones(len(walkers))
    eng = Engine(s, tvd, tdata, n_desired=6, capacity=24, max_bond=D, precision="fp32", seed=1)
    assert eng.path == "general"
    eng.load_walkers([w[0] for w in walkers], [w[1] for w in walkers], one, one, 0 * one)
    eng.prepare()
    got = eng.scalars()["EL"]  # <trial|H|n> over the loaded overlap, 1
    eng.close()
    nonzero = 0
    for b, n in enumerate(configs):
        terms = []
        for i, j, Jc in zip(*s.couplings()):
            x = n.copy()
            x[i], x[j] = n[j], n[i]
            terms += [Jc * (0.25 if n[i] == n[j] else -0.25) * psi(n), 0.5 * Jc * psi(x) * (n[i] != n[j])]
        nonzero += np.abs(terms).sum() > 0
        assert abs(got[b] - np.sum(terms)) <= 1e-13 * np.abs(terms).sum()
    assert nonzero >= 4


@pytest.mark.parametrize("canon", [1, 64])
@pytest.mark.parametrize("D", [11, 16])
def test_frustrated_fp32(D, canon):
    _run_parity(systems.square_periodic(3, J1=1.0, J2=0.5), D, 6, 5 + D, 2, precision="fp32", tol=2e-4,
                check_states=False, canon=canon)

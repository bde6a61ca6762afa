"""The FP32 matrix-core products where their shapes are no multiples of anything: the
unchained kernel (bonds above 64) with operands that no 16-byte load fits and partial
last slices, under every tile table, and the chained overlaps of unequal odd bonds.

Walks: the engine in FP64 on the same inputs and uniforms, at the bars of the tile
tables' test (weights and overlaps 2e-4, local energies 2e-3).  Overlaps: the engine's
inputs rounded to FP32 and summed in FP64 by plain numpy; a site's sums of at most 2 x 64
products and the rounding of its result, 64 x 2^-24 of the sums of magnitudes at
most, over the sites: L x 4e-6 of |other| |walker|."""
import numpy as np
import pytest

from mpsqmc_amd import mps as M
from mpsqmc_amd import systems
from mpsqmc_amd.engine import Engine
from mpsqmc_amd.rng import Random

from .common import random_trial, rel

pytestmark = [pytest.mark.gpu, pytest.mark.usefixtures("require_gpu")]

TABLES = {"all16": [16] * 8, "all32": [32] * 8, "wide": [64] * 8}


def _walk(system, Dt, Dws, precision, canon, tiles=None):
    tvd, tdata = random_trial(system.L, Dt, 11)
    e = Engine(system, tvd, tdata, n_desired=len(Dws), capacity=4 * len(Dws), max_bond=max(Dws), precision=precision,
               seed=1)
    assert e.path == "general"
    rng = np.random.default_rng(7)
    ws = []
    for D in Dws:  # near the trial (overlaps of order 1): its first D states a bond, moved a little
        T = [M.site_tensor(tvd, tdata, k) for k in range(system.L)]
        T = [t + 0.2 * rng.normal(size=t.shape) / np.sqrt(t.shape[1]) for t in T]
        d = [min(D, int(x)) for x in tvd]
        ws.append(M.from_site_tensors([t[:, :d[k], :d[k + 1]] for k, t in enumerate(T)]))
    ws = [(vd, x.astype(np.float32).astype(np.float64)) for vd, x in ws]
    one = np.ones(len(ws))
    e.load_walkers([w[0] for w in ws], [w[1] for w in ws], one, one, 0 * one)
    if tiles:
        e.set_tiles(tiles)
    e.set_canonical_interval(canon)
    e.prepare()
    r = Random(13)
    out = []
    for _ in range(2):
        e.propagate(r.uniforms(e.num_walkers() * e.nC))
        sc = e.scalars()
        out.append((e.indices().copy(), sc["w"].copy(), sc["O"].copy(), sc["EL"].copy()))
    e.close()
    return out


# a lattice and a chain in a field; trial and walkers of the same and of other bonds
@pytest.mark.parametrize("table", sorted(TABLES))
@pytest.mark.parametrize("kind,Dt,Dws", [("snake", 65, [65, 64, 17, 9]), ("snake", 70, [70, 66]),
                                         ("snake", 97, [97, 33]), ("field", 100, [100, 68]),
                                         ("field", 127, [127, 126])])
@pytest.mark.parametrize("canon", [1, 64])
def test_unchained_products_fp32(kind, Dt, Dws, canon, table):
    s = systems.snake_lattice(4, 4) if kind == "snake" else systems.chain(14, h=0.4, periodic=True)
    want = _walk(s, Dt, Dws, "fp64", canon)
    got = _walk(s, Dt, Dws, "fp32", canon, TABLES[table])
    for (i1, w1, O1, E1), (i2, w2, O2, E2) in zip(got, want):
        same = np.all(i1 == i2, axis=1)
        assert same.any()
        assert rel(w1[same], w2[same]) < 2e-4
        assert rel(O1[same], O2[same]) < 2e-4
        assert rel(E1[same], E2[same]) < 2e-3
        if not same.all():
            break


# walker and probe bonds: below, at and above the strips of 16 and 32 columns
@pytest.mark.parametrize("Dw,Do", [(3, 5), (15, 17), (31, 33), (33, 31), (24, 47), (63, 49), (64, 61), (61, 64)])
def test_overlaps_of_odd_bonds_fp32(Dw, Do):
    L = 13
    s = systems.chain(L, h=0.3)  # a field: bonds up to 32 take the general layout too
    tvd, tdata = random_trial(L, Dw, 2)
    eng = Engine(s, tvd, tdata, n_desired=3, capacity=12, max_bond=Dw, precision="fp32", seed=1)
    ws = [random_trial(L, max(1, Dw - 7 * i), 20 + i) for i in range(3)]
    eng.load_walkers([w[0] for w in ws], [w[1] for w in ws])
    ovd, odata = random_trial(L, Do, 30)
    got = eng.overlaps(ovd, odata)
    eng.close()
    f = lambda x: x.astype(np.float32).astype(np.float64)
    for i, (vd, data) in enumerate(ws):
        E = np.ones((1, 1))
        norms = []
        for a, b in ((ovd, odata), (vd, data)):
            N = np.ones((1, 1))
            for k in range(L):
                T = M.site_tensor(a, f(b), k)
                N = sum(T[q].T @ N @ T[q] for q in range(2))
            norms.append(np.sqrt(N[0, 0]))
        for k in range(L):
            A, B = M.site_tensor(vd, f(data), k), M.site_tensor(ovd, f(odata), k)
            E = sum(A[q].T @ E @ B[q] for q in range(2))
        assert abs(got[i] - E[0, 0]) <= 4e-6 * L * norms[0] * norms[1]

"""The cache file of tuned tile tables: a table is taken up again only by an engine that
runs the same products on the same couplings."""
import numpy as np
import pytest

from mpsqmc_amd import systems
from mpsqmc_amd.engine import Engine

from .common import random_trial

pytestmark = [pytest.mark.gpu, pytest.mark.usefixtures("require_gpu")]

ODD = [32, 16, 64, 16, 64, 32, 16, 32]  # no default and no tuner's result


def _tiles(system, D=16, tune=False):
    vd, data = random_trial(system.L, D, 3)
    e = Engine(system, vd, data, n_desired=4, capacity=16, max_bond=D, precision="fp32", seed=1)
    if tune:
        e.load_copies(vd, data, 4)
        e.prepare()
        e.autotune(reps=1)
    t = list(e.tiles)
    e.close()
    return t


def test_tables_of_other_products_are_ignored(tmp_path, monkeypatch):
    cache = tmp_path / "tiles.txt"
    monkeypatch.setenv("MQE_TUNE_CACHE", str(cache))
    s = systems.snake_lattice(3, 3)
    default = _tiles(s)
    _tiles(s, tune=True)
    (line,) = cache.read_text().splitlines()
    key = line.split()[0]
    odd = " ".join(map(str, ODD))
    cache.write_text(f"{key} {odd}\n")
    assert _tiles(s) == ODD  # the same engine again
    monkeypatch.setenv("MQE_NO_CHAIN", "1")
    assert _tiles(s) == default  # other kernels
    monkeypatch.delenv("MQE_NO_CHAIN")
    f, g, _ = s.couplings()
    Jp = np.zeros(36)
    for a, b in sorted((i, (i + d) % 9) for d in (1, 4) for i in range(9)):
        if np.count_nonzero(Jp) < len(f):
            Jp[systems.packed_index(a, b)] = 1.0
    other = systems.System(9, Jp)
    assert len(other.couplings()[0]) == len(f)
    assert _tiles(other) == default  # as many couplings of other pairs
    cache.write_text(f"L9_nC{len(f)}_Dt16_Dw16_d2_fp32 {odd}\n")
    assert _tiles(s) == default  # a line without the products' version

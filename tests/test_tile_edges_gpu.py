"""Walks at the edges of the kernels' tiles, against the FP64 oracle on identical
inputs: the one-wave kernel of nearest-neighbour chains (FP32, bonds up to 16, and
17, the first bond beyond it; more than 64 couplings) and the chained products of
the general kernel in FP64 (strips of 16, bonds up to 64, and 65) with long-range
couplings.  Bars as in the engine's parity tests: 2e-4 in FP32, 1e-10 in FP64."""
import numpy as np
import pytest

from mpsqmc_amd import systems

from .test_engine_gpu import _run_parity

pytestmark = [pytest.mark.gpu, pytest.mark.usefixtures("require_gpu")]


@pytest.mark.parametrize("L,D", [(3, 2), (5, 3), (9, 15), (9, 16), (9, 17), (70, 4)])
@pytest.mark.parametrize("canon", [1, 64])
def test_chain_fp32(L, D, canon):
    _run_parity(systems.chain(L), D, 6, 11 * L + D, 2, precision="fp32", tol=2e-4, check_states=False, canon=canon)


@pytest.mark.parametrize("L,D", [(3, 2), (9, 15), (9, 16), (9, 17), (11, 31), (12, 33), (13, 48), (13, 64), (14, 65)])
def test_ring_fp64(L, D):
    _run_parity(systems.chain(L, periodic=L > 3), D, 3, 7 * L + D, 2, check_states=False, uneven=True, canon=2)


def test_frustrated_fp64():
    _run_parity(systems.square_periodic(3, J1=1.0, J2=0.5), 11, 3, 5, 2, check_states=False, canon=2)

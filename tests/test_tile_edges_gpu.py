"""Walks at the edges of the kernels' tiles, against the FP64 oracle on identical
inputs: the one-wave kernel of nearest-neighbour chains (FP32, bonds up to 16, and
17, the first bond beyond it; more than 64 couplings).  Bars as in the engine's
parity tests: 2e-4."""
import numpy as np
import pytest

from mpsqmc_amd import systems

from .test_engine_gpu import _run_parity

pytestmark = [pytest.mark.gpu, pytest.mark.usefixtures("require_gpu")]


@pytest.mark.parametrize("L,D", [(3, 2), (5, 3), (9, 15), (9, 16), (9, 17), (70, 4)])
@pytest.mark.parametrize("canon", [1, 64])
def test_chain_fp32(L, D, canon):
    _run_parity(systems.chain(L), D, 6, 11 * L + D, 2, precision="fp32", tol=2e-4, check_states=False, canon=canon)

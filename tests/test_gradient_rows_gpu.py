"""The network's gradient over many rows: its workspace does not grow with them beyond a
bound (2048 tiles of 32 rows), and more rows take turns in it.  One tile, exactly the
bound, one row and seven times more (the last tile ragged) against the FP64
restatement at the gradient's bar, 1e-4 of its largest element; the step of an optimiser
batch above the bound against the first step of Adam, lr sign(g)."""
import ctypes

import numpy as np
import pytest

from mpsqmc_amd._lib import lib
from mpsqmc_amd.mlp import MLP, NFEAT, NLABEL
from oracle import mlp as omlp

pytestmark = [pytest.mark.gpu, pytest.mark.usefixtures("require_gpu")]


def _free_bytes():
    free, total = ctypes.c_size_t(), ctypes.c_size_t()
    assert lib().hipMemGetInfo(ctypes.byref(free), ctypes.byref(total)) == 0
    return free.value


@pytest.mark.parametrize("n", [31, 65536, 65537, 262143])
def test_gradient_of_many_rows(n):
    H = 128
    net = MLP(NFEAT, H, NLABEL, seed=3)
    rng = np.random.default_rng(n)
    p = (rng.normal(size=net.num_params) * 0.15).astype(np.float32)
    net.set_params(p)
    X = rng.normal(size=(n, NFEAT)).astype(np.float32)
    Y = rng.normal(size=(n, NLABEL)).astype(np.float32)
    net.loss_grad(X[:1], Y[:1])
    before = _free_bytes()
    loss, g = net.loss_grad(X, Y)
    taken = before - _free_bytes()
    # the rows (inputs, targets, outputs), 190 MB of gradients and the allocator's grain
    assert taken <= 4 * n * (NFEAT + 2 * NLABEL) + (190 << 20) + (16 << 20)
    loss_o, g_o = omlp.loss_grad(p.astype(np.float64), X, Y, NFEAT, H, NLABEL)
    assert loss == pytest.approx(loss_o, rel=1e-5)
    assert np.max(np.abs(g - g_o)) <= 1e-4 * np.max(np.abs(g_o))
    net.close()


def test_adam_step_of_a_batch_above_the_bound():
    n, H, lr = 70001, 32, 1e-3
    net = MLP(NFEAT, H, NLABEL, seed=4)
    p = net.params()
    rng = np.random.default_rng(5)
    X = rng.normal(size=(n, NFEAT)).astype(np.float32)
    Y = rng.normal(size=(n, NLABEL)).astype(np.float32)
    loss = net.fit(X, Y, epochs=1, batch=n, lr=lr, standardize=False)
    loss_o, g_o = omlp.loss_grad(p.astype(np.float64), X, Y, NFEAT, H, NLABEL)
    assert loss == pytest.approx(loss_o, rel=1e-5)
    big = np.abs(g_o) > 1e-2 * np.abs(g_o).max()  # 100 times the gradient's bar; eps = 1e-8 is far below
    assert big.sum() > 100
    # the step in FP32 parameters of order 1: an ulp of them, 1e-7, is 1e-4 of lr
    np.testing.assert_allclose((net.params().astype(np.float64) - p)[big], -lr * np.sign(g_o[big]), atol=1e-3 * lr)
    net.close()

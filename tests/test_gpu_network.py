"""The network's gradient kernel at the edges of its row blocks (64 rows a workgroup, one workgroup a compute unit, then
several row blocks each), and the update kernel's Adam step, against the FP64 network oracle with the kernels' BF16
rounding points. Bars: the oracle rounds the same values, so the gradients differ by FP32 summation (1e-6 of a sum of
terms of one size) and by the few operands that FP32 noise carries over a BF16 rounding boundary (2^-9 of an operand, one
in 2^7 operands: below 1e-4 of the gradient's norm); 1e-3 is ten times that."""
import os
import sys

import numpy as np
import pytest

from spg_amd import native

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "oracle"))
import mlp_oracle as mo  # noqa: E402

pytestmark = pytest.mark.gpu


def _data(n, seed=2):
    rng = np.random.default_rng(seed)
    return (rng.standard_normal((n, 24)).astype(np.float32), (0.5 * rng.standard_normal((n, 3))).astype(np.float32))


@pytest.mark.parametrize("n", [1, 15, 16, 17, 63, 64, 65, 4096, 16384, 16385, 40000])
def test_gradient_at_row_block_edges(n):
    net = native.Mlp(device=0, seed=5)
    rng = np.random.default_rng(9)
    net.set_normalization(0.1 * rng.standard_normal(24), rng.uniform(0.5, 2.0, 24))
    p = net.params() + (0.05 * rng.standard_normal(native.MLP_NUM_PARAMS)).astype(np.float32)  # biases too
    net.set_params(p)
    f, t = _data(n)
    mean, std = net.normalization()
    loss, g = net.loss_grad(f, t)
    el, eg = mo.loss_grad(p, f, t, mean, std, emulate=True)
    assert abs(loss - el) < 1e-4 * el
    assert np.linalg.norm(g - eg) < 1e-3 * np.linalg.norm(eg)
    again = net.loss_grad(f, t)
    assert again[0] == loss and np.array_equal(again[1], g)


@pytest.mark.parametrize("n,batch", [(100, 128), (20000, 20032)])
def test_one_adam_step_follows_the_gradient(n, batch):
    """A first step of Adam from zero moments, from loss_grad's own gradient (the rows are shuffled: the sums over row
    blocks differ in FP32, 1e-5 of an entry whose terms cancel)."""
    net = native.Mlp(device=0, seed=6)
    f, t = _data(n)
    p = net.params()
    _, g = net.loss_grad(f, t)
    lr = 1e-3
    loss = net.train(f, t, epochs=1, batch=batch, lr=lr, seed=3, standardize=False)
    step = lr * g / (np.abs(g) + 1e-8)
    moved = p - net.params()
    sure = np.abs(g) > 1e-3 * np.abs(g).max()  # entries whose sign FP32 noise does not decide
    assert np.allclose(moved[sure], step[sure], rtol=2e-4, atol=1e-7)
    y = net.forward(f)  # the fragments of inference follow the update
    e = mo.forward(net.params(), f, emulate=True)
    assert np.linalg.norm(y - e) < 5e-3 * np.linalg.norm(e)
    assert loss[0] > 0

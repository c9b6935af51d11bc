"""The network's weight gradients on grids whose rows do not fill whole runs
of 8 voxels on some level (24 -> 12 -> 6 -> 3, 8 -> 4 -> 2 -> 1, 40 -> 20 ->
10 -> 5), against the numpy restatement."""
from __future__ import annotations

import numpy as np
import pytest

from oracle import nn_oracle as N
from tests.test_gpu_nn import _net, _params

pytestmark = pytest.mark.gpu


# The restatement's own gradients move by up to 20 % (cosine 0.99) under
# 1e-3 relative input noise, through the BF16 roundings and leaky-ReLU slopes
# it flips: a wrong tap, run or halo is far outside that.
@pytest.mark.parametrize("shape", [(16, 16, 24), (16, 32, 8), (8, 16, 40)])
def test_weight_gradients_of_partial_runs(shape):
    import torch
    print(f"[gpu] wgrad {shape}", flush=True)
    P = _params(7)
    rng = np.random.default_rng(8)
    inp = rng.standard_normal((2,) + shape).astype(np.float32)
    dout = rng.standard_normal(shape).astype(np.float32)
    net = _net(torch, shape, P)
    x = torch.from_numpy(inp).cuda().reshape(2, -1).contiguous()
    out = torch.empty(x.shape[1], device="cuda")
    d = torch.from_numpy(dout).cuda().reshape(-1).contiguous()
    net.zero_grad()
    net.forward(x, out)
    net.backward(d)
    g = net.grads().astype(np.float64)
    on = N.Net(P.astype(np.float64))
    on.forward(inp.astype(np.float64))
    go = on.backward(dout.astype(np.float64))
    L, head, _ = N.layout()
    for li, (ci, co, _, wo, bo) in enumerate(L):
        a, b = g[wo:bo].reshape(co, 27, ci), go[wo:bo].reshape(co, 27, ci)
        if li == 0:
            assert not a[:, :, 2:].any()
            a, b = a[:, :, :2], b[:, :, :2]
        a, b = a.ravel(), b.ravel()
        rel = np.abs(a - b).max() / np.abs(b).max()
        cos = a @ b / (np.linalg.norm(a) * np.linalg.norm(b))
        print(f"[gpu] layer {li} rel {rel:.2e} cos {cos:.6f}", flush=True)
        assert rel < 0.2 and cos > 0.99, li
    # A second sample adds to the gradients of the first.
    net.forward(x, out)
    net.backward(d)
    g2 = net.grads().astype(np.float64)
    assert np.abs(g2 - 2 * g).max() <= 1e-5 * np.abs(g).max()

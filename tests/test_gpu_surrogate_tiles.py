"""Surrogate GEMM tiles at their edges: result tiles that end inside a 64- or 128-wide tile, K chunks
with a remainder, ragged row counts, and each rule that picks a tile size.

Every result is one sum over K in the same order whatever tile computes it, so the forward pass must
agree bit for bit between tile sizes; gradients are compared with the float64 restatement that rounds
to bfloat16 where the kernels do (tolerances of tests/test_gpu_surrogate.py: FP32 accumulation order
and bfloat16 rounding flips)."""
import os
import sys

import numpy as np
import pytest
import torch

import surrogate

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "oracle"))
import surrogate_ref as sr  # noqa: E402

pytestmark = pytest.mark.gpu

# one 64-value K chunk; K of 192 and 320 = 256 + 64; K of 576 and 640 = 2 chunks and a remainder
NETS = [dict(n_freq=32, width=64, depth=1, out_dim=64), dict(n_freq=96, width=192, depth=2, out_dim=320),
        dict(n_freq=160, width=640, depth=2, out_dim=704)]


def make(shape, max_batch, seed=3):
    net = surrogate.Net(in_dim=6, freq_sigma=0.5, seed=seed, max_batch=max_batch, **shape)
    p, B = net.get_params()
    p = p + np.float32(0.01) * np.random.default_rng(2).standard_normal(len(p)).astype(np.float32)
    net.set_params(p)
    return net, p, B


@pytest.mark.parametrize("shape", NETS)
@pytest.mark.parametrize("rows", [1, 65, 2250, 4200])
def test_forward_is_the_same_from_every_tile(shape, rows):
    net, _, _ = make(shape, 64)  # 64 rows a pass: 32x32 tiles
    x = np.random.default_rng(4).random((rows, 6)).astype(np.float32)
    ref = net.forward(x)
    xd = torch.from_numpy(x).to("cuda:0")
    y = torch.full((rows * shape["out_dim"] + 1,), float("nan"), device="cuda:0")
    torch.cuda.synchronize()
    # as many rows a pass as the scratch array takes (4200 x 704: 128x128 tiles, 2250 x 704: 64x64),
    # into a buffer that is only 4-byte aligned
    net.forward_device(rows, xd.data_ptr(), y.data_ptr() + 4)
    assert np.array_equal(y[1:].cpu().numpy().reshape(ref.shape), ref)
    assert bool(torch.isnan(y[0]))


@pytest.mark.parametrize("shape,rows", list(zip(NETS, (64, 192, 576))))
def test_gradients_at_tile_edges(shape, rows):
    net, p, B = make(shape, rows)
    rng = np.random.default_rng(6)
    x, t = rng.random((rows, 6)), rng.standard_normal((rows, shape["out_dim"]))
    w = 1.0 / (rows * (t * t).sum(axis=1))
    loss, g = net.gradients(x, t, w)
    rloss, rg = sr.loss_and_grad(p.astype(np.float64), B, x.astype(np.float32), t.astype(np.float32),
                                 w.astype(np.float32), net.shapes(), emulate=True)
    assert abs(loss - rloss) <= 1e-3 * rloss
    o = 0
    for m, k in net.shapes():
        for size in (m * k, m):
            a, b = np.asarray(g[o:o + size], np.float64), rg[o:o + size]
            assert np.linalg.norm(a - b) <= 1e-2 * np.linalg.norm(b)
            o += size

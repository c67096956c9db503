"""The 128-wide tile where it ends inside the result in both directions, in each of its epilogues, against
the 32-wide tile: the sum over K has one order, so results agree bit for bit. And host queries whose
outputs are more than a page-locked slab's kernels write themselves."""
import os
import re

import numpy as np
import pytest
import torch

import surrogate

pytestmark = pytest.mark.gpu

SRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "dgfem-acoustic_amd", "csrc",
                   "surrogate.hip")


def tile(rows, n):
    """The tile that a layer of `rows` x `n` takes, by the rule and the lines in the source."""
    line = {int(k): int(v) for k, v in re.findall(r"kTiles(\d+) = (\d+)", open(SRC).read())}
    count = lambda t: -(-rows // t) * -(-n // t)  # noqa: E731
    return next((t for t in (128, 64) if count(t) >= line[t]), 32)


# output layer (EPI_BIAS, rows and columns cut off); hidden layers (EPI_BIAS_ACT) and the output
@pytest.mark.parametrize("shape,rows", [(dict(n_freq=32, width=64, depth=1, out_dim=2112), 4100),
                                        (dict(n_freq=32, width=2112, depth=2, out_dim=2112), 4100)])
def test_large_tile_ends_inside_the_result(shape, rows):
    padded = -(-rows // 64) * 64
    assert tile(padded, 2112) == 128 and padded % 128 == 64 and 2112 % 128 == 64
    assert tile(64, 2112) == 32
    x = np.random.default_rng(4).random((rows, 6)).astype(np.float32)
    y = {}
    for max_batch in (64, padded):
        net = surrogate.Net(in_dim=6, freq_sigma=0.5, seed=3, max_batch=max_batch, **shape)
        y[max_batch] = net.forward(x)
        if shape["depth"] == 1:  # all rows in one pass of the scratch array as well
            assert 24576 * padded // 64 <= 16 << 20
            xd = torch.from_numpy(x).cuda()
            yd = torch.full((rows + 1, 2112), float("nan"), device="cuda")
            torch.cuda.synchronize()
            net.forward_device(rows, xd.data_ptr(), yd.data_ptr())
            assert np.array_equal(yd[:rows].cpu().numpy(), y[64])
            assert bool(torch.isnan(yd[rows]).all())
        net.close()
    assert np.array_equal(y[64], y[padded])


@pytest.mark.parametrize("rows", [256, 257, 1023])
def test_outputs_on_either_side_of_the_slab(rows):
    """2 MB of outputs, a row more, and 8 MB, each in one pass, against passes of 64 rows."""
    x = np.random.default_rng(5).random((rows, 6)).astype(np.float32)
    y = []
    for max_batch in (64, 1024):
        net = surrogate.Net(seed=2, n_freq=32, width=64, depth=2, out_dim=2048, max_batch=max_batch)
        y.append(net.forward(x))
        net.close()
    assert np.array_equal(*y)

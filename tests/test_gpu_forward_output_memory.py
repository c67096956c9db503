"""dgs_forward_noalloc with its outputs in memory that a kernel of the network's GPU must not write
directly: pageable and page-locked host memory, in one pass and in several, the last one ragged. The
results go through the scratch array and a copy, and equal those of an output on the device bit for bit."""
import numpy as np
import pytest
import torch

import surrogate

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rows,shape", [(1, dict(n_freq=32, width=64, depth=1, out_dim=64)),
                                        (130, dict(n_freq=64, width=128, depth=2, out_dim=704)),
                                        (3777, dict(n_freq=128, width=512, depth=3, out_dim=2048))])
@pytest.mark.parametrize("locked", [False, True])
def test_outputs_in_host_memory(rows, shape, locked):
    net = surrogate.Net(in_dim=6, seed=3, max_batch=64, **shape)
    x = torch.from_numpy(np.random.default_rng(4).random((rows, 6)).astype(np.float32)).cuda()
    ref = torch.empty(rows, shape["out_dim"], device="cuda")
    # one value of another kind on either side
    y = torch.full((rows * shape["out_dim"] + 2,), -7.0, pin_memory=locked)
    torch.cuda.synchronize()
    net.forward_device(rows, x.data_ptr(), ref.data_ptr())
    net.forward_device(rows, x.data_ptr(), y.data_ptr() + 4)
    assert torch.equal(y[1:-1].view(rows, -1), ref.cpu())
    assert y[0] == -7.0 and y[-1] == -7.0
    net.close()

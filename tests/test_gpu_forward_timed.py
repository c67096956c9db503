"""dgs_forward_timed runs on the rows of the last pass. The time is all that it returns, so the rows are
told apart by what they cost: sinf and cosf reduce arguments of 1e30 by another, longer path than those of
the unit cube. In this network, 2048 frequencies and little else, that is a third of the pass's time; the
time of one set of rows repeats to a few percent, so a tenth tells them apart."""
import numpy as np
import pytest

import surrogate

pytestmark = pytest.mark.gpu

ROWS = 16384


def rows(scale):
    return (scale * np.random.default_rng(1).random((ROWS, 6))).astype(np.float32)


def forward(net, x):
    net.forward(x)


def gradients(net, x):
    net.gradients(x, np.zeros((ROWS, 64)), np.ones(ROWS))


def train(net, x):
    net.set_data(x, np.zeros((ROWS, 64)), np.ones(ROWS))
    net.train(1, ROWS, 0.0)


@pytest.mark.parametrize("call", [forward, gradients, train])
def test_timed_pass_runs_on_the_last_rows(call):
    net = surrogate.Net(seed=1, n_freq=2048, width=64, depth=1, out_dim=64, max_batch=ROWS)
    net.forward_ms(ROWS)
    ms = {}
    for scale in (1.0, 1e30, 1.0, 1e30):
        call(net, rows(scale))
        ms[scale] = min(ms.get(scale, 1e9), net.forward_ms(ROWS))
    print(ms, flush=True)
    assert ms[1e30] > 1.1 * ms[1.0]
    net.close()

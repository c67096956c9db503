"""States in and out in every layout (field planes of the thread-per-node kernel, interleaved fields), on
either side of the size up to which the kernels read and write page-locked memory themselves (2 MB of FP64
planes), alone and at an offset inside a batch group."""
import numpy as np
import pytest

import dgk
from workloads import conf

pytestmark = pytest.mark.gpu

TEXT = conf("Wall=Reflecting\nAbs=Absorbing\n")
# unknown counts of 4 planes: 2,097,120 and 2,097,600 bytes around 2 MB = 2,097,152, and 96 bytes
LINES = [(21845, 2), (21850, 2), (1, 2)]


def state(m, seed):
    return np.random.default_rng(seed).standard_normal((4, m.K * m.Np))


@pytest.mark.parametrize("K,p", LINES)
@pytest.mark.parametrize("precision,flags,variant", [(dgk.FP64, 0, dgk.VARIANT_LDS), (dgk.FP64, 0, dgk.VARIANT_MFMA),
                                                     (dgk.FP32, dgk.FP32_PLAIN_STATE, dgk.VARIANT_LDS),
                                                     (dgk.FP32, dgk.FP32_PLAIN_STATE, dgk.VARIANT_MFMA)])
def test_states_in_and_out(K, p, precision, flags, variant):
    m = dgk.gen_line(K, 1.0, p, [1, 2], "1:Wall;2:Abs", TEXT)
    s = dgk.Solver(m, 340.0, 1.225, precision=precision, fp32_flags=flags, variant=variant)
    for seed in (1, 2):
        u = state(m, seed)
        s.set_state(u)
        got = s.get_state()
        assert np.array_equal(got, u if precision == dgk.FP64 else u.astype(np.float32))
        r = s.rhs(u, 1e-6)
        assert np.isfinite(r).all() and np.array_equal(s.get_state(), got)  # the state is left alone
    u[2:] = 0  # the planes that are no fields of a line: their rates are zero
    assert not s.rhs(u, 1e-6)[2:].any()


def test_members_of_a_batch_group():
    meshes = [dgk.gen_line(K, 1.0, p, [1, 2], "1:Wall;2:Abs", TEXT) for K, p in LINES]
    b = dgk.Batch(meshes, [dict(c0=340.0, rho0=1.225, v0=(0.0, 0.0, 0.0))] * 3, [1e-8] * 3, precision=dgk.FP64)
    us = [state(m, i) for i, m in enumerate(meshes)]
    for order in ((0, 1, 2), (2, 1, 0)):
        for i in order:
            b.set_state(i, us[i])
        for i in order:
            assert np.array_equal(b.get_state(i), us[i])

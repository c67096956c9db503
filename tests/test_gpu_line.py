"""The 1D stage kernel, whose workgroup shares the work of its 16 elements and gives each face one thread,
against the oracle: element counts around one and two tiles and from one workgroup to many, both
addressing forms, with and without a live second velocity component."""
import numpy as np
import pytest

import dgk
import oracle_binding as ob
from test_gpu_parity import mixed_mesh, rel

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("p", [1, 2, 3, 4, 5])
@pytest.mark.parametrize("K", [1, 15, 16, 17, 33, 5003])
@pytest.mark.parametrize("precision,flags", [(dgk.FP64, 0), (dgk.FP32, 0), (dgk.FP32, dgk.FP32_PLAIN_STATE)])
def test_line(p, K, precision, flags):
    m = mixed_mesh(1, p, K)
    v0, steps, dt = (40.0, 0.0, 0.0), 30, 0.1 / K / (380.0 * (2 * p + 1))
    o = ob.Oracle(m, 340.0, 1.225, v0=v0, sign_mode=ob.SIGN_STABLE)
    rng = np.random.default_rng(K + p)
    x = m.node_xyz[:, 0]
    for live in (2, 3):
        u = np.zeros((4, m.K * m.Np))
        for q in range(live):
            u[q] = np.sin(5 * x + rng.random()) * (1.0 if q == 0 else 2e-3)
        ref = o.step(u, steps, dt)
        got = []
        for addr64 in (False, True):
            s = dgk.Solver(m, 340.0, 1.225, v0=v0, precision=precision, flux_sign=dgk.SIGN_STABLE, fp32_flags=flags,
                           addr64=addr64)
            s.set_state(u)
            s.rk4(steps, dt)
            got.append(s.get_state())
            s.close()
        # the bounds of the other parity tests
        assert rel(got[0], ref) <= (1e-12 if precision == dgk.FP64 else 1e-5)
        assert np.array_equal(*got)

"""The record's row goes forward once a step however many workgroups write it: receivers around one
workgroup's 16 and around the 256 workgroups' 4096, over captured sequences of 25 steps with single steps
between them, until the record is full and past it, and from the beginning after it is set again."""
import numpy as np
import pytest

import dgk
import oracle_binding as ob
from interp import interp_weights
from test_gpu_parity import mixed_mesh, rel
from test_gpu_receivers import points, smooth_state

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 16, 17, 4096, 4097])
def test_rows_of_a_record(n):
    m = mixed_mesh(2, 2)
    pts, u0, dt, cap = points(2, n, n), smooth_state(m), 2e-6, 60
    s = dgk.Solver(m, 340.0, 1.225, flux_sign=dgk.SIGN_STABLE)
    s.set_state(u0)
    s.set_receivers(pts, cap)
    found = [interp_weights(m, x) for x in pts]
    nodes = np.array([e * m.Np + np.arange(m.Np) for e, _ in found])
    w = np.array([w for _, w in found])
    o = ob.Oracle(m, 340.0, 1.225, sign_mode=ob.SIGN_STABLE)
    u, ref = u0, []
    for _ in range(cap):
        u = o.step(u, 1, dt)
        ref.append((w * u[0][nodes]).sum(axis=1))
    ref = np.array(ref)
    for again in range(2):
        done = 0
        for steps in (25, 3, 27, 25):  # 80 steps: the last 20 have no row
            s.rk4(steps, dt)
            done = min(done + steps, cap)
            rec = s.get_receivers()
            # the bound of the other receiver tests
            assert rec.shape == (done, n) and rel(rec, ref[:done]) <= 1e-12
        s.set_state(u0)
        s.set_receivers(pts, cap)

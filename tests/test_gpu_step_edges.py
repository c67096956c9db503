"""Receivers and sources between time steps, where one launch does both, and where it does not: one
and several sources (overlapping: the later one wins), more sources than one launch takes, a source of
more nodes than one launch takes, none to many receivers, several captured step sequences."""
import numpy as np
import pytest

import dgk
import oracle_binding as ob
from interp import sample
from test_gpu_parity import mixed_mesh, rel
from test_gpu_receivers import points, smooth_state

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dim,p,nsrc,nrec,precision", [(2, 2, 1, 5, dgk.FP64), (2, 2, 9, 5, dgk.FP64),
                                                       (2, 3, 3, 0, dgk.FP64), (3, 3, 2, 65, dgk.FP64),
                                                       (2, 4, 3, 17, dgk.FP32), (3, 5, 8, 64, dgk.FP32)])
def test_sources_and_receivers_between_steps(dim, p, nsrc, nrec, precision):
    m = mixed_mesh(dim, p)
    u0, dt, steps = smooth_state(m), 2e-6, 30  # a 25-step sequence and one of 5
    rng = np.random.default_rng(nsrc)
    c = m.node_xyz.mean(axis=0)
    src = [[0, *(c + 0.05 * rng.standard_normal(3) * (np.arange(3) < dim)), 0.2, 0.5 + 0.1 * k, 4e3, 0.2 * k,
            (12 + 3 * k) * dt] for k in range(nsrc)]
    ts = np.arange(steps) * dt
    pts = points(dim, max(nrec, 1), 10)[:nrec]
    s = dgk.Solver(m, 340.0, 1.225, flux_sign=dgk.SIGN_STABLE, precision=precision)
    s.set_sources(src)
    s.set_state(u0)
    if nrec:
        s.set_receivers(pts, steps)
    s.rk4(steps, dt, ts)
    o = ob.Oracle(m, 340.0, 1.225, sign_mode=ob.SIGN_STABLE)
    u, rows = u0, []
    for i in range(steps):
        u = o.step(u, 1, dt, t_steps=ts[i:i + 1], sources=src)
        rows.append(sample(m, u, pts) if nrec else [])
    # FP64: the bound of the other parity tests; FP32: theirs after 60 steps
    tol = 1e-12 if precision == dgk.FP64 else 1e-5
    assert rel(s.get_state(), u) <= tol
    if nrec:
        rec = s.get_receivers()
        assert rec.shape == (steps, nrec)
        assert rel(rec, np.array(rows)) <= tol


def test_source_of_many_nodes():
    m = dgk.gen_rect(40, 40, 1.0, 0.8, 3, [1, 2, 1, 2], "1:Wall;2:Abs",
                     "timeStart=0\ntimeEnd=1\ntimeStep=1\ntimeRate=1\nelementType=Lagrange\n"
                     "timeIntMethod=Runge-Kutta\nnumThreads=1\nv0_x=0\nv0_y=0\nv0_z=0\nrho0=1.225\nc0=340\n"
                     "Wall=Reflecting\nAbs=Absorbing\n")
    src = [[0, 0.5, 0.4, 0.0, 0.35, 0.7, 3e3, 0.1, 1.0]]
    assert np.sum(((m.node_xyz - [0.5, 0.4, 0.0]) ** 2).sum(axis=1) < 0.35 ** 2) > 8192
    u0, dt, pts = smooth_state(m), 2e-6, points(2, 3, 4)
    s = dgk.Solver(m, 340.0, 1.225)
    s.set_sources(src)
    s.set_state(u0)
    s.set_receivers(pts, 8)
    ts = np.arange(6) * dt
    s.rk4(6, dt, ts)
    o = ob.Oracle(m, 340.0, 1.225)
    u, rows = u0, []
    for i in range(6):
        u = o.step(u, 1, dt, t_steps=ts[i:i + 1], sources=src)
        rows.append(sample(m, u, pts))
    assert rel(s.get_state(), u) <= 1e-12
    assert rel(s.get_receivers(), np.array(rows)) <= 1e-12

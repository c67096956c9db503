"""What happens around and between time steps: receivers and sources, where one launch does both and
where it does not (one and several sources, overlapping, so that the later one wins; more sources than
one launch takes; a source of more nodes than one launch takes; none to many receivers; several
captured step sequences); points located in the mesh; states handed over."""
import numpy as np
import pytest

import dgk
import oracle_binding as ob
from interp import sample
from test_gpu_parity import mixed_mesh, rel
from test_gpu_receivers import oracle_series, points, smooth_state

pytestmark = pytest.mark.gpu

CONF = ("timeStart=0\ntimeEnd=1\ntimeStep=1\ntimeRate=1\nelementType=Lagrange\ntimeIntMethod=Runge-Kutta\n"
        "numThreads=1\nv0_x=0\nv0_y=0\nv0_z=0\nrho0=1.225\nc0=340\nWall=Reflecting\nAbs=Absorbing\n")


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
    m = dgk.gen_rect(40, 40, 1.0, 0.8, 3, [1, 2, 1, 2], "1:Wall;2:Abs", CONF)
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


@pytest.mark.parametrize("dim,p", [(1, 2), (2, 3), (3, 2)])
def test_many_receivers_and_a_reset_record(dim, p):
    """Hundreds of points spread over the mesh, then the same number at other places with the same
    capacity (buffers and captured steps are kept), then another number."""
    m = mixed_mesh(dim, p)
    u0, dt = smooth_state(m), 2e-6
    s = dgk.Solver(m, 340.0, 1.225, flux_sign=dgk.SIGN_STABLE)
    for n, seed in ((300, 1), (300, 2), (7, 3)):
        pts = points(dim, n, seed)
        s.set_state(u0)
        s.set_receivers(pts, 4)
        s.rk4(4, dt)
        rec = s.get_receivers()
        ref = oracle_series(m, u0, 4, dt, pts)
        assert rec.shape == ref.shape and rel(rec, ref) <= 1e-12


@pytest.mark.parametrize("precision", [dgk.FP64, dgk.FP32])
@pytest.mark.parametrize("cells,p", [((3, 2), 1), ((70, 61), 3), ((151, 149), 5)])
def test_state_hand_over(cells, p, precision):
    """States of 1 KB, 2.7 MB and 30 MB, whose hand-over takes different ways, in and out and through one
    operator evaluation, with and without a live third velocity component."""
    m = dgk.gen_rect(*cells, 1.0, 0.8, p, [1, 2, 1, 2], "1:Wall;2:Abs", CONF)
    rng = np.random.default_rng(3)
    s = dgk.Solver(m, 340.0, 1.225, precision=precision)
    for planes in (3, 4):
        u = np.zeros((4, m.K * m.Np))
        u[:planes] = rng.standard_normal((planes, m.K * m.Np))
        s.set_state(u)
        got = s.get_state()
        if precision == dgk.FP64:
            assert np.array_equal(got, u)
        else:  # an FP32 value and a bfloat16 remainder: 2^-33 of it, 2^-30 as elsewhere in the tests
            assert np.max(np.abs(got - u) / np.maximum(np.abs(u), 1e-30)) <= 2.0 ** -30
        assert not np.any(got[planes:])
        r = s.rhs(u, 1e-6)
        assert not np.any(r[planes:])
        s.euler(1, 1e-6)
        # u + r in the state's precision: u rounded to it, dt L(u) rounded or fused, and the sum rounded
        eps = 2.0 ** -52 if precision == dgk.FP64 else 2.0 ** -22
        assert np.all(np.abs(s.get_state() - (u + r)) <= eps * (np.abs(u) + np.abs(r)))

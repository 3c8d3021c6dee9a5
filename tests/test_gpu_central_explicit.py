"""A central viscous box with the explicit gradient (conschm 643c with difschm
643e: convection 0, deriv_explicit 1).  Only the gradients are explicit there;
the fluxes are differentiated with the compact scheme.  The gradients against
the checker's diff6ec line by line (both sides round alike but for the metric
factor, within 4 eps of it), qrhs against the fluxes of those gradients in
numpy and the checker's df_compact, whole steps against the stage pieces.

Tolerance of qrhs: a node's G is a sum of at most 12 products of a few factors
each, wrong by at most 16 eps times the sum S of their magnitudes; df_compact's
right-hand side sums to 2 (7/9 + 1/36) in magnitude and the inverse of its
system (1/3, 1, 1/3) has the maximum norm 3, its own rounding being smaller; so
each of the three axes is wrong by at most 5 * 16 eps S xi J."""
import numpy as np
import pytest

import astr_gpu_amd as ag
import pyoracle as po
from test_gpu_parity import lines_ref

pytestmark = pytest.mark.gpu
HM = 5
EPS = np.finfo(np.float64).eps


def wrapped(a, dims):
    """the field with halos and the nodes n from the nodes 0..n-1"""
    for ax in range(3):
        a = np.take(a, (np.arange(-HM, dims[ax] + HM + 1) % dims[ax]) + HM, axis=ax)
    return np.asfortranarray(a)


def smooth_state(p):
    dims = (p.im, p.jm, p.km)
    x, y, z = np.meshgrid(*[2 * np.pi * np.arange(-HM, n + HM + 1) / n for n in dims],
                          indexing="ij")
    rho = 1.0 + 0.05 * np.sin(x + 2 * y - z)
    vel = np.stack([np.sin(x) * np.cos(2 * y) * np.cos(z) + 0.3 * np.cos(2 * z),
                    -np.cos(x) * np.sin(y) * np.cos(z), 0.4 * np.sin(x + y) * np.cos(2 * z)], axis=-1)
    tmp = 1.0 + 0.1 * np.cos(x - y) * np.sin(z)
    prs = rho * tmp / (p.gamma * p.mach ** 2)
    rho, prs, tmp = (wrapped(a, dims) for a in (rho, prs, tmp))
    vel = np.asfortranarray(np.stack([wrapped(vel[..., m], dims) for m in range(3)], axis=-1))
    e = prs / (p.gamma - 1.0) + 0.5 * rho * (vel ** 2).sum(axis=-1)
    q = np.asfortranarray(np.stack([rho] + [rho * vel[..., m] for m in range(3)] + [e], axis=-1))
    return dict(q=q, rho=rho, vel=vel, prs=prs, tmp=tmp)


def solver(dims, npdc):
    p = ag.default_params(dims, npdci=npdc[0], npdcj=npdc[1], npdck=npdc[2], deriv_explicit=1)
    s = ag.AstrSolver(p)
    jac, dxi = ag.box_metrics(p)
    s.upload_geom(jac, dxi)
    st = smooth_state(p)
    s.upload_state(st["q"], st["rho"], st["vel"], st["prs"], st["tmp"])
    return s, p, st, jac.flat[0], [dxi[HM, HM, HM, d, d] for d in range(3)]


@pytest.mark.parametrize("npdc", [(3, 3, 3), (4, 3, 3), (3, 4, 4)])
@pytest.mark.parametrize("dims", [(16, 18, 20), (33, 17, 19)])
def test_gradients_are_explicit(dims, npdc):
    print(f"case central explicit gradients {dims} {npdc}", flush=True)
    s, p, st, _, xi = solver(dims, npdc)
    s.rhscal()
    g = s.download_rhs()
    for m in range(4):
        f = st["vel"][..., m] if m < 3 else st["tmp"]
        for d in range(3):
            ref = lines_ref(lambda ln: po.diff6ec(npdc[d], ln), f, d + 1) * xi[d]
            got = g["dvel"][..., m, d] if m < 3 else g["dtmp"][..., d]
            assert np.max(np.abs(got - ref)) <= 4 * EPS * np.max(np.abs(ref)), (m, d)
    s.close()


@pytest.mark.parametrize("dims", [(16, 18, 20), (33, 17, 19)])
def test_qrhs_of_the_explicit_gradients(dims):
    print(f"case central explicit qrhs {dims}", flush=True)
    s, p, st, jac, xi = solver(dims, (3, 3, 3))
    s.rhscal()
    g = s.download_rhs()
    s.close()
    ins = [ag.interior(a, p) for a in (st["q"], st["vel"], st["prs"], st["tmp"])]
    q, vel, prs, tmp = ins
    dv, dt = g["dvel"], g["dtmp"]
    tc = p.sutherland / p.ref_tem
    miu = tmp * np.sqrt(tmp) * (1.0 + tc) / (tmp + tc) / p.reynolds
    hcc = miu / p.prandtl / ((p.gamma - 1.0) * p.mach ** 2)
    div = dv[..., 0, 0] + dv[..., 1, 1] + dv[..., 2, 2]
    sg = np.empty_like(dv)
    for a in range(3):
        for b in range(3):
            sg[..., a, b] = miu * (dv[..., a, b] + dv[..., b, a] - (2.0 / 3.0) * div * (a == b))
    ref, tol = np.zeros_like(q), 0.0
    for d in range(3):
        u = vel[..., d]
        gr = np.empty_like(q)
        gr[..., 0] = -q[..., 0] * u
        for m in range(3):
            gr[..., 1 + m] = sg[..., m, d] - (q[..., 1 + m] * u + (m == d) * prs)
        work = (sg[..., :, d] * vel).sum(axis=-1)
        gr[..., 4] = hcc * dt[..., d] + work - (q[..., 4] + prs) * u
        size = (np.abs(q[..., 4]) + prs) * np.maximum(np.abs(u), 1.0) + np.abs(sg).sum(axis=(-2, -1)) + \
            np.abs(hcc * dt[..., d])
        tol += 5 * 16 * EPS * float(np.max(size)) * xi[d] * jac
        for m in range(5):
            full = np.empty(ag.haloed_shape(p))
            full[HM:-HM, HM:-HM, HM:-HM] = gr[..., m] * (xi[d] * jac)
            ref[..., m] += lines_ref(lambda ln: po.df_compact(3, ln), wrapped(full, dims), d + 1)
    err = float(np.max(np.abs(g["qrhs"] - ref)))
    print(f"  {err:.2e} of {tol:.2e}")
    assert err <= tol


def test_steps_equal_pieces():
    dims, dt = (33, 17, 19), 0.002
    s1, p, _, _, _ = solver(dims, (3, 4, 3))
    s2 = solver(dims, (3, 4, 3))[0]
    for _ in range(2):
        a = s1.time_integration_rk(dt, stats=True)
        for stage in (1, 2, 3):
            s2.filterq()
            s2.qswap()
            s2.rhscal()
            if stage == 1:
                b = s2.statcal()
            s2.rk3_update(stage, dt)
        # the two sum the same terms in another order
        assert all(abs(x - y) <= 1e-13 * abs(y) for x, y in zip(a, b)), (a, b)
    a, b = s1.download_state(), s2.download_state()
    for nm in a:
        # as test_stage_pieces_reproduce_the_fused_step, two steps
        assert np.max(np.abs(a[nm] - b[nm])) <= 2e-14 * np.max(np.abs(b[nm])), nm
    s1.close()
    s2.close()

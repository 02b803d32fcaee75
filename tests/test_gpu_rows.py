"""The 3-D FP64 step's fused positivity, NAD, commit, wall and collision at the
row lengths where its variants change (rows of 4, 8 and 16 values a lane in
registers, longer rows read again), with both limiters firing, the mass sums
around the lengths of their unrolled loop, and particles and walls whose
collision does not scale with g.

Tolerances: 1e-10 relative on g and the moments (the FP64 step's); limiter
flags identical.
"""
from __future__ import annotations

import numpy as np
import pytest

import alebgk4paper_amd as A
import oracle_ctypes as O
from helpers import local_maxwellian, rel_err, setup

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nv,order", [(4, 2), (6, 1), (7, 2), (8, 2), (9, 2), (10, 1), (11, 2)])
def test_step_with_limiters_matches_oracle(nv, order):
    print(f"[rows] cavity3d 7 Nv {nv} order {order}", flush=True)
    case, cl, ocl, *_ = setup("cavity3d", 7, nv, order=order)
    rng = np.random.default_rng(nv)
    # rough enough that some reconstructions go negative and some densities
    # leave their neighbours' range
    cl.g *= rng.uniform(0.02, 2.0, cl.g.shape) * rng.uniform(0.3, 1.0, (cl.N, 1))
    dt = 0.5 * (1e-6 / 6) / 1303.0
    sol = A.Solver(cl, precision=A.PREC_FP64)
    st = O.State(ocl, cl.g, cl.mom)
    fired = 0
    for _ in range(2):
        stats = sol.step(dt, stats=True)
        O.step(ocl, st, dt, case.tau, case.R, cl.cfg.radius, order)
        mom, lim = sol.moments(with_limflag=True)
        assert np.array_equal(lim, st.limflag)
        fired |= (1 if stats["n_positivity"] else 0) | (2 if stats["n_nad"] else 0)
        assert rel_err(sol.g(), st.g) < 1e-10
        for c in range(5):
            assert rel_err(mom[:, c], st.mom[:, c], floor=1e-300) < 1e-10, c
    assert fired == 3


@pytest.mark.parametrize("n,extra", [((6, 6, 6), 0), ((16, 16, 32), -1), ((16, 16, 32), 0),
                                     ((16, 16, 32), 1), ((16, 32, 32), -1), ((16, 32, 32), 0),
                                     ((16, 32, 32), 1), ((24, 24, 24), 0)])
def test_mass_over_many_particles(n, extra):
    """N below, at and above multiples of the sum's 8 x 1024 particles (extra: an
    interior particle less, or one more)."""
    case = A.configure("cavity3d", nx=n[0], nv=3, mls_order=1)
    dx = 1e-6 / (n[0] - 1)
    case.raw.ny, case.raw.nz = n[1], n[2]
    case.raw.dom[2], case.raw.dom[4] = dx * (n[1] - 1), dx * (n[2] - 1)
    cl = A.build_lattice(case, precision=A.PREC_FP64, mls_order=1)
    cl.g, cl.mom = local_maxwellian(cl, case)
    p = np.nonzero(cl.boundary == 0)[0][7]
    q = np.arange(cl.N)
    q = np.delete(q, p) if extra < 0 else np.concatenate([q, np.full(extra, p)])
    for k in ("x", "y", "z", "boundary", "wall", "mom", "g"):
        setattr(cl, k, np.ascontiguousarray(getattr(cl, k)[q]))
    if extra > 0:
        cl.x[-1] += 0.4 * dx
    assert cl.N == n[0] * n[1] * n[2] + extra
    sol = A.Solver(cl, precision=A.PREC_FP64)
    dv = (cl.cfg.vmax - cl.cfg.vmin) / 2
    want = cl.g.sum() * dv ** 3
    assert abs(sol.total_mass() - want) <= 1e-13 * want
    st = sol.step(0.5 * dx / 1303.0, stats=True)
    assert abs(st["mass_old"] - want) <= 1e-13 * want
    assert abs(sol.total_mass() - want) <= 1e-13 * want


@pytest.mark.parametrize("name,nx,nv", [("cavity3d", 10, 6), ("cavity3d", 10, 11),
                                        ("cavity2d", 16, 8), ("cavity2d", 16, 18)])
def test_particles_without_mass_and_walls_that_emit_nothing(name, nx, nv):
    """A hole where g is zero and the moments are not: its particles keep their
    moments, whose Maxwellian the mass rescale after the transport must not
    scale. A wall faster than the velocity grid: density 1, not rescaled either."""
    print(f"[rows] without mass: {name} {nx} Nv {nv}", flush=True)
    case, cl, _, neigh, nn = setup(name, nx, nv, order=1)
    dx = 1e-6 / (nx - 1)
    d3 = cl.cfg.dim == 3
    cl.g *= np.random.default_rng(2).uniform(0.5, 1.5, cl.g.shape)
    c0 = 0.5e-6
    r2 = (cl.x - c0) ** 2 + (cl.y - c0) ** 2 + ((cl.z - c0) ** 2 if d3 else 0.0)
    cl.g[r2 < (3.9 * dx) ** 2] = 0.0
    hole = np.nonzero(r2 < (1.2 * dx) ** 2)[0]
    assert len(hole) and all((cl.g[neigh[i, :nn[i]]] == 0.0).all() for i in hole)
    wall = np.nonzero(cl.boundary)[0]
    w = wall[len(wall) // 2]
    cl.wall[w, 3:6] = 3.0 * cl.cfg.vmax * cl.wall[w, :3]
    ocl = O.Cloud(cl.cfg.dim, nv, cl.cfg.vmin, (cl.cfg.vmax - cl.cfg.vmin) / (nv - 1), cl.x, cl.y,
                  cl.z, cl.boundary, cl.wall, neigh, nn)
    dt = 0.3 * dx / 1303.0
    sol = A.Solver(cl, precision=A.PREC_FP64)
    st = O.State(ocl, cl.g, cl.mom)
    for k in range(2):
        stats = sol.step(dt, stats=True)
        O.step(ocl, st, dt, case.tau, case.R, cl.cfg.radius, 1)
        # the rescale that must not reach them is far from 1
        assert k or abs(stats["mass_old"] / stats["mass_after_transport"] - 1.0) > 1e-6
        mom, lim = sol.moments(with_limflag=True)
        g = sol.g()
        scale = np.abs(st.g).max(axis=1)
        assert scale[hole].min() > 0.0
        assert np.array_equal(lim, st.limflag)
        assert (np.abs(g - st.g).max(axis=1) / scale)[hole].max() < 1e-10
        assert rel_err(g, st.g) < 1e-10
        assert st.mom[w, 0] == 1.0 and mom[w, 0] == 1.0
        for c in range(5):
            assert rel_err(mom[:, c], st.mom[:, c], floor=1e-300) < 1e-10, c


@pytest.mark.parametrize("value", [np.inf, -np.inf, np.nan])
@pytest.mark.parametrize("name,nx,nv,order,p,k", [
    ("cavity3d", 8, 5, 1, 470, 23), ("cavity3d", 8, 5, 2, 231, 4), ("cavity3d", 8, 11, 1, 470, 23),
    ("cavity3d", 8, 5, 1, 267, 8), ("cavity2d", 12, 6, 2, 5, 21), ("cavity2d", 12, 18, 1, 63, 9)])
def test_moments_of_rows_that_are_not_finite(name, nx, nv, order, p, k, value):
    """One value that is not finite, five steps: g is infinite, and not a number,
    where the oracle's is; the moments are finite where its are, and equal there. (From a wall, whose
    density then leaves the limiter no bounds, rows with an infinite mass spread.)"""
    print(f"[rows] not finite: {name} {nx} Nv {nv} order {order} {p} {k} {value}", flush=True)
    case, cl, ocl, *_ = setup(name, nx, nv, order=order)
    cl.g *= np.random.default_rng(5).uniform(0.6, 1.4, cl.g.shape)
    cl.g[p, k] = value
    dt = 0.3 * (1e-6 / (nx - 1)) / 1303.0
    sol = A.Solver(cl, precision=A.PREC_FP64)
    st = O.State(ocl, cl.g, cl.mom)
    for _ in range(5):
        sol.step(dt)
        O.step(ocl, st, dt, case.tau, case.R, cl.cfg.radius, order)
        mom, g = sol.moments(), sol.g()
        assert np.array_equal(np.isfinite(mom), np.isfinite(st.mom))
        assert np.array_equal(np.isnan(g), np.isnan(st.g))
        assert np.array_equal(g == np.inf, st.g == np.inf)
        ok = np.isfinite(st.mom)
        for c in range(5):
            assert rel_err(mom[ok[:, c], c], st.mom[ok[:, c], c], floor=1e-300) < 1e-10, c

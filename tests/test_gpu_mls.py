"""The FP64 formulation's MLS transport where its stencils are not the
lattice's (jittered, degenerate, values that are not finite) and with and
without the step statistics.

Tolerances: transport 1e-12 of each particle's largest |g| (a 10 x 10 solve in
FP64 in another order of sums, on stencils as well conditioned as a lattice's);
everything else exact or stated at the assertion.
"""
from __future__ import annotations

import numpy as np
import pytest

import alebgk4paper_amd as A
import oracle_ctypes as O
from helpers import geom_of, local_maxwellian, setup

pytestmark = pytest.mark.gpu


def _oracle_cloud(cl, neigh, nn):
    return O.Cloud(cl.cfg.dim, cl.cfg.nv, cl.cfg.vmin,
                   (cl.cfg.vmax - cl.cfg.vmin) / (cl.cfg.nv - 1), cl.x, cl.y, cl.z, cl.boundary,
                   cl.wall, neigh, nn)


def _jittered(name, nx, nv, order, amp=0.15):
    case, cl, *_ = setup(name, nx, nv, order=order)
    rng = np.random.default_rng(5)
    dx = 1e-6 / (nx - 1)
    inner = cl.boundary == 0
    for k in ("x", "y", "z")[:cl.cfg.dim]:
        getattr(cl, k)[inner] += amp * dx * rng.uniform(-1, 1, int(inner.sum()))
    neigh, nn, _ = O.neighbours(geom_of(cl.cfg, case), cl.x, cl.y, cl.z)
    return case, cl, _oracle_cloud(cl, neigh, nn), 0.5 * dx / 1303.0


@pytest.mark.parametrize("name,nx,nv,order", [("cavity3d", 9, 4, 2), ("cavity3d", 8, 7, 1),
                                              ("cavity2d", 12, 7, 2), ("cavity2d", 12, 17, 1)])
def test_transport_on_a_jittered_cloud(name, nx, nv, order):
    print(f"[mls] jittered {name} {nx} Nv {nv} order {order}", flush=True)
    case, cl, ocl, dt = _jittered(name, nx, nv, order)
    sol = A.Solver(cl, precision=A.PREC_FP64)
    sol.transport_only(dt)
    want = O.transport(ocl, cl.g, dt, cl.cfg.radius, order)
    scale = np.abs(cl.g).max(axis=1, keepdims=True)
    assert (np.abs(sol.gt() - want) / scale).max() < 1e-12


@pytest.mark.parametrize("nx,nv,amp", [(9, 5, 0.0), (9, 5, 0.15), (13, 7, 0.0)])
def test_step_statistics_match_oracle_and_change_nothing(nx, nv, amp):
    """Flags and overshoots of the transport with stats; the same state, bit
    for bit, without them."""
    case, cl, ocl, dt = _jittered("cavity3d", nx, nv, 2, amp)
    _, fl, ov = O.transport(ocl, cl.g, dt, cl.cfg.radius, 2, flags=True)
    a, b = A.Solver(cl, precision=A.PREC_FP64), A.Solver(cl, precision=A.PREC_FP64)
    st = a.step(dt, stats=True)
    b.step(dt)
    assert np.array_equal(a.g(), b.g())
    assert st["n_mls_degenerate"] == int((fl & 1).astype(bool).sum())
    assert st["n_mls_extrapolate"] == int((fl & 2).astype(bool).sum())
    # an excess is a difference of values: rounding of the larger one, 1e-12 of it
    assert abs(st["mls_ovr_sum"] - ov.sum()) <= 1e-12 * np.abs(cl.g).sum() + 1e-9 * ov.sum()


@pytest.mark.parametrize("name,nx,nv", [("cavity3d", 9, 5), ("cavity3d", 13, 7), ("cavity2d", 9, 5)])
def test_values_outside_the_support_do_not_enter(name, nx, nv):
    """A neighbour that is not finite reaches exactly the nodes whose foot
    point has it in its support, as in the oracle."""
    case, cl, ocl, dt = _jittered(name, nx, nv, 2, 0.0)
    p = cl.N // 2
    cl.g[p] = np.nan
    cl.g[p + 1] = np.inf
    want = O.transport(ocl, cl.g, dt, cl.cfg.radius, 2)
    sol = A.Solver(cl, precision=A.PREC_FP64)
    sol.transport_only(dt)
    got = sol.gt()
    assert np.array_equal(np.isfinite(got), np.isfinite(want))
    ok = np.isfinite(want)
    assert np.abs(got[ok] - want[ok]).max() < 1e-12 * np.abs(cl.g[np.isfinite(cl.g)]).max()


@pytest.mark.parametrize("order", [1, 2])
def test_collinear_stencils_2d(order):
    """Rows of particles out of each other's reach: every stencil is a line
    and A is singular. The nodes that do not leave the line (v_y = 0) have exact
    zeros in A, which the pivoted elimination skips; there the result is the
    oracle's where the line determines its own terms. The others divide rounding by rounding in the reference too."""
    case, cl, *_ = setup("cavity2d", 9, 5, order=order)
    cl.y = np.ascontiguousarray(cl.y * 4.0)
    neigh, nn, _ = O.neighbours(geom_of(cl.cfg, case), cl.x, cl.y, cl.z)
    # neighbours of the same row only, whatever the voxels did with the rows
    N = cl.N
    neigh = np.full((N, A.MAX_NEIGH), 0, np.int32)
    nn = np.zeros(N, np.int32)
    for i in range(N):
        j = [q for q in range(i - i % 9, i - i % 9 + 9)
             if q != i and abs(cl.x[q] - cl.x[i]) < cl.cfg.radius]
        neigh[i, :len(j)], nn[i] = j, len(j)
    cl.neigh, cl.nneigh = neigh, nn
    dt = 0.5 * (1e-6 / 8) / 1303.0
    want = O.transport(_oracle_cloud(cl, neigh, nn), cl.g, dt, cl.cfg.radius, order)
    sol = A.Solver(cl, precision=A.PREC_FP64)
    sol.transport_only(dt)
    got = sol.gt()
    v = A.velocities(cl.cfg)
    # ... and the line itself must determine 1, x, x^2: three neighbours in the
    # support, with room to its edge
    on = np.zeros((N, 25), bool)
    for i in range(N):
        for k in np.nonzero(v[:, 1] == 0.0)[0]:
            d = np.abs(cl.x[neigh[i, :nn[i]]] - (cl.x[i] - v[k, 0] * dt))
            on[i, k] = (d < 0.9 * cl.cfg.radius).sum() >= 3
    on = np.tile(on, 2)
    assert on.sum() > 100
    # elimination of a matrix whose other rows are zero: 1e-11 of the largest value
    scale = np.abs(cl.g).max(axis=1, keepdims=True)
    assert (np.abs(got - want) / scale)[on].max() < 1e-11


# ---- stencils shared by congruent particles --------------------------------------

def _variant(kind, nx, nv, order):
    """A lattice cloud altered so that some, all or no particles share stencils."""
    case, cl, *_ = setup("cavity3d", nx, nv, order=order)
    rng = np.random.default_rng(11)
    dx = 1e-6 / (nx - 1)
    inner = np.nonzero(cl.boundary == 0)[0]
    if kind == "few":                       # a few particles off the lattice
        for p in rng.choice(inner, 5, replace=False):
            cl.x[p] += 0.2 * dx * rng.uniform(-1, 1)
            cl.z[p] += 0.2 * dx * rng.uniform(-1, 1)
    elif kind == "tiny":                    # displaced by less than a lattice check would see
        cl.y[inner[::3]] += 1e-9 * dx
    elif kind == "permuted":                # no two neighbours in row order
        q = rng.permutation(cl.N)
        for k in ("x", "y", "z", "boundary", "wall", "mom", "g"):
            setattr(cl, k, np.ascontiguousarray(getattr(cl, k)[q]))
    elif kind == "holes":                   # particles missing, as inside a body
        keep = np.ones(cl.N, bool)
        keep[rng.choice(inner, 12, replace=False)] = False
        for k in ("x", "y", "z", "boundary", "wall", "mom", "g"):
            setattr(cl, k, np.ascontiguousarray(getattr(cl, k)[keep]))
    elif kind == "twice":                   # two particles at one site
        q = np.concatenate([np.arange(cl.N), inner[40:42]])
        for k in ("x", "y", "z", "boundary", "wall", "mom", "g"):
            setattr(cl, k, np.ascontiguousarray(getattr(cl, k)[q]))
    elif kind == "mesh":                    # particles with a mesh velocity, zero mostly
        cl.mesh = np.zeros((cl.N, 3))
        cl.mesh[inner[10:30]] = (30.0, -20.0, 10.0)
    elif kind == "lid":                     # a wall velocity that varies along the lid
        lid = np.nonzero(np.abs(cl.z - case.dom[4]) < 1e-13)[0]
        cl.wall[lid, 3] = 1e6 * cl.x[lid]
    neigh, nn, _ = O.neighbours(geom_of(cl.cfg, case), cl.x, cl.y, cl.z)
    ocl = _oracle_cloud(cl, neigh, nn) if cl.mesh is None else \
        O.Cloud(3, nv, cl.cfg.vmin, (cl.cfg.vmax - cl.cfg.vmin) / (nv - 1), cl.x, cl.y, cl.z,
                cl.boundary, cl.wall, neigh, nn, cl.mesh)
    return case, cl, ocl, 0.5 * dx / 1303.0


@pytest.mark.parametrize("kind,nx,nv,order", [
    ("lattice", 13, 7, 2), ("lattice", 18, 7, 1), ("lattice", 7, 15, 2), ("lattice", 10, 5, 2),
    ("few", 13, 7, 2), ("tiny", 13, 7, 2), ("permuted", 13, 7, 2), ("holes", 14, 7, 2),
    ("twice", 13, 7, 2), ("mesh", 13, 7, 2), ("lid", 13, 7, 2)])
def test_shared_stencils_match_oracle(kind, nx, nv, order):
    """All but 10^3 / Nv 5 are above the 500,000 values from which stencils are
    shared."""
    print(f"[mls] shared stencils {kind} {nx} Nv {nv} order {order}", flush=True)
    case, cl, ocl, dt = _variant(kind, nx, nv, order)
    sol = A.Solver(cl, precision=A.PREC_FP64)
    sol.transport_only(dt)
    want = O.transport(ocl, cl.g, dt, cl.cfg.radius, order)
    scale = np.abs(cl.g).max(axis=1, keepdims=True)
    assert (np.abs(sol.gt() - want) / scale).max() < 1e-12


def test_stencils_follow_the_cloud():
    """After a transport, particles move and gain a mesh velocity
    (ab_set_wall_state); the next transport, eager and as a replay of a graph
    captured before, sees them."""
    case, cl, ocl, dt = _variant("lattice", 13, 7, 2)
    sols = [A.Solver(cl, precision=A.PREC_FP64) for _ in range(3)]
    graph = A.Graph([sols[1]], dt, 1)
    for s in sols[:2]:
        s.transport_only(dt)
    inner = np.nonzero(cl.boundary == 0)[0]
    p = inner[100:110]
    rng = np.random.default_rng(2)
    xyz = np.stack([cl.x, cl.y, cl.z], 1)[p] + 0.1 * 1e-7 * rng.uniform(-1, 1, (len(p), 3))
    mv = np.tile([5.0, -7.0, 3.0], (len(p), 1))
    for s in sols:
        s.set_wall_state(p, xyz=xyz, mv=mv)
    sols[0].step(dt)
    graph.launch()
    graph.synchronize()
    sols[2].step(dt)
    assert np.array_equal(sols[0].g(), sols[2].g())
    assert np.array_equal(sols[1].g(), sols[2].g())
    graph.close()
    for k, a in enumerate((cl.x, cl.y, cl.z)):
        a[p] = xyz[:, k]
    cl.mesh = np.zeros((cl.N, 3))
    cl.mesh[p] = mv
    nb, nn = sols[0].neighbours()
    ocl = O.Cloud(3, 7, cl.cfg.vmin, (cl.cfg.vmax - cl.cfg.vmin) / 6, cl.x, cl.y, cl.z, cl.boundary,
                  cl.wall, nb, nn, cl.mesh)
    st = O.State(ocl, cl.g, cl.mom)
    O.step(ocl, st, dt, case.tau, case.R, cl.cfg.radius, 2)
    assert np.abs(sols[0].g() - st.g).max() < 1e-10 * np.abs(st.g).max()


def _ball_lists(n, reach, chebyshev=None):
    """Neighbour lists of an n[0] x n[1] x n[2] lattice: the sites nearer than
    reach spacings, or (chebyshev) at most that many lattice steps away per axis."""
    ix, iy, iz = (a.ravel() for a in np.meshgrid(*[np.arange(k) for k in n], indexing="ij"))
    at = np.empty(n, np.int64)
    p = ix + n[0] * (iy + n[1] * iz)
    at[ix, iy, iz] = p
    N = len(p)
    neigh, nn = np.zeros((N, A.MAX_NEIGH), np.int32), np.zeros(N, np.int32)
    m = int(np.ceil(reach)) if chebyshev is None else chebyshev
    for oz in range(-m, m + 1):
        for oy in range(-m, m + 1):
            for ox in range(-m, m + 1):
                if (ox, oy, oz) == (0, 0, 0) or \
                        (chebyshev is None and ox * ox + oy * oy + oz * oz >= reach * reach):
                    continue
                jx, jy, jz = ix + ox, iy + oy, iz + oz
                ok = (jx >= 0) & (jx < n[0]) & (jy >= 0) & (jy < n[1]) & (jz >= 0) & (jz < n[2])
                i = p[ok]
                neigh[i, nn[i]] = at[jx[ok], jy[ok], jz[ok]]
                nn[i] += 1
    return neigh, nn


def _against_oracle(cl, ocl, dt, order, tol=1e-12):
    """Transport (over a gt that held NaN), the step's statistics, and the step
    with and without them, from values so rough that many outputs leave their
    neighbours' range. tol: of each particle's largest |g|."""
    R = cl.cfg.radius
    cl.g = cl.g * np.random.default_rng(4).uniform(0.5, 1.5, cl.g.shape)
    want, fl, ov = O.transport(ocl, cl.g, dt, R, order, flags=True)
    sol, g = A.Solver(cl, precision=A.PREC_FP64), cl.g
    cl.g = np.full_like(g, np.nan)
    sol.upload(cl)
    sol.transport_only(dt)
    assert np.isnan(sol.gt()).all()
    cl.g = g
    sol.upload(cl)
    sol.transport_only(dt)
    scale = np.abs(g).max(axis=1, keepdims=True)
    err = np.abs(sol.gt() - want) / scale
    print(f"[mls] error {np.nanmax(err):.1e}", flush=True)
    assert not (err >= tol).any() and not np.isnan(err).any(), \
        f"{(~(err < tol)).sum()} of {err.size} outputs, largest {np.nanmax(err):.2e}"
    st = sol.step(dt, stats=True)
    other = A.Solver(cl, precision=A.PREC_FP64)
    other.step(dt)
    assert np.array_equal(sol.g(), other.g())
    assert st["n_mls_degenerate"] == int((fl & 1).astype(bool).sum())
    # every excess may be off by what its output may be
    dv3 = ((cl.cfg.vmax - cl.cfg.vmin) / (cl.cfg.nv - 1)) ** 3
    off = tol * scale.sum() * g.shape[1] * dv3
    assert off < 1e-3 * ov.sum()           # rows counted twice show
    assert abs(st["mls_ovr_sum"] - ov.sum()) <= off


# radius in lattice spacings, lists: sites nearer than this many spacings, or the
# 26 nearest. From sqrt(3) to 2 (and with the 26 nearest) every interior particle's
# stencil reaches one step to each side, so stencils of runs one above the other
# have fewer rows in common than at 2.5.
@pytest.mark.parametrize("nx,order,radius,lists", [
    (13, 2, 1.8, 1.8), (13, 2, 1.95, 1.95), (18, 1, 1.8, 1.8), (13, 2, 2.5, "26 nearest"),
    (18, 1, 2.5, "26 nearest"), (13, 2, 2.1, 2.1), (13, 2, 2.5, 2.5), (13, 2, 2.9, 2.9)])
def test_shared_stencils_of_other_reach(nx, order, radius, lists):
    print(f"[mls] shared stencils {nx} order {order} radius {radius} lists {lists}", flush=True)
    case, cl, *_ = setup("cavity3d", nx, 7, order=order)
    dx = 1e-6 / (nx - 1)
    cl.cfg.radius = radius * dx
    cl.neigh, cl.nneigh = _ball_lists((nx,) * 3, 0, 1) if lists == "26 nearest" else \
        _ball_lists((nx,) * 3, lists)
    _against_oracle(cl, _oracle_cloud(cl, cl.neigh, cl.nneigh), 0.3 * dx / 1303.0, order)


# first row y0 + frac spacings from the voxel grid's origin y0; the grid's own
# guess of the spacing off by eps (a lattice so long that its rows fall out of
# step with that guess by half a spacing)
@pytest.mark.parametrize("n,nv,order,y0,frac,eps", [
    ((13, 13, 13), 7, 2, -5e-7, 0.5, 0.0), ((13, 13, 13), 7, 2, 1e-7, 0.5, 0.0),
    ((13, 13, 13), 7, 2, 0.0, 0.5, 0.0), ((14, 15, 13), 7, 2, -5e-7, 0.5, 0.0),
    ((13, 14, 13), 7, 2, 3e-7, 1.5, 0.0), ((13, 13, 13), 7, 2, 0.0, 0.27, 0.0),
    ((18, 21, 17), 7, 1, -5e-7, 0.5, 0.0), ((13, 13, 13), 7, 2, 0.0, 0.499, 1e-4),
    ((7, 1100, 7), 4, 1, 0.0, 0.0, 4.8e-4)])
def test_shared_stencils_off_the_voxel_origin(n, nv, order, y0, frac, eps):
    print(f"[mls] shared stencils {n} Nv {nv} from {y0} + {frac} spacings, off {eps}", flush=True)
    case = A.configure("cavity3d", nx=n[0], nv=nv, mls_order=order)
    dx = 1e-6 / (n[0] - 1)
    case.raw.ny, case.raw.nz = n[1], n[2]
    case.raw.dom[2], case.raw.dom[4] = dx * (n[1] - 1), dx * (n[2] - 1)
    cl = A.build_lattice(case, precision=A.PREC_FP64, mls_order=order)
    cl.g, cl.mom = local_maxwellian(cl, case)
    row = np.rint((cl.y - cl.y.min()) / dx)
    cl.y = y0 + (row + frac) * dx
    cl.cfg.ybottom = y0
    cl.cfg.vbox *= 1.0 + eps
    cl.neigh, cl.nneigh = _ball_lists(n, 2.5)
    _against_oracle(cl, _oracle_cloud(cl, cl.neigh, cl.nneigh), 0.5 * dx / 1303.0, order)


def test_shared_stencils_follow_a_relayout():
    """A hole that fills (more particles than the class arrays had room for),
    then one that opens (fewer): each step is, bit for bit, that of a fresh
    upload of the cloud it starts from."""
    nx, nv = 16, 7
    case, cl, *_ = setup("cavity3d", nx, nv)
    dx = 1e-6 / (nx - 1)
    c0 = np.array([0.51e-6, 0.49e-6, 0.5e-6])
    pos = np.stack([cl.x, cl.y, cl.z], 1)
    keep = (cl.boundary == 1) | (((pos - c0) ** 2).sum(1) > (4.6 * dx) ** 2)
    k = np.arange(12) + 0.5
    zk, ph = 1.0 - 2.0 * k / 12, k * np.pi * (3.0 - np.sqrt(5.0))
    nrm = np.stack([np.sqrt(1 - zk * zk) * np.cos(ph), np.sqrt(1 - zk * zk) * np.sin(ph), zk], 1)
    surf = c0 + 0.7 * dx * nrm
    wall = np.zeros((12, 7))
    wall[:, :3], wall[:, 6] = nrm, case.Tw
    p = int(np.argmax(cl.boundary == 0))
    cat = lambda a, b: np.ascontiguousarray(np.concatenate([a[keep], b]))
    cloud = A.Cloud(cl.cfg, cat(cl.x, surf[:, 0]), cat(cl.y, surf[:, 1]), cat(cl.z, surf[:, 2]),
                    cat(cl.boundary, np.ones(12, np.uint8)), cat(cl.wall, wall),
                    cat(cl.mom, np.tile(cl.mom[p], (12, 1))), cat(cl.g, np.tile(cl.g[p], (12, 1))))
    dt = 0.3 * dx / 1303.0
    dom = (0.0, 1e-6) * 3
    sol = A.Solver(cloud, precision=A.PREC_FP64)
    ids = np.concatenate([np.full(int(keep.sum()), -1, np.int32), np.zeros(12, np.int32)])
    n0 = sol.N
    sizes = []
    for size in (None, 0.7, 3.1, 2.5):
        if size is not None:
            _, counts = sol.cloud_manage([A.body(A.BODY_SPHERE, c0, size * dx)], ids, dx, 0.3 * dx, dom)
            ids = sol.body_ids()
            sizes.append((sol.N, tuple(counts)))
        q, mom = sol.particles(), sol.moments()
        now = A.Cloud(cl.cfg, q["x"], q["y"], q["z"], q["boundary"], q["wall"], mom, sol.g())
        now.neigh, now.nneigh = sol.neighbours()
        sol.step(dt)
        other = A.Solver(now, precision=A.PREC_FP64)
        other.step(dt)
        assert np.array_equal(sol.g(), other.g())
        assert np.array_equal(sol.moments(), other.moments())
    print(f"[mls] relayout {n0} -> {sizes}", flush=True)
    assert sizes[0][0] > n0 + n0 // 16 and sizes[1][0] < sizes[0][0]

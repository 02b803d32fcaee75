"""GPU: the moving-body block where its parts can go wrong: a surface list
longer than the scratch starts with and spread over several list blocks, a step
after which the cloud management has particles to remove, merge or refill, and
body ids without a body.

The body is given so much mass that its motion is nil, so the block must leave
what its parts leave when called one by one on a twin cloud: the loads of
ab_body_loads (the same sums in the same order), and the cloud of
ab_cloud_manage. The surface positions pass through c + (x - c): a rounding of
2^-52 of the box (1e-6 m), 1e-14 of dx, which the refill's inverse-distance
weights see squared; hence 1e-11 for its values.
"""
from __future__ import annotations

import ctypes as C

import numpy as np
import pytest

import alebgk4paper_amd as A

pytestmark = pytest.mark.gpu


def _make(case, nx, walls):
    cs = A.configure(case, nx=nx, nv=4, mls_order=2)
    cl = A.build_case(cs, mls_order=2)
    if walls:
        cl.body_id = np.where(cl.boundary == 1, 0, cl.body_id).astype(np.int32)
    rng = np.random.default_rng(3)
    cl.g = np.ascontiguousarray(cl.g * (1.0 + 0.3 * rng.uniform(-1, 1, size=cl.g.shape)))
    return cs, cl, A.Solver(cl, precision=A.PREC_FP64)


def _still(cl, size=1.0):
    b = cl.bodies[0]
    b.mass = 1e300
    b.vel[:] = [0.0] * 3
    b.om[:] = [0.0] * 3
    b.angular_vel = 0.0
    b.size *= size
    return b


# walls: the box walls belong to the body too; size: of the body's record (a
# larger body swallows particles); pitch: of the lattice that the management is
# told, in dx (a finer one leaves sites to refill); mind: merging distance in dx
CASES = [("cavity3d-cube", 12, False, 1.0, 1.0, 0.0), ("cavity3d-cube", 12, True, 1.0, 1.0, 0.0),
         ("cavity3d-cube", 12, False, 1.6, 1.0, 0.0), ("cavity3d-cube", 12, True, 1.0, 1.0, 1.05),
         ("cavity2d-circle", 24, False, 3.0, 1.0, 0.0),
         ("cavity2d-circle", 24, False, 1.0, 0.5, 0.0), ("cavity2d-circle", 40, True, 1.0, 1.0, 1.05)]


@pytest.mark.parametrize("case,nx,walls,size,pitch,mind", CASES)
def test_block_leaves_what_its_parts_leave(case, nx, walls, size, pitch, mind):
    cs, cl, sol = _make(case, nx, walls)
    _, _, twin = _make(case, nx, walls)
    b = _still(cl, size)
    surf = np.nonzero((cl.boundary == 1) & (cl.body_id >= 0))[0].astype(np.int32)
    assert not walls or sol.dim == 2 or len(surf) > 512
    area = 6.0 * b.size * b.size / b.npts if sol.dim == 3 else 2.0 * np.pi * b.size / b.npts
    want = twin.body_loads(surf, np.zeros(len(surf), np.int32), [b.c[:]], [area])[0]
    dx = pitch * cl.geo[0]
    min_dist = mind * cl.geo[0] if mind else 0.5 * dx
    dom = A.box(cs)
    loads, counts = sol.body_step(cs.dt, [b], dx, min_dist, dom)
    print(f"[body block] {case} {nx} size {size} pitch {pitch} min {mind}: {len(surf)} on the "
          f"surface, {counts}", flush=True)
    # (the area's two spellings may round apart)
    assert np.abs(loads[0, :6] - want).max() <= 2.0 ** -52 * np.abs(want).max()
    ab = A.body(b.shape, b.c[:], b.size, o=b.o[:], rm=b.rm[:])
    src, wcounts = twin.cloud_manage([ab], cl.body_id, dx, min_dist, dom)
    assert counts == tuple(wcounts)
    assert any(counts) == (size != 1.0 or pitch != 1.0 or mind != 0.0)
    assert sol.N == twin.N
    assert np.array_equal(sol.body_ids(), twin.body_ids())
    p, q = sol.particles(), twin.particles()
    for k in ("x", "y", "z"):
        assert np.abs(p[k] - q[k]).max() <= 4 * 2.0 ** -52 * 1e-6, k
    ga, gb = sol.g(), twin.g()
    kept = src >= 0
    assert np.array_equal(ga[kept], gb[kept])
    assert np.abs(ga[~kept] - gb[~kept]).max(initial=0.0) <= 1e-11 * np.abs(gb).max()
    # the lists are those of the cloud it leaves
    lists = [np.array(a) for a in sol.neighbours()]
    sol.rebuild_neighbours()
    for s, t in zip(lists, sol.neighbours()):
        assert np.array_equal(s, t)


def test_body_ids_without_a_body_are_refused():
    """Ids past the bodies given (and past the most there can be): refused, and
    the cloud and the body are as they were."""
    cs, cl, _ = _make("cavity2d-circle", 24, False)
    cl.body_id = np.where(cl.body_id >= 0, 700, cl.body_id).astype(np.int32)
    sol = A.Solver(cl, precision=A.PREC_FP64)
    x0 = sol.particles()["x"].copy()
    n = int(((cl.boundary == 1) & (cl.body_id >= 0)).sum())
    with pytest.raises(A.ALEBGKError, match=f"{n} surface particles carry a body id"):
        sol.body_step(cs.dt, cl.bodies, cl.geo[0], cl.geo[3], A.box(cs))
    assert np.array_equal(sol.particles()["x"], x0)


def test_tasks_that_share_bodies_follow_one_another():
    """Two tasks on one body array: the second starts from the bodies the first
    leaves, as two calls do."""
    made = [_make("cavity2d-circle", 24, False) for _ in range(4)]
    cs, cl, _ = made[0]
    one = (A.ABRigidBody * 1)(cl.bodies[0])
    two = (A.ABRigidBody * 1)(cl.bodies[0])
    lib, d6 = A.hip_lib(), (C.c_double * 6)(*A.box(cs))
    n, cnt = C.c_int(), (C.c_int * 3)()
    for m in made[:2]:
        assert lib.ab_body_step(m[2]._ctx, C.c_double(cs.dt), 1, one, C.c_double(cl.geo[0]),
                                C.c_double(cl.geo[3]), d6, None, C.byref(n), cnt) == 0
    tasks = (A.ABBodyTask * 2)()
    for t in tasks:
        t.dt, t.nbodies, t.dx, t.min_dist = cs.dt, 1, cl.geo[0], cl.geo[3]
        t.bodies = C.cast(two, C.POINTER(A.ABRigidBody))
        t.dom[:] = list(A.box(cs))
    ctxs = (C.c_void_p * 2)(*[m[2]._ctx.value for m in made[2:]])
    assert lib.ab_body_step_many(2, ctxs, tasks) == 0
    assert bytes(one) == bytes(two)
    for a, b in zip(made[:2], made[2:]):
        assert np.array_equal(a[2].g(), b[2].g())
        assert np.array_equal(a[2].particles()["x"], b[2].particles()["x"])

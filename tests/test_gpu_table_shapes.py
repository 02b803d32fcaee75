"""Transport launch shapes of the tables on lattices that their blocks do not
tile: the last block of a row overlaps the one before it, and the planes are
cut into items of four and more.

Tolerance: 1e-6 (FP32) and 1e-13 (FP64) of the largest |g| against single
columns: the same 81 products per value in another order, two steps.
"""
from __future__ import annotations

import numpy as np
import pytest

import alebgk4paper_amd as A
from helpers import local_maxwellian

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("prec,tol", [(A.PREC_MIXED, 1e-6), (A.PREC_FP64_TABLE, 1e-13)])
@pytest.mark.parametrize("n,nv", [((13, 13, 13), 5), ((11, 9, 13), 4), ((10, 8, 7), 6),
                                  ((7, 12, 9), 5), ((8, 15, 6), 4), ((23, 10, 5), 4),
                                  ((6, 6, 12), 4), ((9, 8, 11), 9), ((14, 14, 14), 8),
                                  ((8, 9, 40), 5)])
def test_block_shapes_on_ragged_lattices(n, nv, prec, tol):
    print(f"[shapes] lattice {n} Nv {nv} precision {prec}", flush=True)
    case = A.configure("cavity3d", nx=n[0], nv=nv, mls_order=2)
    dx = 1e-6 / (n[0] - 1)
    case.raw.ny, case.raw.nz = n[1], n[2]
    case.raw.dom[2], case.raw.dom[4] = dx * (n[1] - 1), dx * (n[2] - 1)
    cl = A.build_lattice(case, precision=prec, mls_order=2)
    cl.g, cl.mom = local_maxwellian(cl, case)
    dt = 0.4 * dx / 1303.0
    base = A.Solver(cl, precision=prec)
    table, _ = base.autotune(dt, reps=1)
    base.set_transport_shape(0)
    base.steps(dt, 2)
    ref = base.g()
    for i, name, _ in table + [(-1, "default", 0.0)]:
        s = A.Solver(cl, precision=prec)
        s.set_transport_shape(i)
        s.steps(dt, 2)
        assert np.abs(s.g() - ref).max() <= tol * np.abs(ref).max(), name
        s.close()


@pytest.mark.parametrize("n", [(5, 12, 11), (9, 5, 12), (13, 13, 12)])
def test_single_column_shapes_keep_their_indices(n):
    """FP64 shapes 0 to 3 are single columns in z blocks of 9, 8, 7 and 6, on any
    lattice, and agree bit for bit."""
    case = A.configure("cavity3d", nx=n[0], nv=4, mls_order=2)
    dx = 1e-6 / (n[0] - 1)
    case.raw.ny, case.raw.nz = n[1], n[2]
    case.raw.dom[2], case.raw.dom[4] = dx * (n[1] - 1), dx * (n[2] - 1)
    cl = A.build_lattice(case, precision=A.PREC_FP64_TABLE, mls_order=2)
    cl.g, cl.mom = local_maxwellian(cl, case)
    sol = A.Solver(cl, precision=A.PREC_FP64_TABLE)
    names = {i: name for i, name, _ in sol.autotune(0.4 * dx / 1303.0, reps=1)[0]}
    assert [names[i] for i in range(4)] == ["K9/W2", "K8/W2", "K7/W2", "K6/W2"]
    ref = None
    for i in range(4):
        s = A.Solver(cl, precision=A.PREC_FP64_TABLE)
        s.set_transport_shape(i)
        s.steps(0.4 * dx / 1303.0, 2)
        ref = s.g() if ref is None else ref
        assert np.array_equal(s.g(), ref), names[i]

"""The 3-D table step's row passes (boundary and interior lists in one launch,
Newton solves and boundary list in one launch) and its two-launch mass sums, on
lattices whose lists end inside a block and whose particles end inside a
reduction range, against the FP64 formulation of the same step.

Tolerance: 1e-10 relative on g and the moments, the FP64 tables' against the
oracle (the two paths sum the same stencils in another order).
"""
from __future__ import annotations

import numpy as np
import pytest

import alebgk4paper_amd as A
from helpers import rel_err, setup

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("collision", [A.COLLISION_CONTINUOUS, A.COLLISION_DISCRETE])
@pytest.mark.parametrize("nx,nv", [(5, 6), (6, 5), (7, 6), (9, 4)])
def test_small_lattices_match_the_fp64_formulation(nx, nv, collision):
    print(f"[table rows] cavity3d {nx} Nv {nv} collision {collision}", flush=True)
    case, cl, *_ = setup("cavity3d", nx, nv, order=1)
    rng = np.random.default_rng(nx)
    cl.g *= rng.uniform(0.95, 1.05, cl.g.shape)
    dt = 0.5 * (1e-6 / (nx - 1)) / 1303.0
    a = A.Solver(cl, precision=A.PREC_FP64, collision=collision)
    b = A.Solver(cl, precision=A.PREC_FP64_TABLE, collision=collision)
    for _ in range(3):
        sa, sb = a.step(dt, stats=True), b.step(dt, stats=True)
        assert abs(sa["mass_old"] - sb["mass_old"]) <= 1e-12 * sa["mass_old"]
    assert abs(a.total_mass() - b.total_mass()) <= 1e-12 * a.total_mass()
    assert rel_err(b.g(), a.g()) < 1e-10
    ma, mb = a.moments(), b.moments()
    for c in range(5):
        assert rel_err(mb[:, c], ma[:, c], floor=1e-300) < 1e-10, c

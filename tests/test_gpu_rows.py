"""The 3-D FP64 step's fused positivity, NAD, commit, wall and collision at the
row lengths where its variants change (rows of 4, 8 and 16 values a lane in
registers, longer rows read again), with both limiters firing, and the mass
sums around the lengths of their unrolled loop.

Tolerances: 1e-10 relative on g and the moments (the FP64 step's); limiter
flags identical.
"""
from __future__ import annotations

import numpy as np
import pytest

import alebgk4paper_amd as A
import oracle_ctypes as O
from helpers import rel_err, setup

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


@pytest.mark.parametrize("nx", [6, 20, 21, 24])
def test_mass_over_many_particles(nx):
    """N below, at and above multiples of the sum's 8 x 1024 particles."""
    case, cl, *_ = setup("cavity3d", nx, 3, order=1)
    sol = A.Solver(cl, precision=A.PREC_FP64)
    dv = (cl.cfg.vmax - cl.cfg.vmin) / 2
    want = cl.g.sum() * dv ** 3
    assert abs(sol.total_mass() - want) <= 1e-13 * want
    st = sol.step(0.5 * (1e-6 / (nx - 1)) / 1303.0, stats=True)
    assert abs(st["mass_old"] - want) <= 1e-13 * want
    assert abs(sol.total_mass() - want) <= 1e-13 * want

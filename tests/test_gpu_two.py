"""Two stencil stages of a level in one pass (psb_two.h) against one kernel per
stage (a context created with PSB_NO_TWO set).  The values are the same bit for
bit; the rho partials are summed over other blocks, which moves rho by some
1e-16 of itself.  After two iterations that leaves FP64 solutions equal to well
under 1e-12; in the FP32 iterations alpha, beta and the K-cycle's factors can
round to the neighbouring float: 2^-24 of an update each, under 1e-6 in all.
Shapes: tiles with a remainder of rows, columns and planes, rows split along k,
more than 64 KB of LDS, coarsening in two directions, solid cells."""
import os

import numpy as np
import pytest

import psb

pytestmark = pytest.mark.gpu


def solver(shape, env, d):
    for name in env:
        os.environ[name] = "1"
    try:
        s = psb.Solver(*shape)
    finally:
        for name in env:
            os.environ.pop(name, None)
    if d["off"].any():
        s.set_active(d["off"])
    s.set_matrix(d)
    s.set_geometry(d["dxc"], d["dyc"], d["dzc"])
    return s


MIXED = dict(precision=psb.PSB_MIXED, inner_adapt=2, inner_rtol=1e-2)
SEMI = dict(stretch_z=2.0, lz=2.0, cylinder=True, cyl_d=0.2)


@pytest.mark.parametrize("shape, gen, stop, tail", [
    ((64, 64, 64), {}, dict(MIXED, ac_store=1, ac_kcycle=-1), True),
    ((64, 64, 64), {}, dict(MIXED, ac_store=0), True),
    ((64, 64, 64), {}, dict(ac_kcycle=-1), True),
    # FP16 operator, flexible beta without a K-cycle; sweeps of which one stage fuses
    ((40, 72, 48), {}, dict(MIXED, ac_store=2, ac_flexible=1), True),
    ((40, 72, 48), {}, dict(MIXED, ac_store=1, ac_pre=3, ac_post=1), True),
    ((40, 72, 48), {}, dict(ac_pre=1, ac_post=2), True),
    # few planes, rows and columns; every level through the passes
    ((16, 20, 24), {}, dict(MIXED, ac_store=1), False),
    ((20, 36, 40), {}, dict(ac_kcycle=2), False),
    ((36, 16, 16), {}, dict(), False),
    # FP64: rows of 192 vectors whole (68 KB of LDS), of 200 and 256 split
    ((16, 16, 384), {}, dict(), True),
    ((16, 20, 400), {}, dict(), True),
    ((20, 16, 512), {}, dict(ac_kcycle=2), True),
    # FP32: 200 vectors, split
    ((16, 20, 800), {}, dict(MIXED, ac_store=1), True),
    # x and y halved alone, solid cells
    ((32, 32, 128), SEMI, dict(MIXED, ac_store=1, ac_kcycle=-1, ac_coarsen=1, ac_cfac=1.0), False),
    ((32, 40, 64), SEMI, dict(ac_kcycle=2, ac_coarsen=1, ac_cfac=1.0), False),
    ((32, 32, 32), SEMI, dict(MIXED, ac_store=1), True),
])
def test_two_stages_in_one_pass(shape, gen, stop, tail):
    d = psb.generate(*shape, nsph=4, rmin=0.08, rmax=0.2, rho_in=1.0, rho_out=1000.0, seed_sph=3,
                     seed_vel=1003, **gen)
    n = int(np.prod(shape))
    kw = dict(precond=psb.PSB_PREC_AC, norm=psb.PSB_NORM_L2REL, res_rat=1e-8, res_tol=0.0, **stop)
    env = [] if tail else ["PSB_NO_TAIL"]
    two, one = solver(shape, env, d), solver(shape, env + ["PSB_NO_TWO"], d)
    x2, _ = two.solve(np.zeros(n), d["rhs"], max_iter=2, **kw)
    x1, _ = one.solve(np.zeros(n), d["rhs"], max_iter=2, **kw)
    mixed = "precision" in stop
    assert np.linalg.norm(x1) > 0
    assert np.linalg.norm(x2 - x1) <= (1e-6 if mixed else 1e-12) * np.linalg.norm(x1)
    _, r2 = two.solve(np.zeros(n), d["rhs"], max_iter=400, **kw)
    _, r1 = one.solve(np.zeros(n), d["rhs"], max_iter=400, **kw)
    assert r1["converged"] and r2["converged"]
    assert abs(r1["iterations"] - r2["iterations"]) <= 1

"""The two-stage passes where the size of the level decides on them, against one
kernel per stage (a context created with PSB_NO_TWO set).

As BiCGS's preconditioner the V-cycle forms no rho, so that nothing of a solve
depends on the passes' blocks: solutions, histories and counts are compared bit
for bit, on both sides of the line for levels of the marching sweeps and of the
span sweeps (one and two vectors a thread), with remainders of tiles and slabs,
rows split along k, semi-coarsening, solid cells, and a matrix (pure Neumann)
and one with a time term.

As CG's, the finest level's second sweep leaves the rho partials, which the pass
sums over other blocks: rho moves by some 1e-16 of itself, an FP64 solution after
two iterations by well under 1e-12; in the FP32 iterations alpha, beta and the
K-cycle's factors can round to the neighbouring float, 2^-24 of an update each,
under 1e-6 in all.  Shapes above the line, and which kernels ran: the profile
counts a launch of the first post-sweep alone below it and none above."""
import os

import numpy as np
import pytest

import psb

pytestmark = pytest.mark.gpu

MIXED = dict(precision=psb.PSB_MIXED, inner_adapt=2, inner_rtol=1e-2)
SEMI = dict(stretch_z=2.0, lz=2.0, cylinder=True, cyl_d=0.2)


def case(shape, gen, shift=1.0):
    d = psb.generate(*shape, nsph=4, rmin=0.08, rmax=0.2, rho_in=1.0, rho_out=1000.0, seed_sph=3,
                     seed_vel=1003, **gen)
    d["c"] = d["c"] * shift
    return d


def solver(shape, d, two):
    if not two:
        os.environ["PSB_NO_TWO"] = "1"
    try:
        s = psb.Solver(*shape)
    finally:
        os.environ.pop("PSB_NO_TWO", None)
    if d["off"].any():
        s.set_active(d["off"])
    s.set_matrix(d)
    s.set_geometry(d["dxc"], d["dyc"], d["dzc"])
    return s


@pytest.mark.parametrize("shape, gen, shift, stop", [
    ((64, 64, 64), {}, 1.0, dict(MIXED, ac_store=1)),
    ((40, 72, 96), {}, 1.0, dict(MIXED, ac_store=1)),
    ((40, 72, 96), {}, 1.0, dict(MIXED, ac_store=0, ac_kcycle=-1)),
    ((40, 72, 96), {}, 1.01, dict(ac_kcycle=-1)),
    ((48, 56, 112), {}, 1.0, dict()),
    ((20, 36, 400), {}, 1.0, dict()),
    ((20, 36, 800), {}, 1.0, dict(MIXED, ac_store=1)),
    ((48, 96, 80), SEMI, 1.0, dict(MIXED, ac_store=1, ac_coarsen=1, ac_cfac=1.0)),
    ((48, 96, 80), SEMI, 1.0, dict(ac_kcycle=-1, ac_coarsen=1, ac_cfac=1.0)),
    ((24, 24, 24), {}, 1.0, dict()),
])
def test_cycle_of_the_bicgs_is_bit_identical(shape, gen, shift, stop):
    d = case(shape, gen, shift)
    n = int(np.prod(shape))
    out = []
    for two in (True, False):
        s = solver(shape, d, two)
        x, r = s.solve(np.zeros(n), d["rhs"], method=psb.PSB_BICGS, precond=psb.PSB_PREC_AC,
                       norm=psb.PSB_NORM_L2REL, res_rat=1e-8, res_tol=0.0, max_iter=4, **stop)
        out.append((x, r, s.history()))
        s.close()
    (x2, r2, h2), (x1, r1, h1) = out
    assert np.linalg.norm(x1) > 0
    assert np.array_equal(x2, x1)
    assert np.array_equal(h2, h1)
    assert r2 == r1


@pytest.mark.parametrize("shape, gen, stop", [
    ((40, 72, 96), {}, dict(MIXED, ac_store=1, ac_kcycle=-1)),
    ((40, 72, 96), {}, dict(ac_kcycle=-1)),
    ((40, 72, 96), {}, dict(MIXED, ac_store=2, ac_flexible=1)),
    ((36, 20, 400), {}, dict(ac_flexible=1, ac_kcycle=2)),
    ((16, 48, 384), {}, dict()),
    ((20, 36, 800), {}, dict(MIXED, ac_store=1)),
    ((48, 96, 80), SEMI, dict(MIXED, ac_store=1, ac_kcycle=-1, ac_coarsen=1, ac_cfac=1.0)),
    ((48, 96, 80), SEMI, dict(ac_kcycle=2, ac_coarsen=1, ac_cfac=1.0)),
])
def test_rho_of_the_pass(shape, gen, stop):
    d = case(shape, gen)
    n = int(np.prod(shape))
    kw = dict(precond=psb.PSB_PREC_AC, norm=psb.PSB_NORM_L2REL, res_rat=1e-8, res_tol=0.0, **stop)
    two, one = solver(shape, d, True), solver(shape, d, False)
    x2, _ = two.solve(np.zeros(n), d["rhs"], max_iter=2, **kw)
    x1, _ = one.solve(np.zeros(n), d["rhs"], max_iter=2, **kw)
    assert np.linalg.norm(x1) > 0
    assert (np.linalg.norm(x2 - x1) <=
            (1e-6 if "precision" in stop else 1e-12) * np.linalg.norm(x1))
    _, r2 = two.solve(np.zeros(n), d["rhs"], max_iter=400, **kw)
    _, r1 = one.solve(np.zeros(n), d["rhs"], max_iter=400, **kw)
    assert r1["converged"] and r2["converged"]
    assert abs(r1["iterations"] - r2["iterations"]) <= 1


@pytest.mark.parametrize("shape, one_pass", [((32, 32, 32), False), ((64, 64, 64), False),
                                             ((192, 32, 32), False), ((72, 64, 64), True),
                                             ((96, 96, 96), True)])
@pytest.mark.parametrize("stop", [dict(MIXED, ac_store=1), dict()])
def test_small_levels_keep_one_kernel_per_post_sweep(shape, one_pass, stop):
    d = case(shape, {})
    s = solver(shape, d, True)
    db, dx = psb.DeviceArray.from_host(d["rhs"]), psb.DeviceArray(int(np.prod(shape)))
    dx.zero()
    _, stats, _ = s.profile_solve_device(dx.addr, db.addr, precond=psb.PSB_PREC_AC,
                                         norm=psb.PSB_NORM_L2REL, res_rat=1e-8, res_tol=0.0,
                                         max_iter=4, **stop)
    assert stats["sweep_last"]["launches"] > 0
    assert (stats["sweep_prol"]["launches"] == 0) == one_pass

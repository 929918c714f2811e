"""The lowest smoothing level in one workgroup (psb_tail.h) against the same
cycle with one launch per phase (a context created with PSB_NO_TAIL set): the
same arithmetic and the same order of every sum, so the solutions are compared
bit for bit.  Shapes: the largest level that fits (1024 four-wide vectors, one
per thread), levels whose blocks are not full, rows that take scalar cells,
coarsening in one or two directions only, solid cells, and one level too large,
which keeps its launches."""
import os

import numpy as np
import pytest

import psb

pytestmark = pytest.mark.gpu


def solver(shape, tail, d):
    os.environ.pop("PSB_NO_TAIL", None)
    if not tail:
        os.environ["PSB_NO_TAIL"] = "1"
    try:
        s = psb.Solver(*shape)
    finally:
        os.environ.pop("PSB_NO_TAIL", None)
    if d["off"].any():
        s.set_active(d["off"])
    s.set_matrix(d)
    s.set_geometry(d["dxc"], d["dyc"], d["dzc"])
    return s


MIXED = dict(precision=psb.PSB_MIXED, inner_adapt=2, inner_rtol=1e-2)


@pytest.mark.parametrize("shape, gen, stop", [
    # FP32, lowest level 16^3 (1024 vectors), K-cycle on it and on 32^3
    ((64, 64, 64), {}, dict(MIXED, ac_store=1, ac_kcycle=-1)),
    ((64, 64, 64), {}, dict(MIXED, ac_store=0, ac_kcycle=-1)),
    # V-cycle; one and three sweeps
    ((64, 64, 64), {}, dict(MIXED, ac_store=1, ac_pre=1, ac_post=1)),
    ((64, 32, 64), {}, dict(MIXED, ac_store=1, ac_kcycle=4, ac_pre=3, ac_post=3)),
    # 20 x 18 x 22 and 9 x 20 x 16: blocks not full, scalar cells
    ((40, 36, 44), {}, dict(MIXED, ac_store=1, ac_kcycle=2)),
    ((18, 40, 64), {}, dict(MIXED, ac_store=1, ac_kcycle=4)),
    ((36, 20, 36), {}, dict(MIXED, ac_store=1, ac_kcycle=2)),
    # FP64: 10 x 10 x 20 (1000 vectors), 9^3 (scalar), 16^3 (too large)
    ((40, 40, 80), {}, dict(ac_kcycle=4)),
    ((36, 36, 36), {}, dict(ac_kcycle=2)),
    ((64, 64, 64), {}, dict(ac_kcycle=-1)),
    # z halved alone at the end, solid cells
    ((32, 32, 128), dict(stretch_z=2.0, lz=2.0, cylinder=True, cyl_d=0.2),
     dict(MIXED, ac_store=1, ac_kcycle=-1, ac_coarsen=1, ac_cfac=1.0)),
    ((32, 32, 64), dict(stretch_z=2.0, lz=2.0, cylinder=True, cyl_d=0.3),
     dict(ac_kcycle=4, ac_coarsen=1, ac_cfac=1.0)),
])
def test_lowest_level_in_one_workgroup_is_bit_identical(shape, gen, stop):
    d = psb.generate(*shape, nsph=4, rmin=0.08, rmax=0.2, rho_in=1.0, rho_out=1000.0, seed_sph=3,
                     seed_vel=1003, **gen)
    n = int(np.prod(shape))
    kw = dict(precond=psb.PSB_PREC_AC, norm=psb.PSB_NORM_L2REL, res_rat=1e-8, res_tol=0.0,
              max_iter=300, **stop)
    out = []
    for tail in (True, False):
        x, r = solver(shape, tail, d).solve(np.zeros(n), d["rhs"], **kw)
        out.append((x, r["iterations"], r["rel_l2"]))
    assert out[0][1] == out[1][1] and out[0][2] == out[1][2]
    assert np.array_equal(out[0][0], out[1][0])

"""The folded scalar steps of CG-di on both sides of their line, which the blocks
of the two kernels set (88 x 76 x 76 folds, 96 x 64 x 64 does not), and in the
reference's cycle, which folds up to 2^20 two-wide cells whatever the blocks: its
finest level with tiles and slabs that leave a remainder, odd numbers of
iterations, solves whose last step nobody asks for (V, F, W) and solves whose
verdict is read (flex), scalar cells.  Against one launch per step (a context
created with PSB_NO_FOLD set): the same sums in the same order, so everything is
compared bit for bit.  (Grids from 2^19 cells of tests/test_gpu_fold*.py run
unfolded on both sides outside the cycle.)"""
import os

import numpy as np
import pytest

import psb

pytestmark = pytest.mark.gpu


def solver(shape, fold, d):
    if not fold:
        os.environ["PSB_NO_FOLD"] = "1"
    try:
        s = psb.Solver(*shape)
    finally:
        os.environ.pop("PSB_NO_FOLD", None)
    s.set_matrix(d)
    s.set_geometry(d["dxc"], d["dyc"], d["dzc"])
    return s


def case(shape):
    return psb.generate(*shape, nsph=3, rmin=0.08, rmax=0.2, rho_in=1.0, rho_out=100.0,
                        seed_sph=3, seed_vel=1003)


@pytest.mark.parametrize("shape", [(88, 76, 76), (80, 80, 80), (96, 64, 64), (97, 72, 72),
                                   (1400, 16, 16)])
def test_folded_cg_at_the_line_of_its_blocks(shape):
    d = case(shape)
    out = []
    for fold in (True, False):
        s = solver(shape, fold, d)
        x, r = s.solve(np.zeros(int(np.prod(shape))), d["rhs"], max_iter=24, res_rat=1e-8)
        out.append((x, r, s.history()))
        s.close()
    (x1, r1, h1), (x0, r0, h0) = out
    assert r1 == r0
    assert np.array_equal(h1, h0)
    assert np.array_equal(x1, x0)


@pytest.mark.parametrize("shape, cyc", [
    ((95, 90, 110), dict(loop="V")),
    ((95, 90, 110), dict(loop="V", max_iter=(3, 5, 7))),
    ((95, 90, 110), dict(loop="flex", max_iter=(15, 25, 15), smooth_res_rat=0.9, max_visits=30)),
    ((128, 88, 92), dict(loop="V", init="V", max_iter=(1, 2, 3), smooth_res_rat=1e-12)),
    ((128, 128, 64), dict(loop="F", max_iter=(5, 40, 5))),
    ((45, 45, 45), dict(loop="W", max_iter=(4, 9, 3))),
    ((45, 45, 45), dict(loop="flex", smooth_res_rat=0.5, max_stale=(2, 2, 2), max_visits=30)),
    ((75, 65, 45), dict(loop="V")),
])
def test_folded_cycle_is_bit_identical(shape, cyc):
    d = case(shape)
    out = []
    for fold in (True, False):
        s = solver(shape, fold, d)
        x, r = s.ac_vcycle(np.zeros(int(np.prod(shape))), d["rhs"], max_cycles=2,
                           stop_if_div=0, **cyc)
        out.append((x, r))
        s.close()
    (x1, r1), (x0, r0) = out
    assert np.linalg.norm(x0) > 0
    assert r1 == r0
    assert np.array_equal(x1, x0)

"""Device memory a context holds after a solve: the AC cycle's levels keep the
fifth vector of their CG only where the folded steps read it, and the dense
operator of the coarsest level keeps none of the arrays it was formed in.
Compared with a context that does without (PSB_NO_FOLD, PSB_NO_DENSE set); the
runtime hands memory out in pieces of up to 2 MB."""
import ctypes
import os

import numpy as np
import pytest

import psb

pytestmark = pytest.mark.gpu

PIECE = 4 << 20


def held(shape, env, run):
    """Device memory that a context holds after run(solver, rhs)."""
    d = psb.generate(*shape, nsph=2, rmin=0.1, rmax=0.2, rho_in=1.0, rho_out=100.0, seed_sph=3,
                     seed_vel=1003)

    def free():
        a, b = ctypes.c_size_t(), ctypes.c_size_t()
        assert psb.hip().hipMemGetInfo(ctypes.byref(a), ctypes.byref(b)) == 0
        return a.value

    if env:
        os.environ[env] = "1"
    try:
        before = free()
        s = psb.Solver(*shape)
    finally:
        os.environ.pop(env or "", None)
    s.set_matrix(d)
    s.set_geometry(d["dxc"], d["dyc"], d["dzc"])
    run(s, d["rhs"])
    used = before - free()
    s.close()
    return used


def cycle(s, b):
    s.ac_vcycle(np.zeros(b.size), b, max_cycles=1)


def solve(s, b):
    s.solve(np.zeros(b.size), b, precond=psb.PSB_PREC_AC, max_iter=4)


@pytest.mark.parametrize("shape, folds", [((128, 128, 128), False), ((96, 96, 96), True)])
def test_cycle_keeps_the_fifth_vector_where_it_folds(shape, folds):
    held(shape, None, cycle)  # (the library's own first allocations)
    extra = held(shape, None, cycle) - held(shape, "PSB_NO_FOLD", cycle)
    vector = 8 * int(np.prod(shape))
    below = 2 * vector // 8  # the coarser levels' vectors, which fold on both
    if folds:
        assert extra >= vector - PIECE
    assert extra <= (vector if folds else 0) + below + PIECE


@pytest.mark.parametrize("shape", [(48, 48, 48), (64, 64, 64), (128, 128, 128)])
def test_dense_operator_keeps_no_scratch(shape):
    held(shape, None, solve)
    assert held(shape, None, solve) <= held(shape, "PSB_NO_DENSE", solve) + PIECE

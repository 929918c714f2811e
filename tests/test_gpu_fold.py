"""CG-di with the scalar steps folded into the streaming kernels (k_cg_pq_di,
k_cg_xr_di) against one launch per step (a context created with PSB_NO_FOLD
set): the same sums in the same order, so solutions, residual histories and
counts are compared bit for bit.  Shapes: scalar cells, one partly filled
block, spans of more than one vector per thread, marching tiles of one and
several planes, the largest grid that folds; symmetric and 7-array matrices;
every way a solve can end."""
import os

import numpy as np
import pytest

import psb

pytestmark = pytest.mark.gpu


def solver(shape, fold, d):
    os.environ.pop("PSB_NO_FOLD", None)
    if not fold:
        os.environ["PSB_NO_FOLD"] = "1"
    try:
        s = psb.Solver(*shape)
    finally:
        os.environ.pop("PSB_NO_FOLD", None)
    s.set_matrix(d)
    s.set_geometry(d["dxc"], d["dyc"], d["dzc"])
    return s


def both(shape, d, **kw):
    out = []
    for fold in (True, False):
        s = solver(shape, fold, d)
        x, r = s.solve(np.zeros(int(np.prod(shape))), d["rhs"], **kw)
        out.append((x, r, s.history()))
        s.close()
    (x1, r1, h1), (x0, r0, h0) = out
    assert r1 == r0, (r1, r0)
    assert np.array_equal(h1, h0)
    assert np.array_equal(x1, x0)
    return r1


@pytest.mark.parametrize("shape", [(4, 3, 5), (9, 7, 11), (57, 45, 39), (16, 16, 16),
                                   (32, 32, 32), (33, 40, 50), (64, 64, 64), (96, 96, 96),
                                   (128, 64, 128)])
def test_folded_cg_is_bit_identical(shape):
    d = psb.generate(*shape, nsph=3, rmin=0.08, rmax=0.2, rho_in=1.0, rho_out=100.0, seed_sph=3,
                     seed_vel=1003)
    both(shape, d, max_iter=60, res_rat=1e-8)


@pytest.mark.parametrize("stop", [
    dict(max_iter=300, res_rat=1e-6),                 # converges on the ratio
    dict(max_iter=300, res_rat=0.0, res_tol=1e-9),    # ... on the tolerance
    dict(max_iter=7, res_rat=1e-12),                  # runs out of iterations
    dict(max_iter=1, res_rat=1e-12),
    dict(max_iter=300, min_iter=9, res_rat=0.5),      # MinIter holds it back
    dict(max_iter=300, res_rat=1e-300, res_tol=0.0, stalecount=3),  # stalls
    dict(max_iter=300, res_rat=1e-8, norm=1, graph_chunk=2),
    dict(max_iter=300, res_tol=1e300),                # returns at once
])
def test_folded_cg_ends_alike(stop):
    shape = (24, 20, 18)
    d = psb.generate(*shape, nsph=2, rmin=0.1, rmax=0.2, rho_in=1.0, rho_out=10.0, seed_sph=5,
                     seed_vel=1005)
    both(shape, d, **stop)


def test_folded_cg_on_seven_arrays():
    shape = (17, 14, 12)
    d = psb.generate(*shape, nsph=2, rmin=0.1, rmax=0.2, rho_in=1.0, rho_out=10.0, seed_sph=5,
                     seed_vel=1005)
    rng = np.random.default_rng(1)
    for k in "ent":
        d[k] = d[k] * rng.uniform(1.0, 1.05, d[k].size)
    d["c"] = d["c"] * 1.2
    both(shape, d, max_iter=30, res_rat=1e-8)

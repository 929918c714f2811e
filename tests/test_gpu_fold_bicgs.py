"""BiCGS with the scalar steps folded into the streaming kernels (k_bi1, k_bi2,
k_bi3) against one launch per step (a context created with PSB_NO_FOLD set):
the same sums in the same order, so solutions, residual histories and counts
are compared bit for bit.  Shapes: scalar cells, one partly filled block, spans
of more than one vector per thread, the largest grid that folds and one that
does not; symmetric and 7-array matrices; the ways a solve can end."""
import os

import numpy as np
import pytest

import psb

pytestmark = pytest.mark.gpu


def both(shape, d, **kw):
    out = []
    for fold in (True, False):
        os.environ.pop("PSB_NO_FOLD", None)
        if not fold:
            os.environ["PSB_NO_FOLD"] = "1"
        try:
            s = psb.Solver(*shape)
        finally:
            os.environ.pop("PSB_NO_FOLD", None)
        s.set_matrix(d)
        s.set_geometry(d["dxc"], d["dyc"], d["dzc"])
        x, r = s.solve(np.zeros(int(np.prod(shape))), d["rhs"], method=psb.PSB_BICGS, **kw)
        out.append((x, r, s.history()))
        s.close()
    (x1, r1, h1), (x0, r0, h0) = out
    assert r1 == r0, (r1, r0)
    assert np.array_equal(h1, h0)
    assert np.array_equal(x1, x0)


def case(shape, seven=False):
    d = psb.generate(*shape, nsph=3, rmin=0.08, rmax=0.2, rho_in=1.0, rho_out=100.0, seed_sph=3,
                     seed_vel=1003)
    if seven:
        rng = np.random.default_rng(1)
        for k in "ent":
            d[k] = d[k] * rng.uniform(1.0, 1.05, d[k].size)
        d["c"] = d["c"] * 1.2
    return d


@pytest.mark.parametrize("shape, seven", [
    ((4, 3, 5), False), ((9, 7, 11), False), ((16, 16, 16), True), ((17, 14, 12), True),
    ((65, 48, 80), False), ((96, 96, 96), True), ((128, 64, 128), False), ((128, 66, 128), False)])
def test_folded_bicgs_is_bit_identical(shape, seven):
    both(shape, case(shape, seven), max_iter=40, res_rat=1e-8)


@pytest.mark.parametrize("stop", [
    dict(max_iter=300, res_rat=1e-6),                 # converges on the ratio
    dict(max_iter=300, res_rat=0.0, res_tol=1e-9),    # on the tolerance, a small s, a breakdown
    dict(max_iter=300, res_rat=0.0, res_tol=1e-4),
    dict(max_iter=7, res_rat=1e-12),                  # runs out of iterations
    dict(max_iter=1, res_rat=1e-12),
    dict(max_iter=300, min_iter=9, res_rat=0.5),      # MinIter holds it back
    dict(max_iter=300, res_rat=1e-300, res_tol=0.0, stalecount=3),  # stalls
    dict(max_iter=300, res_rat=1e-8, norm=1, graph_chunk=2),
    dict(max_iter=300, res_tol=1e300),                # returns at once
])
def test_folded_bicgs_ends_alike(stop):
    shape = (24, 20, 18)
    both(shape, case(shape, True), **stop)

"""The coarsest level's dense operator formed on the device (psb_dense.h)
against the host's (a context created with PSB_NO_DENSE set): the same
operations in the same order, every sum included, so solutions and counts are
compared bit for bit.  Shapes of the coarsest level: full and odd, the widest
band that fits the LDS (195 of 9 x 13 x 15) and one too wide (225), which stays
on the host; solid cells; a non-singular matrix."""
import os

import numpy as np
import pytest

import psb

pytestmark = pytest.mark.gpu
SEMI = dict(stretch_z=2.0, lz=2.0, cylinder=True, cyl_d=0.3)


@pytest.mark.parametrize("shape, gen, shift, stop", [
    ((32, 32, 32), {}, 1.0, {}),
    ((24, 24, 24), {}, 1.0, {}),
    ((22, 18, 20), {}, 1.0, {}),
    ((18, 26, 30), {}, 1.0, {}),
    ((16, 30, 30), {}, 1.0, {}),
    ((36, 16, 16), {}, 1.02, {}),
    ((32, 24, 32), SEMI, 1.0, {}),
    ((40, 32, 64), SEMI, 1.0, dict(ac_coarsen=1, ac_cfac=1.0)),
])
def test_dense_operator_on_the_device(shape, gen, shift, stop):
    d = psb.generate(*shape, nsph=4, rmin=0.08, rmax=0.2, rho_in=1.0, rho_out=1000.0, seed_sph=3,
                     seed_vel=1003, **gen)
    d["c"] = d["c"] * shift
    n = int(np.prod(shape))
    kw = dict(precond=psb.PSB_PREC_AC, norm=psb.PSB_NORM_L2REL, res_rat=1e-8, res_tol=0.0, **stop)
    out = []
    for env in ((), ("PSB_NO_DENSE",)):
        for e in env:
            os.environ[e] = "1"
        try:
            s = psb.Solver(*shape)
        finally:
            for e in env:
                os.environ.pop(e, None)
        if d["off"].any():
            s.set_active(d["off"])
        s.set_matrix(d)
        s.set_geometry(d["dxc"], d["dyc"], d["dzc"])
        x, _ = s.solve(np.zeros(n), d["rhs"], max_iter=2, **kw)
        _, r = s.solve(np.zeros(n), d["rhs"], max_iter=400, **kw)
        assert r["converged"]
        out.append((x, r))
    (x1, r1), (x0, r0) = out
    assert np.linalg.norm(x0) > 0
    assert np.array_equal(x1, x0)
    assert r1 == r0

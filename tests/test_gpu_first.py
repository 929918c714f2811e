"""The first sweep formed in the pass of the second and the restriction (the
finest level, 2^22 cells and more) against one kernel per stage (a context
created with PSB_NO_TWO set), at the smallest grid that takes it and one with
remainders of tiles and slabs; one sweep and three, which do not take it, too.
Values are the same bit for bit but for the sums of rho (see test_gpu_two.py):
after two iterations FP64 solutions agree to 1e-12, those of the FP32
iterations to 1e-6."""
import os

import numpy as np
import pytest

import psb

pytestmark = pytest.mark.gpu

MIXED = dict(precision=psb.PSB_MIXED, inner_adapt=2, inner_rtol=1e-2)


@pytest.mark.parametrize("shape, stop", [
    ((256, 128, 128), dict(MIXED, ac_store=1, ac_kcycle=-1)),
    ((160, 168, 160), dict(MIXED, ac_store=0)),
    ((160, 168, 160), dict(ac_kcycle=-1)),
    ((128, 128, 256), dict(MIXED, ac_store=1, ac_pre=3)),
    ((128, 128, 256), dict(ac_pre=1)),
])
def test_first_sweep_in_the_pass(shape, stop):
    d = psb.generate(*shape, nsph=4, rmin=0.05, rmax=0.1, rho_in=1.0, rho_out=1000.0, seed_sph=3,
                     seed_vel=1003)
    n = int(np.prod(shape))
    kw = dict(precond=psb.PSB_PREC_AC, norm=psb.PSB_NORM_L2REL, res_rat=1e-8, res_tol=0.0, **stop)
    out = []
    for env in (False, True):
        if env:
            os.environ["PSB_NO_TWO"] = "1"
        try:
            s = psb.Solver(*shape)
        finally:
            os.environ.pop("PSB_NO_TWO", None)
        s.set_matrix(d)
        s.set_geometry(d["dxc"], d["dyc"], d["dzc"])
        out.append(s.solve(np.zeros(n), d["rhs"], max_iter=2, **kw)[0])
        s.close()
    assert np.linalg.norm(out[1]) > 0
    assert (np.linalg.norm(out[0] - out[1]) <=
            (1e-6 if "precision" in stop else 1e-12) * np.linalg.norm(out[1]))

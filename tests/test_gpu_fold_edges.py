"""The folded scalar steps at the largest grids that take them and just past
them (cg_di_fold and BiCGS's line), against one launch per step: bit for bit."""
import os

import numpy as np
import pytest

import psb

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape, method", [
    ((64, 64, 128), psb.PSB_CG), ((66, 64, 128), psb.PSB_CG),
    ((64, 33, 61), psb.PSB_CG), ((64, 35, 61), psb.PSB_CG),
    ((96, 64, 128), psb.PSB_BICGS), ((97, 64, 128), psb.PSB_BICGS),
    ((96, 64, 63), psb.PSB_BICGS), ((96, 66, 65), psb.PSB_BICGS)])
def test_folded_steps_at_the_line(shape, method):
    d = psb.generate(*shape, nsph=3, rmin=0.08, rmax=0.2, rho_in=1.0, rho_out=100.0, seed_sph=3,
                     seed_vel=1003)
    out = []
    for env in (False, True):
        if env:
            os.environ["PSB_NO_FOLD"] = "1"
        try:
            s = psb.Solver(*shape)
        finally:
            os.environ.pop("PSB_NO_FOLD", None)
        s.set_matrix(d)
        s.set_geometry(d["dxc"], d["dyc"], d["dzc"])
        out.append(s.solve(np.zeros(int(np.prod(shape))), d["rhs"], method=method, max_iter=24,
                           res_rat=1e-8))
        s.close()
    assert out[0][1] == out[1][1]
    assert np.array_equal(out[0][0], out[1][0])

"""psb_stop.ac_fuse: 1 runs the FP32 post-sweeps in one pass on every level whose
shape allows it, 0 only on those where it is faster (tests/test_gpu_two_line.py).
The profile of a 64^3 solve counts a launch of the first post-sweep alone with 0
and none with 1; a context that changes the setting between solves replays each
setting's own graph and gives what a context of its own gives, bit for bit."""
import numpy as np
import pytest

import psb

pytestmark = pytest.mark.gpu

MIXED = dict(precond=psb.PSB_PREC_AC, precision=psb.PSB_MIXED, inner_adapt=2, inner_rtol=1e-2,
             norm=psb.PSB_NORM_L2REL, res_rat=1e-9, res_tol=0.0, max_iter=100, ac_store=1)


def solver():
    n = 64
    d = psb.generate(n, n, n, 4, 0.05, 0.15, 1.0, 1000.0, 9, 1009)
    s = psb.Solver(n, n, n)
    s.set_matrix(d)
    s.set_geometry(d["dxc"], d["dyc"], d["dzc"])
    return s, d["rhs"]


@pytest.mark.parametrize("fuse", [0, 1])
def test_setting_chooses_the_kernels(fuse):
    s, b = solver()
    db, dx = psb.DeviceArray.from_host(b), psb.DeviceArray(b.size)
    dx.zero()
    _, stats, _ = s.profile_solve_device(dx.addr, db.addr, **dict(MIXED, ac_fuse=fuse))
    assert stats["sweep_last"]["launches"] > 0
    assert (stats["sweep_prol"]["launches"] == 0) == bool(fuse)


def test_settings_keep_their_own_graphs():
    alone = []
    for fuse in (0, 1):
        s, b = solver()
        alone.append(s.solve(np.zeros(b.size), b, ac_fuse=fuse, **MIXED))
        s.close()
    s, b = solver()
    for fuse in (0, 1, 0, 1):
        x, r = s.solve(np.zeros(b.size), b, ac_fuse=fuse, **MIXED)
        assert np.array_equal(x, alone[fuse][0])
        assert r == alone[fuse][1]

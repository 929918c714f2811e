"""The projection on planes smaller than a block and than a wave, where a block's
threads belong to several slabs and a slab ends inside it: against the oracle,
bit for bit, without and with solid cells (tests/test_gpu_project.py has the
wider planes)."""
import numpy as np
import pytest

import psb
import psb_oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape", [(300, 3, 5), (40000, 2, 2), (9000, 8, 9), (70, 17, 16),
                                   (2, 1, 3), (19, 300, 130)])
@pytest.mark.parametrize("solid", [False, True])
def test_projection_on_thin_planes(shape, solid):
    rng = np.random.default_rng(7)
    nx, ny, nz = shape
    met = []
    for n in shape:
        xc = np.cumsum(rng.uniform(0.5, 1.5, n + 2))
        d = np.concatenate([[1.0], np.diff(xc)])
        met.append((rng.uniform(0.5, 1.5, n), d[1:n + 1].copy(), np.diff(xc)[1:n + 1].copy()))
    rho = rng.uniform(1.0, 1000.0, (nx + 2, ny + 2, nz + 2))
    off = (rng.random(shape) < 0.2).astype(np.uint8) if solid else None
    p = rng.standard_normal(shape)
    u = rng.standard_normal((nx + 1, ny, nz))
    v = rng.standard_normal((nx, ny + 1, nz))
    w = rng.standard_normal((nx, ny, nz + 1))
    s = psb.Solver(nx, ny, nz)
    s.assemble_pressure(rho, *met, off=off)
    dr, dp, du, dv, dw = (psb.DeviceArray.from_host(a.ravel()) for a in (rho, p, u, v, w))
    s.project_device(dr.addr, dp.addr, du.addr, dv.addr, dw.addr, dt=0.37, mask=7)
    ref = O.project(*met, rho, p, u, v, w, dt=0.37, off=off, mask=7)
    for a, b in zip((du, dv, dw), ref):
        assert np.array_equal(a.download(), np.ravel(b))

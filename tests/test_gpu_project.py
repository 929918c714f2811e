"""Momentum::project's marching kernel against the oracle, bit for bit, where its
tiles and slabs can go wrong: planes of less and more than one block, a last
tile that is partly empty, one plane, slabs of one to sixteen planes with a
remainder, single rows and columns; with solid cells and each face mask."""
import numpy as np
import pytest

import psb
import psb_oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape", [(1, 16, 16), (5, 1, 9), (4, 9, 1), (33, 7, 11), (17, 16, 17),
                                   (129, 40, 33), (40, 150, 70)])
@pytest.mark.parametrize("mask, solid", [(7, False), (7, True), (1, True), (6, False)])
def test_projection_at_the_edges_of_its_tiles(shape, mask, solid):
    rng = np.random.default_rng(5)
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
    s.project_device(dr.addr, dp.addr, du.addr, dv.addr, dw.addr, dt=0.37, mask=mask)
    ref = O.project(*met, rho, p, u, v, w, dt=0.37, off=off, mask=mask)
    for a, b in zip((du, dv, dw), ref):
        assert np.array_equal(a.download(), np.ravel(b))

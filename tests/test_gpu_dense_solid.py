"""The coarsest level's dense operator formed on the device where solid cells
come first: the sum of the inverse's entries begins with whole rows of zeros.
Against the host's operator (a context created with PSB_NO_DENSE set), the same
operations in the same order, bit for bit; and a new matrix with solid cells in
the first half of the grid costs no more than twice one without (it took 3.7
times as long while the zeros were added one by one; now 1.0)."""
import os
import time

import numpy as np
import pytest

import psb

pytestmark = pytest.mark.gpu


def prepare(n, solid, dense):
    if not dense:
        os.environ["PSB_NO_DENSE"] = "1"
    try:
        s = psb.Solver(n, n, n)
    finally:
        os.environ.pop("PSB_NO_DENSE", None)
    off = np.zeros((n, n, n), np.uint8)
    off[:solid] = 1
    rng = np.random.default_rng(11)
    b = rng.standard_normal((n, n, n))
    b[:solid] = 0.0
    b[solid:] -= b[solid:].mean()
    met = [tuple(np.full(n, 1.0 / n) for _ in range(3)) for _ in range(3)]
    rho = rng.uniform(1.0, 10.0, (n + 2,) * 3)

    def matrix():
        s.assemble_pressure(rho, *met, off=off if solid else None)

    matrix()
    return s, b.ravel(), matrix


@pytest.mark.parametrize("n, solid", [(32, 16), (32, 3), (48, 24), (24, 20)])
def test_dense_operator_behind_solid_cells(n, solid):
    out = []
    for dense in (True, False):
        s, b, _ = prepare(n, solid, dense)
        out.append(s.solve(np.zeros(b.size), b, precond=psb.PSB_PREC_AC, max_iter=3, res_rat=1e-12))
        s.close()
    (x1, r1), (x0, r0) = out
    assert np.linalg.norm(x0) > 0
    assert np.array_equal(x1, x0)
    assert r1 == r0


def test_solid_cells_first_cost_no_more():
    ms = []
    for solid in (24, 0):
        s, b, matrix = prepare(48, solid, True)
        db, dx = psb.DeviceArray.from_host(b), psb.DeviceArray(b.size)
        ts = []
        for _ in range(6):
            matrix()
            dx.zero()
            t = time.perf_counter()
            s.solve_device(dx.addr, db.addr, precond=psb.PSB_PREC_AC, max_iter=2, res_rat=1e-12)
            ts.append(time.perf_counter() - t)
        ms.append(1e3 * float(np.median(ts[1:])))
        s.close()
    assert ms[0] <= 2.0 * ms[1], ms

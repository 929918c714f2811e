"""A batch's two-stage passes where the systems' tiles differ: long rows split
beside systems of short ones (rows of 48 to 200 vectors, a last piece that is
partly empty, more rows than a tile's), long rows alone, and tiles so unlike that
the level keeps one kernel per stage.  Against contexts created with PSB_NO_TWO
set; tolerances as in tests/test_gpu_two_batch.py: values are the same bit for
bit, dot products are summed over other blocks, after which alpha, beta and the
K-cycle's factors can round to the neighbouring float, 2^-24 of an update each,
under 1e-6 in all after two iterations."""
import os

import numpy as np
import pytest

import psb

pytestmark = pytest.mark.gpu


def batch(shapes, two):
    if not two:
        os.environ["PSB_NO_TWO"] = "1"
    try:
        B = psb.Batch(shapes)
    finally:
        os.environ.pop("PSB_NO_TWO", None)
    rhs = []
    for q, shape in enumerate(shapes):
        d = psb.generate(*shape, 1 + q % 4, 0.05, 0.15, 1.0, 1000.0, 11 + q, 1011 + q)
        B.systems[q].set_matrix(d)
        B.systems[q].set_geometry(d["dxc"], d["dyc"], d["dzc"])
        rhs.append(d["rhs"])
    return B, rhs


@pytest.mark.parametrize("shapes", [
    [(32, 32, 32), (16, 36, 192)],
    [(48, 48, 48), (16, 16, 400), (20, 28, 272)],
    [(12, 40, 800), (64, 24, 16)],
    [(20, 36, 256), (16, 16, 192)],
    [(256, 8, 8)] * 3 + [(8, 8, 256)],
])
def test_mixed_tiles(shapes):
    xs, its = [], []
    for two in (True, False):
        B, rhs = batch(shapes, two)
        x0 = [np.zeros(b.size) for b in rhs]
        xs.append(B.solve(x0, rhs, res_rat=1e-8, max_iter=2)[0])
        _, res, rc = B.solve(x0, rhs, res_rat=1e-8, max_iter=400)
        assert rc == psb.PSB_OK
        its.append([r["iterations"] for r in res])
        B.close()
    for x2, x1 in zip(*xs):
        assert np.linalg.norm(x1) > 0
        assert np.linalg.norm(x2 - x1) <= 1e-6 * np.linalg.norm(x1)
    assert all(abs(a - b) <= 1 for a, b in zip(*its)), its

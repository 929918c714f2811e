"""The two-stage passes over a batch (kb_pre_restrict, kb_post_two) against one
kernel per stage (contexts created with PSB_NO_TWO set).  The values are the
same bit for bit; dot products are summed over other blocks, after which alpha,
beta and the K-cycle's factors can round to the neighbouring float: 2^-24 of an
update each, under 1e-6 in all after two iterations.  Shapes: systems of
different depth together, tiles with a remainder of rows and planes, more rows
than one block's, rows split along k, semi-coarsened levels (which keep their
own kernels), one system alone, solid cells."""
import os

import numpy as np
import pytest

import psb

pytestmark = pytest.mark.gpu


def batch(shapes, two, solid):
    if not two:
        os.environ["PSB_NO_TWO"] = "1"
    try:
        B = psb.Batch(shapes)
    finally:
        os.environ.pop("PSB_NO_TWO", None)
    rhs = []
    for q, shape in enumerate(shapes):
        gen = dict(stretch_z=2.0, lz=2.0, cylinder=True, cyl_d=0.25) if solid else {}
        d = psb.generate(*shape, 1 + q % 4, 0.05, 0.15, 1.0, 1000.0, 11 + q, 1011 + q, **gen)
        if solid:
            B.systems[q].set_active(d["off"])
        B.systems[q].set_matrix(d)
        B.systems[q].set_geometry(d["dxc"], d["dyc"], d["dzc"])
        rhs.append(d["rhs"])
    return B, rhs


@pytest.mark.parametrize("shapes, solid, stop", [
    ([(32, 32, 32), (48, 32, 16), (16, 48, 32), (32, 16, 64), (24, 24, 24)], False, {}),
    ([(96, 64, 32), (40, 72, 48), (32, 128, 64)], False, dict(ac_kcycle=0, ac_flexible=0)),
    ([(36, 20, 80), (20, 36, 40)], False, dict(ac_pre=3)),
    ([(16, 16, 1024)], False, {}),
    ([(16, 16, 400), (64, 64, 64)], False, dict(ac_post=1)),
    ([(32, 32, 64), (40, 48, 32)], True, {}),
    ([(12, 32, 32)], False, dict(ac_post=3)),
])
def test_two_stage_passes_of_a_batch(shapes, solid, stop):
    xs = []
    its = []
    for two in (True, False):
        B, rhs = batch(shapes, two, solid)
        x0 = [np.zeros(b.size) for b in rhs]
        xs.append(B.solve(x0, rhs, res_rat=1e-8, max_iter=2, **stop)[0])
        _, res, rc = B.solve(x0, rhs, res_rat=1e-8, max_iter=400, **stop)
        assert rc == psb.PSB_OK
        its.append([r["iterations"] for r in res])
    for x2, x1 in zip(*xs):
        assert np.linalg.norm(x1) > 0
        assert np.linalg.norm(x2 - x1) <= 1e-6 * np.linalg.norm(x1)
    assert all(abs(a - b) <= 1 for a, b in zip(*its)), its

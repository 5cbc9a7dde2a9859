"""The CG step's early loads at their edges, through the C ABI: one-rings of 4 to 30 slots around the
4 and 8 a lane loads ahead, free vertices from a part of one slice to one past a block of 256, in
both precisions, against the oracle's direct solve."""
import numpy as np
import pytest

import meshgen
import mdarap
import oracle

pytestmark = pytest.mark.gpu

POS_TOL = {mdarap.PREC_FP64: 1e-7, mdarap.PREC_FP32_REFINE: 1e-5}


@pytest.fixture(scope="module")
def ctx():
    if mdarap.device_count() == 0:
        pytest.fail("no GPU visible: the HIP path cannot run")
    c = mdarap.Context(0)
    yield c
    c.close()


@pytest.mark.parametrize("rings,segs", [(4, 4), (6, 5), (10, 8), (10, 9), (18, 15), (18, 30)])
def test_pcg_edges(ctx, rings, segs):
    xyz, tri = meshgen.uv_sphere(rings, segs)
    held = 1 + (rings // 2) * segs + np.arange(segs, dtype=np.int32)  # one ring
    tgt = xyz[held] + np.where(xyz[held][:, :1] > 0, 0.1, 0.0) * np.array([0.0, 0.0, 1.0])
    ref = oracle.Arap(xyz, tri)
    ref.set_constraints(held, tgt)
    assert ref.deform(2)
    for prec, tol in POS_TOL.items():
        print("case: rings=%d segs=%d precision=%d" % (rings, segs, prec), flush=True)
        m = mdarap.Mesh(ctx, xyz, tri, mdarap.config(
            precision=prec, solver=mdarap.SOLVER_PCG, pcg_iters=400, refine_steps=2,
            pcg_tol=1e-12 if prec == mdarap.PREC_FP64 else 1e-7))
        m.set_constraints(held, tgt)
        assert m.deform(2)
        assert meshgen.relative_error(m.mesh, ref.mesh) < tol
        m.close()

"""Device factorization at the edges of its tiles, through the C ABI: pivot blocks of 1 to 260
columns around the panel (4), block (16) and tile (64) sizes of the sweeps, alone (amalgamation 1:
one supernode without off rows) and with off rows (the default amalgamation), in both precisions,
against the oracle."""
import numpy as np
import pytest

import meshgen
import mdarap
import oracle

pytestmark = pytest.mark.gpu

POS_TOL = {mdarap.PREC_FP64: 1e-9, mdarap.PREC_FP32_REFINE: 1e-5}


@pytest.fixture(scope="module")
def ctx():
    if mdarap.device_count() == 0:
        pytest.fail("no GPU visible: the HIP path cannot run")
    c = mdarap.Context(0)
    yield c
    c.close()


def _problem(nf):
    """A sphere with all but nf vertices held (the free ones around the equator's start)."""
    xyz, tri = meshgen.uv_sphere(16, 24)
    xyz = meshgen.radial_noise(xyz, 0.01, nf)
    order = np.argsort(np.abs(xyz[:, 2]), kind="stable")
    held = np.sort(order[nf:]).astype(np.int32)
    tgt = xyz[held] + np.where(xyz[held][:, 2:3] > 0, 0.2, 0.0) * np.array([1.0, 0.0, 1.0])
    return xyz, tri, held, tgt


@pytest.mark.parametrize("nf", [1, 3, 4, 5, 15, 16, 17, 31, 32, 33, 47, 49, 63, 64, 65, 79, 127, 128, 129, 191, 193, 260])
@pytest.mark.parametrize("ratio", [0.3, 1.0])
def test_factor_edges(ctx, nf, ratio):
    xyz, tri, held, tgt = _problem(nf)
    ref = oracle.Arap(xyz, tri)
    ref.set_constraints(held, tgt)
    assert ref.deform(3)
    for prec, tol in POS_TOL.items():
        print("case: nf=%d ratio=%g precision=%d" % (nf, ratio, prec), flush=True)
        m = mdarap.Mesh(ctx, xyz, tri, mdarap.config(precision=prec, amalg_ratio=ratio, subtree_budget=0))
        m.set_constraints(held, tgt)
        assert m.deform(3)
        assert m.stats()["nf"] == nf
        assert meshgen.relative_error(m.mesh, ref.mesh) < tol
        m.close()

"""Factor and sweep layouts, with the shapes that a case is about asserted from the mesh's statistics: every
sweep (level tiles, small and large bottom subtrees) without level pairs, on meshes whose whole system would
be one dense front with them; and the column limits of merged tops, 400 where the factor is redone with every
rest pose and 700 where it is kept, just below and just above."""
import os

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


@pytest.mark.parametrize("name", ["sphere_obj", "bar_obj", "uv_sphere"])
@pytest.mark.parametrize("budget", [0, 64, 256, 1024])
def test_sweeps_without_level_pairs(ctx, golden_dir, name, budget):
    with np.load(os.path.join(golden_dir, name + ".npz")) as z:
        g = {k: z[k] for k in z.files}
    for prec, tol in POS_TOL.items():
        print("case: %s budget=%d precision=%d" % (name, budget, prec), flush=True)
        m = mdarap.Mesh(ctx, g["xyz"], g["tri"], mdarap.config(precision=prec, subtree_budget=budget, level_pairs=False))
        m.set_constraints(g["con_idx"], g["con_xyz"])
        assert m.deform(int(g["iters"]))
        st = m.stats()
        assert st["supernodes"] > 8
        assert st["subtrees"] > 0 if budget else st["subtrees"] == 0 and st["levels"] > 1
        assert meshgen.relative_error(m.mesh, g["pos"]) < tol
        m.close()


# rings and segments of a UV sphere, free vertices (around the equator), and the widest front and the levels
# of a factor that is redone and of one that is kept
TOPS = [
    (72, 96, 3300, (399, 2), (399, 2)),  # the top levels have 399 columns, with the next 920
    (36, 48, 1468, (227, 2), (407, 1)),  # 227, with the next 407
    (72, 96, 2814, (276, 2), (700, 1)),  # 276, with the next 700
    (72, 96, 2817, (256, 2), (256, 2)),  # 256, with the next 704
]


@pytest.mark.parametrize("rings,segs,nf,redone,kept", TOPS)
def test_limits_of_merged_tops(ctx, rings, segs, nf, redone, kept):
    xyz, tri = meshgen.uv_sphere(rings, segs)
    xyz = meshgen.radial_noise(xyz, 0.01, nf)
    held = np.sort(np.argsort(np.abs(xyz[:, 2]), kind="stable")[nf:]).astype(np.int32)
    tgt = xyz[held] + np.where(xyz[held][:, 2:3] > 0, 0.2, 0.0) * np.array([1.0, 0.0, 1.0])
    ref = oracle.Arap(xyz, tri)
    ref.set_constraints(held, tgt)
    assert ref.deform(3)
    for rest, shape in ((mdarap.REST_REFERENCE, redone), (mdarap.REST_FIXED, kept)):
        for prec, tol in POS_TOL.items():
            print("case: nf=%d rest=%d precision=%d" % (nf, rest, prec), flush=True)
            m = mdarap.Mesh(ctx, xyz, tri, mdarap.config(precision=prec, rest_mode=rest))
            m.set_constraints(held, tgt)
            assert m.deform(3)
            st = m.stats()
            assert (st["max_sn_width"], st["levels"]) == shape
            assert meshgen.relative_error(m.mesh, ref.mesh) < tol
            m.close()

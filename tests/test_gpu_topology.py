"""The analysis' counted neighbour lists through the C ABI: cotan weights of meshes with repeated and
flipped faces (edges of more than two faces) and of one-rings below and above the 32 neighbours that
are searched linearly, equal to the oracle's."""
import numpy as np
import pytest

import meshgen
import mdarap
import oracle

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("segs", [3, 31, 32, 33, 70])
@pytest.mark.parametrize("extra", [0, 1, 40])
def test_cotan_of_irregular_faces(segs, extra):
    if mdarap.device_count() == 0:
        pytest.fail("no GPU visible: the HIP path cannot run")
    xyz, tri = meshgen.uv_sphere(6, segs)
    rng = np.random.default_rng(segs + extra)
    more = tri[rng.integers(0, len(tri), size=extra)]
    more[::2] = more[::2, ::-1]  # every other one flipped
    tri = rng.permutation(np.concatenate([tri, more])).astype(np.int32)
    print("case: segs=%d extra=%d" % (segs, extra), flush=True)
    ctx = mdarap.Context(0)
    m = mdarap.Mesh(ctx, xyz, tri, mdarap.config())
    assert m.deform(0)
    rp0, ci0, w0 = oracle.cotan_csr(xyz, tri)
    rp, ci, w = m.cotan()
    assert np.array_equal(rp, rp0) and np.array_equal(ci, ci0)
    np.testing.assert_allclose(w, w0, rtol=1e-12, atol=0)
    m.close()
    ctx.close()


@pytest.mark.parametrize("segs", [15, 16, 17, 24, 79, 80, 81, 150])
@pytest.mark.parametrize("poles", [1, 4, 5, 6])
def test_long_one_rings(segs, poles):
    """Three spheres whose poles have `segs` neighbours, `poles` of the six held (held vertices share one
    slice: at most four long rings in a slice are taken by the wavefront, more lane by lane)."""
    if mdarap.device_count() == 0:
        pytest.fail("no GPU visible: the HIP path cannot run")
    one, tri1 = meshgen.uv_sphere(5, segs)
    n = len(one)
    xyz = np.concatenate([one + np.array([3.0 * k, 0.0, 0.0]) for k in range(3)])
    tri = np.concatenate([tri1 + k * n for k in range(3)]).astype(np.int32)
    pole = np.array([0, n - 1, n, 2 * n - 1, 2 * n, 3 * n - 1])[:poles]
    side = np.concatenate([k * n + 1 + 2 * segs + np.arange(3) for k in range(3)])  # on each equator
    held = np.sort(np.concatenate([pole, side])).astype(np.int32)
    tgt = xyz[held] + np.where(np.isin(held, pole)[:, None], np.array([0.05, 0.0, 0.1]), 0.0)
    ref = oracle.Arap(xyz, tri)
    ref.set_constraints(held, tgt)
    assert ref.deform(3)
    ctx = mdarap.Context(0)
    for prec, tol in ((mdarap.PREC_FP64, 1e-9), (mdarap.PREC_FP32_REFINE, 1e-5)):
        print("case: segs=%d poles=%d precision=%d" % (segs, poles, prec), flush=True)
        m = mdarap.Mesh(ctx, xyz, tri, mdarap.config(precision=prec))
        m.set_constraints(held, tgt)
        assert m.deform(3)
        assert meshgen.relative_error(m.mesh, ref.mesh) < tol
        m.close()
    ctx.close()

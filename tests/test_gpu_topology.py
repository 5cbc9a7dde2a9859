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

"""The local step's rotation does not depend on the covariance's scale: the host build of its code over the
range of each precision, and scaled meshes on the device against the oracle."""
import numpy as np
import pytest

import meshgen
import mdarap
import oracle


def _polar(cov):
    """argmax tr(R cov) over rotations, by numpy's SVD."""
    u, _, vt = np.linalg.svd(cov)
    d = np.sign(np.linalg.det(vt.transpose(0, 2, 1) @ u.transpose(0, 2, 1)))
    v = vt.transpose(0, 2, 1).copy()
    v[:, :, 2] *= d[:, None]
    return v @ u.transpose(0, 2, 1)


def _matrix(q):
    x, y, z, w = q.T
    return np.stack([1 - 2 * (y * y + z * z), 2 * (x * y - w * z), 2 * (x * z + w * y),
                     2 * (x * y + w * z), 1 - 2 * (x * x + z * z), 2 * (y * z - w * x),
                     2 * (x * z - w * y), 2 * (y * z + w * x), 1 - 2 * (x * x + y * y)], 1).reshape(-1, 3, 3)


@pytest.mark.parametrize("fp64", [False, True])
def test_rotation_at_every_scale(fp64):
    """Powers of two over the normal range give bitwise the rotation at scale one (entries of one sign of
    magnitude within 1/16 .. 2, so none leaves the range), and that rotation is the polar factor's."""
    rng = np.random.default_rng(7)
    cov = rng.choice([-1.0, 1.0], (300, 3, 3)) * rng.uniform(0.0625, 2.0, (300, 3, 3))
    if not fp64:
        cov = cov.astype(np.float32).astype(np.float64)
    base, _ = mdarap.host_best_rotation(cov, fp64=fp64)
    s = np.linalg.svd(cov, compute_uv=False)
    sure = s[:, 1] + np.sign(np.linalg.det(cov)) * s[:, 2] > 0.05 * s[:, 0]  # (else nearly ambiguous)
    assert sure.sum() > 200
    err = np.abs(_matrix(base) - _polar(cov))[sure].max()
    assert err < (1e-12 if fp64 else 2e-4)
    for e in ([-1000, -300, -160, -40, 40, 160, 300, 1000] if fp64 else [-120, -64, -40, -30, -20, 15, 20, 30, 64, 120]):
        q, _ = mdarap.host_best_rotation(cov * 2.0 ** e, fp64=fp64)
        assert np.array_equal(q, base), e


@pytest.mark.gpu
@pytest.mark.parametrize("scale", [1e-2, 1.0, 1e3, 1e5, 1e7])
def test_scaled_mesh_on_the_device(scale):
    if mdarap.device_count() == 0:
        pytest.fail("no GPU visible: the HIP path cannot run")
    ctx = mdarap.Context(0)
    pr = meshgen.sphere_problem(12, 20)
    idx, tgt = pr.constraints()
    ref = oracle.Arap(pr.xyz * scale, pr.tri)
    ref.set_constraints(idx, tgt * scale)
    assert ref.deform(5)
    for prec, tol in ((mdarap.PREC_FP64, 1e-9), (mdarap.PREC_FP32_REFINE, 1e-5)):
        print("case: scale=%g precision=%d" % (scale, prec), flush=True)
        m = mdarap.Mesh(ctx, pr.xyz * scale, pr.tri, mdarap.config(precision=prec))
        m.set_constraints(idx, tgt * scale)
        assert m.deform(5)
        assert meshgen.relative_error(m.mesh, ref.mesh) < tol
        m.close()
    ctx.close()

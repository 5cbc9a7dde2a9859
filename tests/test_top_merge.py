"""Merged tops of the factor at the edges of their rule: systems of 1 to 402 free columns around the 400
that become one dense supernode, alone and as two components (two roots), on the host emulation
against scipy; and on the device, in both rest modes, against the oracle."""
import numpy as np
import pytest
import scipy.sparse as sp
import scipy.sparse.linalg as spla

import meshgen
import mdarap
import oracle


def _system(nf, parts):
    """Cotan systems of `parts` spheres side by side, nf free vertices each (a band around the equator
    last to be held)."""
    blocks, pos = [], []
    for k in range(parts):
        xyz, tri = meshgen.uv_sphere(24, 32)
        xyz = meshgen.radial_noise(xyz, 0.01, nf + k)
        rp, ci, w = oracle.cotan_csr(xyz, tri)
        W = sp.csr_matrix((w, ci, rp), shape=(len(xyz), len(xyz)))
        free = np.sort(np.argsort(np.abs(xyz[:, 2]), kind="stable")[:nf])
        deg = np.asarray(W.sum(axis=1)).ravel()
        blocks.append(sp.diags(deg[free]) - W[free][:, free])
        pos.append(xyz[free] + np.array([3.0 * k, 0.0, 0.0]))
    L = sp.block_diag(blocks, format="csr")
    L.sort_indices()
    return L, np.concatenate(pos)


@pytest.mark.parametrize("nf,parts", [(1, 1), (2, 2), (64, 1), (65, 1), (130, 2), (200, 2), (201, 2), (399, 1), (400, 1),
                                      (401, 1), (402, 2)])
@pytest.mark.parametrize("emulation", [False, True])
def test_merged_top_matches_scipy(nf, parts, emulation):
    L, fx = _system(nf, parts)
    b = np.random.default_rng(nf).standard_normal((3, L.shape[0]))
    x, entries, levels = mdarap.host_factor_solve(L.indptr, L.indices, L.data, fx, b, subtree_budget=0, level_pairs=True,
                                                  device_factor_emulation=emulation)
    ref = spla.spsolve(L.tocsc(), b.T).T
    np.testing.assert_allclose(x, ref, rtol=1e-9, atol=1e-11 * np.abs(ref).max())
    if 64 < nf and nf * parts <= 400:  # (smaller supernodes may merge or stay apart)
        assert levels == 1 and entries == parts * nf * nf


@pytest.mark.gpu
@pytest.mark.parametrize("nf", [64, 400, 401, 999, 1500])
def test_merged_top_on_the_device(nf):
    xyz, tri = meshgen.uv_sphere(36, 48)
    xyz = meshgen.radial_noise(xyz, 0.01, nf)
    held = np.sort(np.argsort(np.abs(xyz[:, 2]), kind="stable")[nf:]).astype(np.int32)
    tgt = xyz[held] + np.where(xyz[held][:, 2:3] > 0, 0.2, 0.0) * np.array([1.0, 0.0, 1.0])
    ref = oracle.Arap(xyz, tri)
    ref.set_constraints(held, tgt)
    assert ref.deform(3)
    ctx = mdarap.Context(0)
    for prec, tol in ((mdarap.PREC_FP64, 1e-9), (mdarap.PREC_FP32_REFINE, 1e-5)):
        for rest in (mdarap.REST_REFERENCE, mdarap.REST_FIXED):
            print("case: nf=%d precision=%d rest=%d" % (nf, prec, rest), flush=True)
            m = mdarap.Mesh(ctx, xyz, tri, mdarap.config(precision=prec, rest_mode=rest))
            m.set_constraints(held, tgt)
            assert m.deform(3)
            st = m.stats()
            if nf == 400:
                assert st["levels"] == 1 and st["max_sn_width"] == nf
            assert meshgen.relative_error(m.mesh, ref.mesh) < tol
            m.close()
    ctx.close()

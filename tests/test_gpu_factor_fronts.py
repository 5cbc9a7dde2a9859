"""Device factorization on fronts of chosen shapes, without level pairs: w pivot columns and noff off rows at
the edges of the sweeps' panels (4), blocks (16) and tiles (64), on leaves and on fronts with two children
(their update matrices land on pivot rows and on off rows). Against the oracle, in both precisions; the shapes
are checked by the panel entries of the analysis."""
import numpy as np
import pytest

import meshgen
import mdarap
import oracle

POS_TOL = {mdarap.PREC_FP64: 1e-9, mdarap.PREC_FP32_REFINE: 1e-5}
EDGES = [1, 15, 16, 17, 63, 64, 65, 127, 128, 129]
CASES = ([(x, 65, 40, 33) for x in EDGES] + [(65, x, max(1, x // 2), max(33, x - x // 2)) for x in EDGES] +
         [(20, x + 10, x, 65) for x in EDGES] + [(20, 65 + min(x, 10), 65, x) for x in EDGES])


def tree_of_cliques(a, no, s, r):
    """A mesh whose free vertices are two cliques A and B under a clique S, twice, under a clique R, placed so
    that nested dissection cuts R, then S, out: A (a columns, no off rows: S and some of R) and B end up as
    leaves, S (s columns, off rows R) as a front with two children, R as the root with two. Every edge between free
    vertices is a face whose third vertex is one of twelve held ones. Returns xyz, tri, held, targets and the
    panel entries of that tree."""
    rng = np.random.default_rng([a, no, s, r])
    b = a + s
    b2 = b + (r + 1) // 2
    sizes = dict(A1=a, S1=s, B1=b, R=r, A2=b2 - s, S2=s, B2=b2)
    place = dict(A1=(-4, -1.5), S1=(-4, -0.4), B1=(-4, 1.5), R=(-2, 0), A2=(4, -1.5), S2=(4, -0.4), B2=(4, 1.5))
    ids, pos, n = {}, [], 0
    for k, c in sizes.items():
        ids[k] = np.arange(n, n + c)
        n += c
        pos.append(rng.uniform(-0.5, 0.5, (c, 3)) + np.array([place[k][0], place[k][1], 0.0]))
    rows = {}
    for k in ("1", "2"):
        c = no - s if k == "1" else r // 2
        rows["A" + k] = np.concatenate([ids["S" + k], rng.choice(ids["R"], c, replace=False)])
        part = ids["R"] if k == "2" else rng.choice(ids["R"], (r + 1) // 2, replace=False)
        rows["B" + k] = np.concatenate([ids["S" + k], part])
        rows["S" + k] = ids["R"]
    rows["R"] = np.zeros(0, int)
    edges, entries = [], 0
    for k, v in ids.items():
        i, j = np.triu_indices(len(v), 1)
        edges.append(np.stack([v[i], v[j]], 1))
        edges.append(np.stack([np.repeat(v, len(rows[k])), np.tile(rows[k], len(v))], 1))
        entries += len(v) * (len(v) + len(rows[k]))
    edges = np.concatenate(edges)
    held = np.arange(n, n + 12)
    d = rng.standard_normal((12, 3))
    pos.append(6.0 * d / np.linalg.norm(d, axis=1, keepdims=True))
    xyz = np.concatenate(pos)
    tri = np.concatenate([edges, rng.choice(held, (len(edges), 1))], 1)
    # a held vertex of every free one, so that none hangs by its own clique only
    ring = np.stack([np.arange(n), rng.choice(held[:6], n), rng.choice(held[6:], n)], 1)
    tgt = xyz[held] + np.where(np.arange(12)[:, None] < 6, 0.0, 1.0) * np.array([0.3, 0.1, -0.2])
    return xyz, np.concatenate([tri, ring]).astype(np.int32), held.astype(np.int32), tgt, entries


@pytest.fixture(scope="module")
def ctx():
    if mdarap.device_count() == 0:
        pytest.fail("no GPU visible: the HIP path cannot run")
    c = mdarap.Context(0)
    yield c
    c.close()


@pytest.mark.gpu
@pytest.mark.parametrize("a,no,s,r", CASES)
def test_fronts(ctx, a, no, s, r):
    xyz, tri, held, tgt, entries = tree_of_cliques(a, no, s, r)
    ref = oracle.Arap(xyz, tri)
    ref.set_constraints(held, tgt)
    assert ref.deform(2)
    for prec, tol in POS_TOL.items():
        print("case: a=%d no=%d s=%d r=%d precision=%d" % (a, no, s, r, prec), flush=True)
        m = mdarap.Mesh(ctx, xyz, tri, mdarap.config(precision=prec, amalg_ratio=0.0, subtree_budget=0, level_pairs=False))
        m.set_constraints(held, tgt)
        assert m.deform(2)
        st = m.stats()
        assert st["supernodes"] == 7 and st["levels"] == 3
        assert st["panel_entries"] == entries
        assert meshgen.relative_error(m.mesh, ref.mesh) < tol
        m.close()


def expander(n, degree, seed=0):
    """A random graph (every edge a face with one of sixteen held vertices as its apex): its separators are
    about half of what is left, so its fronts are nearly as large as the system."""
    rng = np.random.default_rng(seed)
    e = rng.integers(0, n, (n * degree // 2, 2))
    e = np.unique(np.sort(e[e[:, 0] != e[:, 1]], axis=1), axis=0)
    held = np.arange(n, n + 16)
    d = rng.standard_normal((16, 3))
    xyz = np.concatenate([rng.uniform(-1.0, 1.0, (n, 3)), 3.0 * d / np.linalg.norm(d, axis=1, keepdims=True)])
    tri = np.concatenate([e, rng.choice(held, (len(e), 1))], 1)
    ring = np.stack([np.arange(n), rng.choice(held[:8], n), rng.choice(held[8:], n)], 1)
    tgt = xyz[held] + np.where(np.arange(16)[:, None] < 8, 0.0, 1.0) * np.array([0.3, 0.1, -0.2])
    return xyz, np.concatenate([tri, ring]).astype(np.int32), held.astype(np.int32), tgt


@pytest.mark.gpu
def test_fronts_of_more_rows_than_one_map(ctx):
    """Fronts of more than 8,192 rows are assembled by ranges of rows. Against the Jacobi-PCG global step to
    1e-13 (the oracle's factorization of the same system would take many minutes)."""
    n = 11000
    xyz, tri, held, tgt = expander(n, 16)
    out = []
    for kw in (dict(level_pairs=False), dict(solver=mdarap.SOLVER_PCG, pcg_iters=400, pcg_tol=1e-13)):
        print("case: n=%d %s" % (n, sorted(kw)), flush=True)
        m = mdarap.Mesh(ctx, xyz, tri, mdarap.config(precision=mdarap.PREC_FP64, **kw))
        m.set_constraints(held, tgt)
        assert m.deform(2)
        if not out:
            assert m.stats()["max_sn_rows"] > 8192
        out.append(m.mesh.copy())
        m.close()
    assert np.all(np.isfinite(out[0]))
    assert meshgen.relative_error(out[0], out[1]) < POS_TOL[mdarap.PREC_FP64]

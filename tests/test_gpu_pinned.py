"""Calls that find no pinned host memory, forced by tests/cpp/pinned_shim.c in a process of their own: they
do without it (bitwise the same results), and a failed allocation leaves nothing behind that a later call
would report."""
import os
import subprocess
import sys

import pytest

pytestmark = pytest.mark.gpu

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

HEAD = """
import ctypes, sys
shim = ctypes.CDLL(sys.argv[1], mode=ctypes.RTLD_GLOBAL)
sys.path[:0] = [%r, %r]
import numpy as np
import mdarap, meshgen

def refuse(lo, hi):
    ctypes.c_size_t.in_dll(shim, "shim_lo").value = lo
    ctypes.c_size_t.in_dll(shim, "shim_hi").value = hi

def refused():
    return ctypes.c_int.in_dll(shim, "shim_refused").value

def mesh(ctx, pr, **kw):
    m = mdarap.Mesh(ctx, pr.xyz, pr.tri, mdarap.config(**kw))
    m.set_constraints(*pr.constraints())
    return m
""" % (os.path.join(ROOT, "mesh-deform_amd"), os.path.join(ROOT, "oracle"))


@pytest.fixture(scope="module")
def shim(tmp_path_factory):
    so = str(tmp_path_factory.mktemp("shim") / "pinned_shim.so")
    subprocess.check_call(["gcc", "-O1", "-shared", "-fPIC", "-o", so, os.path.join(ROOT, "tests", "cpp", "pinned_shim.c"),
                           "-ldl"])
    return so


def run(shim, body):
    p = subprocess.run([sys.executable, "-u", "-c", HEAD + body, shim], stdout=subprocess.PIPE, stderr=subprocess.STDOUT,
                       timeout=100, text=True)
    print(p.stdout, flush=True)
    assert p.returncode == 0 and p.stdout.rstrip().endswith("done"), p.stdout


def test_failed_block_leaves_no_error_behind(shim):
    """The call after one whose pinned block (about 1.3 MB) was refused succeeds."""
    run(shim, """
ctx = mdarap.Context(0)
pr = meshgen.sphere_problem(12, 20)
ref = mesh(ctx, pr)
assert ref.deform(5)
other = mdarap.Context(0)
m = mesh(other, pr)
refuse(1 << 20, 1 << 40)
try:
    m.deform(5)
except mdarap.MDError as e:
    print("refused:", e)
assert refused() > 0
refuse(1, 0)
n = mesh(other, pr)
assert n.deform(5) and np.array_equal(n.mesh, ref.mesh)
print("done")
""")


def test_failed_pack_entries_leave_no_error_behind(shim):
    """The server's requests after one whose pack entries (64 bytes a result) were refused succeed."""
    run(shim, """
ctx = mdarap.Context(0)
prs = [meshgen.sphere_problem(12, 20), meshgen.sphere_problem(14, 24)]
ms = [mesh(ctx, pr, rest_mode=mdarap.REST_FIXED) for pr in prs]
for m, pr in zip(ms, prs):
    m.prepare(pr.xyz)
srv = mdarap.Server(ctx)
ids = [srv.add_mesh(m) for m in ms]
refuse(64, 256)
try:
    srv.wait(srv.submit(ids[0], *prs[0].constraints(), 3), prs[0].n)
except mdarap.MDError as e:
    print("refused:", e)
assert refused() > 0
refuse(1, 0)
for k in range(4):
    pos, _ = srv.wait(srv.submit(ids[1], *prs[1].constraints(), 3), prs[1].n)
    assert np.all(np.isfinite(pos))
srv.close()
print("done")
""")


@pytest.mark.parametrize("solver", ["direct", "host factor", "pcg"])
def test_calls_without_a_block(shim, solver):
    """Prepare, deform (frames and drags, small and of more than the block's size, short and long, a factor
    that fails), download and normals with every pinned block refused: as with it."""
    run(shim, """
solver = %r
kw = dict(solver=mdarap.SOLVER_PCG, pcg_iters=30) if solver == "pcg" else dict(factor_device=solver == "direct")
prs = [meshgen.sphere_problem(12, 20)]
if solver != "host factor":
    prs.append(meshgen.noisy_icosphere_problem(6))

def calls(blocks):
    refuse(*((1, 0) if blocks else (1 << 20, 1 << 40)))
    before = refused()
    out = []
    for pr in prs:
        for rest in (mdarap.REST_REFERENCE, mdarap.REST_FIXED):
            print("case:", solver, "n", pr.n, "rest", rest, "blocks", blocks, flush=True)
            ctx = mdarap.Context(0)
            m = mesh(ctx, pr, rest_mode=rest, **kw)
            idx, tgt = pr.constraints()
            for k in (0, 3, 12):
                m.set_constraints(idx, tgt + 0.01 * k)
                assert m.deform(k)
                out.append(m.mesh.copy())
            m.deform(2)
            out += [m.download(), m.normals()]
            other = mesh(ctx, pr, rest_mode=rest, **kw)
            other.prepare(pr.xyz)
            other.iterate(2)
            out.append(other.download())
            m.close()
            other.close()
            ctx.close()
    a, b = meshgen.sphere_problem(10, 16), meshgen.sphere_problem(8, 12)
    if solver != "pcg":
        ctx = mdarap.Context(0)
        xyz = np.concatenate([a.xyz, b.xyz + np.array([5.0, 0.0, 0.0])])
        m = mdarap.Mesh(ctx, xyz, np.concatenate([a.tri, b.tri + a.n]).astype(np.int32), mdarap.config(**kw))
        m.set_constraints(*a.constraints())
        for k in (2, 20):
            assert not m.deform(k) and np.array_equal(m.mesh, xyz)
        far = a.n + np.arange(3)
        m.set_constraints(far, xyz[far])
        assert m.deform(4)
        out.append(m.mesh.copy())
        m.close()
        ctx.close()
    assert blocks == (refused() == before)
    return out

with_blocks, without = calls(True), calls(False)
assert len(with_blocks) == len(without)
for x, y in zip(with_blocks, without):
    assert np.all(np.isfinite(x)) and np.array_equal(x, y)
print("done")
""" % solver)


def test_served_results_without_pack_entries(shim):
    """A server whose pack entries (64 bytes a result) are refused gives what it gives with them."""
    run(shim, """
prs = [meshgen.sphere_problem(12, 20), meshgen.sphere_problem(14, 24), meshgen.noisy_icosphere_problem(4)]
out = []
for lo, hi in ((1, 0), (64, 256)):
    ctx = mdarap.Context(0)
    ms = [mesh(ctx, pr, rest_mode=mdarap.REST_FIXED) for pr in prs]
    for m, pr in zip(ms, prs):
        m.prepare(pr.xyz)
    srv = mdarap.Server(ctx)
    ids = [srv.add_mesh(m) for m in ms]
    refuse(lo, hi)
    before = refused()
    got = []
    for k in range(3):
        tickets = [srv.submit(i, pr.constraints()[0], pr.constraints()[1] + 0.01 * k, 3) for i, pr in zip(ids, prs)]
        got += [srv.wait(t, pr.n)[0] for t, pr in zip(tickets, prs)]
    assert (refused() > before) == (lo <= hi)
    refuse(1, 0)
    srv.close()
    out.append(got)
for x, y in zip(*out):
    assert np.all(np.isfinite(x)) and np.array_equal(x, y)
print("done")
""")

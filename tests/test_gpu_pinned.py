"""Calls that find no pinned host memory, forced by tests/cpp/pinned_shim.c in a process of their own: a
failed allocation leaves nothing behind that a later call would report."""
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

"""The rule that splits the subtree launches of several meshes by LDS, on the host: launches are split only
where the subtrees together are more than fill the chip at once (1,024), and a mesh without subtrees adds
none of its own."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "mesh-deform_amd", "csrc")


@pytest.fixture(scope="module")
def prog(tmp_path_factory):
    exe = str(tmp_path_factory.mktemp("classes") / "test_subtree_classes")
    subprocess.check_call(["g++", "-std=c++17", "-O1", "-Wall", "-I" + CSRC, "-I" + os.path.join(ROOT, "include"), "-o", exe,
                           os.path.join(ROOT, "tests", "cpp", "test_subtree_classes.cpp"),
                           os.path.join(CSRC, "md_analysis.cpp")])
    return exe


@pytest.mark.parametrize("meshes,classes", [
    ([], []),
    ([(5000, 1024)], [0]),                                    # alone: one launch, whatever its size
    ([(0, 0), (91, 512)], [0, 0]),                            # a merged whole system beside an ordinary mesh
    ([(8, 100), (91, 512), (300, 1000)], [0, 0, 0]),          # all of them in flight at once
    ([(24, 192), (1000, 1024)], [0, 0]),                      # 1,024 together
    ([(25, 192), (1000, 1024)], [0, 2]),                      # 1,025: by LDS
    ([(600, 192), (600, 193), (600, 576), (600, 577)], [0, 1, 1, 2]),
    ([(0, 0), (700, 500), (0, 0), (700, 900)], [1, 1, 1, 2]),  # without subtrees: the first class there is
    ([(0, 0), (0, 0)], [0, 0]),
    ([(2000, 128), (0, 0), (2000, 1024)], [0, 0, 2]),
])
def test_classes(prog, meshes, classes):
    out = subprocess.check_output([prog] + ["%d,%d" % m for m in meshes], text=True)
    assert [int(x) for x in out.split()] == classes

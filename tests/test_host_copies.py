"""The copies between a caller's arrays and the device (akx_copy.hpp) on a host
stand-in for the runtime whose copies happen as late as they may: sizes at the
edges of the small, one-slot, one-lane and threaded copies, several uploads in a
row, and page-locked memory that runs out at any point."""
import os
import subprocess

import pytest

HERE = os.path.join(os.path.dirname(os.path.abspath(__file__)), "host")
KB, MB = 1 << 10, 1 << 20
EDGES = [1, 16 * KB, 16 * KB + 1, 128 * KB, 128 * KB + 1, MB, MB + 1, 2 * MB + 5, 8 * MB, 8 * MB + 1, 17 * MB + 3]


@pytest.fixture(scope="module")
def program(tmp_path_factory):
    out = str(tmp_path_factory.mktemp("copies") / "copies")
    subprocess.run([os.environ.get("CXX", "g++"), "-O2", "-std=c++17", "-pthread", "-Wall",
                    "-D_GLIBCXX_ASSERTIONS", "-I", HERE,
                    os.path.join(HERE, "copies.cc"), "-o", out], check=True)
    return out


@pytest.mark.parametrize("pinned", [1000, 0, 1, 2, 5])
@pytest.mark.parametrize("sizes", [[5, 70 * KB, 3, 9, 128 * KB, 1], EDGES, EDGES[::-1],
                                   [130 * KB, 2, 130 * KB, 3, 900 * KB, 4, 2 * MB, 5]])
def test_copies(program, sizes, pinned):
    r = subprocess.run([program, str(pinned)] + [str(n) for n in sizes], capture_output=True,
                       text=True, timeout=100)
    assert r.returncode == 0, (r.returncode, r.stdout, r.stderr[-2000:])

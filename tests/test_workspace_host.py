"""The evaluation workspaces' growth (speo-gpu-single-control_amd/csrc/workspace.h) on
the host, over a device of a given size: what a call can do without is never the
reason for its failure, is not asked for again and again, and is not allocated
inside a stream capture; a buffer that does is kept until a larger one is there."""
import shutil
import subprocess

import pytest

from conftest import REPO


@pytest.fixture(scope="module")
def exe(tmp_path_factory):
    gxx = shutil.which("g++")
    if not gxx:
        pytest.skip("g++ not available")
    out = tmp_path_factory.mktemp("workspace") / "workspace_check"
    subprocess.run([gxx, "-O1", "-std=c++17", f"-I{REPO / 'speo-gpu-single-control_amd' / 'csrc'}",
                    str(REPO / "tests" / "cpp" / "workspace_check.cpp"), "-o", str(out)], check=True)
    return out


# lines, and for each R: (status, floats held, allocations tried, waits, live buffers)
CASES = {
    "room": (["M 1000", "R 10 100 1", "R 50 100 1", "R 120 200 1"], [(0, 100, 1, 1, 1), (0, 100, 0, 0, 1),
                                                                     (0, 200, 1, 1, 1)]),
    "no room for the wanted": (["M 90", "R 10 100 1", "R 10 100 1", "R 10 300 1", "R 40 60 1"],
                               [(0, 10, 2, 1, 1), (0, 10, 0, 0, 1), (0, 10, 0, 0, 1), (0, 60, 1, 1, 1)]),
    "no room at all": (["M 5", "R 10 100 1", "M 500", "R 10 100 1"], [(-1, 0, 2, 1, 0), (0, 10, 1, 1, 1)]),
    "optional": (["M 90", "R 0 80 1", "R 0 85 1", "R 0 85 1", "R 0 70 1"],
                 [(0, 80, 1, 0, 1), (0, 80, 1, 0, 1), (0, 80, 0, 0, 1), (0, 80, 0, 0, 1)]),
    "capture": (["M 1000", "R 0 100 0", "R 10 100 0", "R 10 20 1", "R 10 100 0", "R 10 100 1"],
                [(0, 0, 0, 0, 0), (7, 0, 0, 1, 0), (0, 20, 1, 1, 1), (0, 20, 0, 0, 1), (0, 100, 1, 1, 1)]),
}


@pytest.mark.parametrize("name", CASES)
def test_reserve(exe, name):
    lines, expect = CASES[name]
    res = subprocess.run([str(exe)], input="\n".join(lines).encode(), capture_output=True, check=True)
    assert [tuple(map(int, ln.split())) for ln in res.stdout.decode().splitlines()] == expect

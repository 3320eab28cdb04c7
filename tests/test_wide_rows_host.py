"""Row addresses of the wide tile kernel (speo-gpu-single-control_amd/csrc/
wide_core.h) on the host: no load in range leaves the caller's rows, which end with
the last row's last column (a column slice of a wider matrix owns nothing behind
it), none that the arithmetic needs is out of range, and no offset passes 31 bits."""
import shutil
import subprocess

import pytest

from conftest import REPO

PKG = REPO / "speo-gpu-single-control_amd"


@pytest.fixture(scope="module")
def exe(tmp_path_factory):
    hipcc = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
    if not shutil.which(hipcc):
        pytest.skip("hipcc not available")
    out = tmp_path_factory.mktemp("wide") / "wide_rows_check"
    subprocess.run([hipcc, "-O2", "--offload-arch=gfx950", "-x", "hip", "-std=c++17",
                    f"-I{REPO / 'include'}", f"-I{PKG / 'csrc'}",
                    str(REPO / "tests" / "cpp" / "wide_rows_check.cpp"), "-o", str(out)],
                   check=True, capture_output=True)
    return out


def _run(exe, cases):
    res = subprocess.run([str(exe)], input="".join(" ".join(map(str, c)) + "\n" for c in cases).encode(),
                         capture_output=True, check=True)
    return res.stdout.decode().splitlines()


def test_loads_stay_in_the_callers_rows(exe):
    # (rows a block, waves) of the batch and of the engine kernel; whole and short
    # tiles; contiguous rows, padded rows and column slices at every remainder
    cases = [(rb, nw, nrows, ld, dim) for rb, nw in ((128, 8), (64, 4)) for nrows in (1, 7, 63, 64, rb)
             for dim in (129, 130, 131, 132, 159, 160, 161, 232, 257, 1000)
             for ld in ((dim + 3) // 4 * 4, (dim + 3) // 4 * 4 + 4, 1024) if ld >= dim]
    for case, got in zip(cases, _run(exe, cases)):
        assert got == "0 0 0", case


def test_strides_within_31_bits(exe):
    # 128 rows x 2^22 floats are 2^31 bytes: refused; one group less is taken
    cases = [(128, 8, 128, 2 ** 22, 1000), (128, 8, 128, 2 ** 22 - 4, 1000), (64, 4, 64, 2 ** 22, 1000)]
    assert _run(exe, cases) == ["refused", "0 0 0", "0 0 0"]

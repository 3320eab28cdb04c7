"""Device memory that problems take: the rotation in the layouts that something
reads, and no other."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _layout_bytes(D, generic):
    """A component's arrays: the rotation in FP64 and FP32, its three BF16 and three FP16
    parts, up to 128 columns the zero-padded FP32 and 16-bit operands, from 129 columns on
    the FP32 and six 16-bit arrays of 256-column tiles (none for the generic kernel's
    objectives), the FP64 kernel's fragments, the shift and the weights."""
    up = lambda n, m: (n + m - 1) // m * m  # noqa: E731
    b = D * (D * 8 + up(D, 4) * 4 + 6 * 2 * up(D, 32))
    b += 128 * 128 * 4 + 6 * 2 * 128 * up(D, 32) if D <= 128 else 0
    b += 0 if D <= 128 or generic else 16 * up(up(D, 16), 256) * up(D, 32)
    b += up(D, 16) * up(D, 8) * 8
    return b + D * (8 + 4 + 4 + 4)


@pytest.mark.parametrize("D,obj,count", [(10, 2, 256), (100, 3, 128), (500, 9, 16), (500, 2, 16)])
def test_problem_memory(cuda, speo, D, obj, count):
    import torch
    rng = np.random.default_rng(D)
    o = rng.uniform(-80, 80, (1, D))
    M = np.linalg.qr(rng.standard_normal((D, D)))[0][None]
    first = speo.Problem([obj], o, M)  # (what a first creation loads)
    torch.cuda.synchronize()
    free0 = torch.cuda.mem_get_info()[0]
    probs = [speo.Problem([obj], o, M) for _ in range(count)]
    each = (free0 - torch.cuda.mem_get_info()[0]) / count
    print(f"D {D} objective {obj}: {each / 1024:.0f} KiB a problem, layouts {_layout_bytes(D, obj > 8) / 1024:.0f}",
          flush=True)
    # 32 arrays rounded up to 256 bytes; of the two allocations the driver rounds the
    # tables' up to 64 KiB, the data's as well or, from 2 MiB on, to whole 2 MiB
    data = _layout_bytes(D, obj > 8) + 32 * 256
    unit = 65536 if data < 2 << 20 else 2 << 20
    assert each <= -(-data // unit) * unit + 65536
    for p in probs + [first]:
        p.close()


@pytest.mark.parametrize("prec", range(6))
def test_narrow_islands_beside_wide_ones(cuda, speo, prec):
    """Islands of up to 128 columns beside wider ones take the tile kernel as those do:
    the bits of the 64-row form, composition and single objective."""
    rng = np.random.default_rng(4)
    probs = []
    for D, objs in ((129, [2]), (40, [3]), (128, [1, 2]), (7, [7])):
        probs.append(speo.Problem(objs, np.float32(rng.uniform(-80, 80, (len(objs), D))).astype(np.float64),
                                  np.stack([np.linalg.qr(rng.standard_normal((D, D)))[0] for _ in objs]),
                                  sigma=[10.0 * (c + 1) for c in range(len(objs))]))
    out = []
    for on in (1, 0):
        prev, _ = speo.wide_eval(on)
        print(f"precision {prec} tile kernel {on}", flush=True)
        e = speo.Engine(probs, [64, 70, 33, 100], [0, 1, 2, 3], mode=speo.MODE_FUSED, precision=prec, seed=8,
                        rows_per_block=32)
        speo.wide_eval(prev)
        e.run(4)
        out.append(e.read() + e.read_trials())
        e.close()
    for a, b in zip(*out):
        np.testing.assert_array_equal(a, b)
    for p in probs:
        p.close()


_HOST = """
import resource, sys
import numpy as np, torch
sys.path.insert(0, {pkg!r})
import speo_de as S
torch.zeros(1, device="cuda")
rng = np.random.default_rng(1)
D, nc = 1200, 8
S.Problem([2], rng.random((1, D)), rng.random((1, D, D))).close()
o, M = rng.random((nc, D)), rng.random((nc, D, D))
before = resource.getrusage(resource.RUSAGE_SELF).ru_maxrss
S.Problem([2] * nc, o, M)
print("grown", resource.getrusage(resource.RUSAGE_SELF).ru_maxrss - before, flush=True)
"""


def test_host_memory_of_a_composition(cuda, speo):
    """The host holds the arrays of one component of a wide composition at a time: 24
    bytes an element twice (made and gathered), not of all eight."""
    import subprocess
    import sys
    from conftest import REPO
    res = subprocess.run([sys.executable, "-c", _HOST.format(pkg=str(REPO / "speo-gpu-single-control_amd"))],
                         capture_output=True, text=True, timeout=100, check=True)
    grown = int(res.stdout.split("grown")[1]) * 1024
    print(f"{grown / 2 ** 20:.0f} MiB", flush=True)
    assert grown < 3 * 24 * 1200 ** 2 + (32 << 20)

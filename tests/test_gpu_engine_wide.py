"""Engines with islands wider than 128 columns: the evaluation on the tile kernel
equals the K-chunked kernel's bit for bit (populations and fitness after
generations with a migration), for every rows-per-block arithmetic, precision
and mode, with island sizes off the 64-row tile and single objectives next to a
composition."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _problems(speo):
    rng = np.random.default_rng(77)
    out = []
    for D, objs in ((129, [2]), (300, [1, 2, 3]), (40, [3]), (257, [5]), (160, [6])):
        o = np.float32(rng.uniform(-80, 80, (len(objs), D))).astype(np.float64)
        M = np.stack([np.linalg.qr(rng.standard_normal((D, D)))[0] for _ in objs])
        out.append(speo.Problem(objs, o, M, sigma=[10.0 * (c + 1) for c in range(len(objs))],
                                bias=[100.0 * c for c in range(len(objs))],
                                rate=[0.05 if q == 6 else 1.0 for q in objs]))
    return out


@pytest.mark.parametrize("tile", [16, 32, 64])
@pytest.mark.parametrize("prec", range(6))
def test_tile_kernel_equals_chunked_kernel(cuda, speo, tile, prec):
    probs = _problems(speo)
    sizes, which = [63, 64, 65, 128, 200, 8, 70], [0, 1, 2, 1, 0, 3, 4]
    state = {}
    for on in (1, 0):
        prev, _ = speo.wide_eval(on)
        engines = [speo.Engine(probs, sizes, which, seed=9, interval=3, migration_size=2, precision=prec,
                               mode=m, rows_per_block=tile) for m in (speo.MODE_PLAIN, speo.MODE_FUSED)]
        speo.wide_eval(prev)
        for e in engines:
            print(f"tile {tile} precision {prec} tile kernel {on} mode {e.cfg.mode}", flush=True)
            e.run(5)
            state[on, e.cfg.mode] = e.read()
            e.close()
    X, f = state[0, speo.MODE_PLAIN]
    assert np.isfinite(f).all()
    for key, (Xb, fb) in state.items():
        np.testing.assert_array_equal(fb, f, err_msg=str(key))
        np.testing.assert_array_equal(Xb, X, err_msg=str(key))
    for p in probs:
        p.close()


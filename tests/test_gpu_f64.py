"""The FP64 kernels at the edges of their tiles: evaluate_f64 (16-row tiles,
16-column tiles of z, K steps of 8, one to four column tiles per wave up to
1024 columns, one block per row beyond), the drop-in FP64 functions on the
caller's M^T, and Engine.best over islands of one and of several 128-column
chunks.  Reference: z by numpy in FP64 and the oracle's FP64 objectives;
tolerance 1e-11 relative, the bound of the FP64 objectives' other tests."""
import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu
RTOL = 1e-11


def _t(a, cuda):
    import torch
    return torch.from_numpy(np.ascontiguousarray(a)).to(cuda)


def _rotation(rng, D):
    return np.linalg.qr(rng.standard_normal((D, D)))[0]


def _values(oracle, obj, Z):
    return np.array([oracle.basic(obj, z) for z in Z])


def _composition(oracle, X, objs, o, M, rate, sigma, bias):
    fit, logw = [], []
    for c, obj in enumerate(objs):
        v = X - o[c]
        fit.append(_values(oracle, obj, (v * rate[c]) @ M[c].T) + bias[c])
        d = (v * v).sum(1)
        logw.append(-0.5 * np.log(d) - d / (2.0 * X.shape[1] * sigma[c] ** 2))
    w = np.exp(np.array(logw) - np.max(logw, axis=0))
    return (w / w.sum(0) * np.array(fit)).sum(0)


@pytest.mark.parametrize("D", [2, 7, 8, 9, 16, 17, 33, 128, 129, 255, 256, 257, 513, 1000, 1024, 1025])
@pytest.mark.parametrize("kind", ["fused", "generic"])
def test_evaluate_f64_tile_edges(cuda, speo, oracle, D, kind):
    import torch
    if kind == "generic" and D > 1024:
        pytest.skip("generic objectives take dim <= 1024")
    rng = np.random.default_rng(D)
    objs = [1, 2, 3] if kind == "fused" else [speo.OBJ_GRIEWANK, speo.OBJ_KATSUURA, speo.OBJ_GRIE_ROSEN]
    rate = [1.0, 0.0512, 1.0] if kind == "fused" else [6.0, 0.05, 0.05]
    sigma, bias = [10.0, 20.0, 30.0], [0.0, 100.0, 200.0]
    o = np.float32(rng.uniform(-80, 80, (3, D))).astype(np.float64)
    M = np.stack([_rotation(rng, D) for _ in range(3)])
    prob = speo.Problem(objs, o, M, sigma=sigma, bias=bias, rate=rate)
    for n in (1, 15, 16, 17, 33):
        X = rng.uniform(-100, 100, (n, D)).astype(np.float32)
        f = torch.zeros(n, dtype=torch.float64, device=cuda)
        print(f"{kind} D={D} n={n}", flush=True)
        speo.evaluate_f64(prob, _t(X, cuda), f)
        ref = _composition(oracle, X.astype(np.float64), objs, o, M, rate, sigma, bias)
        np.testing.assert_allclose(f.cpu().numpy(), ref, rtol=RTOL)
    prob.close()


def test_cosine_of_large_arguments(cuda, speo):
    """Ackley without rotation or shift: mean cos(2 pi z) at |z| from 1 to
    1e30 (both reductions), against numpy's cosine of the same products."""
    import torch
    D = 64
    rng = np.random.default_rng(5)
    X = (rng.choice([-1.0, 1.0], (40, D)) * 10.0 ** rng.uniform(0, 30, (40, 1)) *
         rng.uniform(1, 2, (40, D))).astype(np.float32)
    prob = speo.Problem([speo.OBJ_ACKLEY], np.zeros((1, D)))
    f = torch.zeros(40, dtype=torch.float64, device=cuda)
    speo.evaluate_f64(prob, _t(X, cuda), f)
    z = X.astype(np.float64)
    ref = (np.e - 20.0 * np.exp(-0.2 * np.sqrt((z * z).mean(1))) + 20.0 -
           np.exp(np.cos(2.0 * np.pi * z).mean(1)))
    np.testing.assert_allclose(f.cpu().numpy(), ref, rtol=1e-13)
    prob.close()


@pytest.mark.parametrize("D", [9, 100, 130, 257, 300])
def test_dropin_fp64_function_tile_edges(cuda, speo, oracle, D):
    """F4 (Rosenbrock) through API_evaluateFitness: M^T and the shift are the
    caller's FP32 arrays."""
    import torch
    L, n = speo.lib(), 19
    Dp = L.SPEO_NextPow2Dim(D)
    rng = np.random.default_rng(D)
    M = _rotation(rng, D).astype(np.float32)
    X, shift, B = np.zeros((n, Dp), np.float32), np.zeros(Dp, np.float32), np.zeros((Dp, D), np.float32)
    X[:, :D] = rng.uniform(-100, 100, (n, D))
    shift[:D] = rng.uniform(-80, 80, D)
    B[:D] = M.T
    Xd, sd, Bd = _t(X, cuda), _t(shift, cuda), _t(B, cuda)
    f = torch.zeros(n, dtype=torch.float32, device=cuda)
    p = lambda t: ctypes.c_void_p(t.data_ptr())  # noqa: E731
    L.API_evaluateFitness(p(f), None, None, p(Xd), p(sd), p(Bd), None, None, None, None, n, D, 0.0, 4)
    assert L.API_CheckCUDAError() == 0
    z = ((X[:, :D].astype(np.float64) - shift[:D].astype(np.float64)) * 0.02048) @ M.astype(np.float64).T
    np.testing.assert_allclose(f.cpu().numpy(), _values(oracle, speo.OBJ_ROSENBROCK, z), rtol=2e-7)


@pytest.mark.parametrize("dims", [(2, 9, 128), (100, 129, 300), (1000,)])
def test_best_rows(cuda, speo, oracle, dims):
    """Islands of different widths (one chunk, several), one of them on a
    composition: the lowest row of each and its FP64 value."""
    rng = np.random.default_rng(sum(dims))
    probs, data = [], []
    for k, D in enumerate(dims + dims[-1:]):
        objs = [1, 2, 3] if k == len(dims) else [(2, 3, 1)[k % 3]]
        nc = len(objs)
        o = np.float32(rng.uniform(-80, 80, (nc, D))).astype(np.float64)
        M = np.stack([_rotation(rng, D) for _ in range(nc)])
        sigma, bias = [10.0 * (c + 1) for c in range(nc)], [100.0 * c for c in range(nc)]
        probs.append(speo.Problem(objs, o, M, sigma=sigma, bias=bias))
        data.append((D, objs, o, M, [1.0] * nc, sigma, bias))
    I = len(probs)
    eng = speo.Engine(probs, [24 + 8 * i for i in range(I)], list(range(I)), seed=3,
                      mode=speo.MODE_PLAIN, rows_per_block=16)
    eng.run(2)
    rows, f32, f64 = eng.best()
    X, f = eng.read()
    for i, (D, objs, o, M, rate, sigma, bias) in enumerate(data):
        r0, r1 = int(eng.row_off[i]), int(eng.row_off[i + 1])
        assert rows[i] == r0 + int(np.argmin(f[r0:r1])) and f32[i] == f[rows[i]]
        x = X[rows[i]:rows[i] + 1, :D].astype(np.float64)
        if len(objs) == 1:
            ref = _values(oracle, objs[0], (x - o[0]) @ M[0].T)[0]
        else:
            ref = _composition(oracle, x, objs, o, M, rate, sigma, bias)[0]
        assert f64[i] == pytest.approx(ref, rel=RTOL), (i, D)
    eng.close()
    for p in probs:
        p.close()


@pytest.mark.parametrize("D,objs", [(3, [1, 2, 3]), (40, [10, 9]), (100, [2]), (300, [3, 6, 7])])
def test_values_independent_of_the_batch(cuda, speo, D, objs):
    """Blocks hold 1, 2, 4, 8 or 16 rows as the batch has more than 256, 512, ... of them:
    a row's value is the same bits in all (FP64 values, and FP32 ones of objectives
    that the FP64 kernel evaluates)."""
    import torch
    rng = np.random.default_rng(D)
    o = np.float32(rng.uniform(-80, 80, (len(objs), D))).astype(np.float64)
    prob = speo.Problem(objs, o, np.stack([_rotation(rng, D) for _ in objs]), sigma=[10.0 * (c + 1) for c in range(len(objs))])
    X = _t(rng.uniform(-100, 100, (4101, D)).astype(np.float32), cuda)
    whole = torch.zeros(4101, dtype=torch.float64, device=cuda)
    speo.evaluate_f64(prob, X, whole)
    w32 = torch.zeros(4101, device=cuda)
    speo.evaluate(prob, X, w32)
    for n in (1, 2, 255, 256, 257, 511, 513, 1025, 2048, 2049, 4096, 4097):
        print(f"D={D} n={n}", flush=True)
        f = torch.full((n,), -1.0, dtype=torch.float64, device=cuda)
        speo.evaluate_f64(prob, X[4101 - n:], f)
        np.testing.assert_array_equal(f.cpu().numpy(), whole[4101 - n:].cpu().numpy())
        if max(objs) > 8:
            g = torch.full((n,), -1.0, device=cuda)
            speo.evaluate(prob, X[4101 - n:], g)
            np.testing.assert_array_equal(g.cpu().numpy(), w32[4101 - n:].cpu().numpy())
    prob.close()

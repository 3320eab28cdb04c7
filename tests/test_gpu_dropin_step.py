"""The drop-in generation finds each sub-island's best member in its own launch:
bits of the oracle's generation with the argmin as `best`, for every strategy,
with sub-islands that are and are not a multiple of a block's rows, larger than
one in-launch search, and populations on either side of a wave a row; rows that
allow 16-byte accesses and rows that do not.  The drop-in evaluation of up to
128 columns equals the problem path's 16-row tiles bit for bit."""
import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _dev(a, cuda):
    import torch
    return torch.from_numpy(np.ascontiguousarray(a)).to(cuda)


def _info(speo, cuda, subs, strategy):
    import torch
    return torch.frombuffer(bytearray(speo.de_info_bytes([0.9] * subs, [0.5] * subs, strategy)),
                            dtype=torch.uint8).to(cuda)


@pytest.mark.parametrize("n,subs,D,strategy", [(16, 1, 5, 2), (24, 2, 30, 6), (20, 2, 33, 3), (64, 4, 100, 0),
                                               (64, 4, 100, 1), (100, 5, 128, 8), (4096, 1, 128, 4),
                                               (8192, 2, 20, 7), (8200, 1, 100, 7), (16384, 4, 20, 2),
                                               (16384, 1024, 21, 5)])
def test_generation_finds_best(cuda, speo, oracle, n, subs, D, strategy):
    import torch
    from speo_de._lib import GPU_IslandInfo, GPU_Population, ProblemInfo, SPEO_RandState
    print(f"n {n} sub-islands {subs} D {D} strategy {strategy}", flush=True)
    rng = np.random.default_rng([n, D])
    L = speo.lib()
    ld = L.SPEO_NextPow2Dim(D)
    X = np.zeros((n, ld), np.float32)
    X[:, :D] = rng.uniform(-100, 100, (n, D))
    f = rng.integers(0, max(2, n // 3), n).astype(np.float32)  # ties
    perm = rng.permutation(n).astype(np.int32)
    Xd, fd, pd = _dev(X, cuda), _dev(f, cuda), _dev(perm, cuda)
    U = torch.full((n, ld), 7.0, device=cuda)
    fu = torch.zeros(n, device=cuda)
    best = torch.full((subs,), -1, dtype=torch.int32, device=cuda)
    rs = SPEO_RandState(77, 3, 0)
    pi = ProblemInfo(D, 9, 1, 10000, 77, 0, 0, 100.0, -100.0)
    speo.check(L.API_DE_GenerateNewPopulation(
        GPU_Population(U.data_ptr(), fu.data_ptr()), GPU_Population(Xd.data_ptr(), fd.data_ptr()),
        ctypes.c_void_p(best.data_ptr()), GPU_IslandInfo(n, subs, pd.data_ptr()),
        ctypes.c_void_p(_info(speo, cuda, subs, strategy).data_ptr()), ctypes.byref(rs), pi))
    torch.cuda.synchronize()
    S = n // subs
    expect = [min(perm[s * S:(s + 1) * S], key=lambda i: (f[i], i)) for s in range(subs)]
    assert best.cpu().numpy().tolist() == [int(e) for e in expect]
    ref, *_ = oracle.de_generate(X, ld, n, D, subisland_num=subs, perm=perm, strategy=[strategy] * subs,
                                 best=np.array(expect, np.int32), seed=77, gen=3,
                                 U=np.full((n, ld), 7.0, np.float32))
    np.testing.assert_array_equal(U.cpu().numpy(), ref)


@pytest.mark.parametrize("D,ld,shift", [(6, 7, 0), (6, 8, 1), (7, 8, 0), (128, 130, 0), (65, 68, 2)])
def test_generation_and_selection_rows(cuda, speo, oracle, D, ld, shift):
    import torch
    n = 40
    print(f"D {D} ld {ld} offset {shift}", flush=True)
    rng = np.random.default_rng(D)
    X = rng.uniform(-100, 100, (n, ld)).astype(np.float32)

    def place(a):  # rows `shift` floats past a 16-byte boundary
        t = torch.zeros(n * ld + 4, device=cuda)
        v = t[shift:shift + n * ld].view(n, ld)
        v.copy_(torch.from_numpy(a))
        return v
    Xd, Ud = place(X), place(np.full((n, ld), 7.0, np.float32))
    speo.de_generate(Ud, Xd, D, _info(speo, cuda, 2, 4), subisland_num=2, seed=5, gen=1)
    torch.cuda.synchronize()
    ref, *_ = oracle.de_generate(X, ld, n, D, subisland_num=2, strategy=[4, 4], seed=5, gen=1,
                                 U=np.full((n, ld), 7.0, np.float32))
    np.testing.assert_array_equal(Ud.cpu().numpy(), ref)
    fX, fU = rng.uniform(0, 1, (2, n)).astype(np.float32)
    fXd, fUd = _dev(fX, cuda), _dev(fU, cuda)
    speo.de_select(Xd, fXd, Ud, fUd, D)
    torch.cuda.synchronize()
    acc = fU < fX
    out = X.copy()
    out[acc, :D] = ref[acc, :D]
    np.testing.assert_array_equal(Xd.cpu().numpy(), out)
    np.testing.assert_array_equal(fXd.cpu().numpy(), np.where(acc, fU, fX))


@pytest.mark.parametrize("n,D", [(1, 2), (15, 5), (16, 16), (17, 17), (100, 33), (1024, 100), (31, 127), (33, 128)])
def test_dropin_evaluation_equals_problem(cuda, speo, n, D):
    import torch
    print(f"n {n} D {D}", flush=True)
    rng = np.random.default_rng(D)
    L = speo.lib()
    ld = L.SPEO_NextPow2Dim(D)
    shift = np.float32(rng.uniform(-80, 80, D))
    M = np.float32(np.linalg.qr(rng.standard_normal((D, D)))[0])
    X = torch.zeros((n, ld), device=cuda)
    X[:, :D] = _dev(rng.uniform(-100, 100, (n, D)).astype(np.float32), cuda)
    B = np.zeros((ld, D), np.float32)
    B[:D] = M.T
    sd, Bd = _dev(np.pad(shift, (0, ld - D)), cuda), _dev(B, cuda)
    for fid, obj in ((5, speo.OBJ_ACKLEY), (1, speo.OBJ_ELLIPTIC)):
        f, g = torch.zeros(n, device=cuda), torch.zeros(n, device=cuda)
        L.API_evaluateFitness(ctypes.c_void_p(f.data_ptr()), None, None, ctypes.c_void_p(X.data_ptr()),
                              ctypes.c_void_p(sd.data_ptr()), ctypes.c_void_p(Bd.data_ptr()), None, None, None,
                              None, n, D, 0.0, fid)
        assert L.API_CheckCUDAError() == 0
        p = speo.Problem([obj], shift.astype(np.float64), M.astype(np.float64))
        speo.evaluate(p, X, g)
        torch.cuda.synchronize()
        np.testing.assert_array_equal(f.cpu().numpy(), g.cpu().numpy())
        p.close()


@pytest.mark.parametrize("prec", range(6))
@pytest.mark.parametrize("n,D", [(1, 2), (33, 30), (100, 128), (5000, 17), (20000, 5), (40000, 64)])
def test_composition_components_in_one_launch(cuda, speo, n, D, prec):
    """A composition of up to 128 columns (its components in one launch) against the
    same sum of its components evaluated as problems of their own: 16, 32 and 64-row
    tiles."""
    import torch
    print(f"n {n} D {D} precision {prec}", flush=True)
    rng = np.random.default_rng([n, D])
    objs = [speo.OBJ_ELLIPTIC, speo.OBJ_RASTRIGIN, speo.OBJ_ACKLEY]
    o = np.float32(rng.uniform(-80, 80, (3, D))).astype(np.float64)
    M = np.stack([np.linalg.qr(rng.standard_normal((D, D)))[0] for _ in objs])
    X = torch.from_numpy(rng.uniform(-100, 100, (n, D)).astype(np.float32)).to(cuda)
    sigma, bias, lam = [10.0, 20.0, 30.0], [0.0, 100.0, 200.0], [1e-6, 1.0, 1.0]
    comp = speo.Problem(objs, o, M, sigma=sigma, bias=bias, lam=lam)
    f, g = torch.zeros(n, device=cuda), torch.zeros(3, n, device=cuda)
    speo.evaluate(comp, X, f, precision=prec)
    for c in range(3):
        p = speo.Problem(objs[c:c + 1], o[c:c + 1], M[c:c + 1], bias=[bias[c]], lam=[lam[c]])
        speo.evaluate(p, X, g[c], precision=prec)
        torch.cuda.synchronize()
        p.close()
    x, g = X.cpu().numpy().astype(np.float64), g.cpu().numpy().astype(np.float64)
    d = ((x[:, None, :] - o[None]) ** 2).sum(2)
    lw = -0.5 * np.log(d) - d / (2.0 * D * np.array(sigma) ** 2)
    w = np.exp(lw - lw.max(1, keepdims=True))
    want = (w * g.T).sum(1) / w.sum(1)
    # The weights' exponents are FP32 sums of D squares up to 4e4 each, so a weight
    # is off by up to (D + 4) 2^-24 times |lw| <= 2e2 relative; the values are sums
    # of non-negative terms and carry it as it is.
    bound = (D + 4) * 2.0 ** -24 * (np.abs(lw).max() + 8)
    np.testing.assert_allclose(f.cpu().numpy(), want, rtol=2 * bound)
    comp.close()


@pytest.mark.parametrize("n,subs,strategy", [(1024, 1, 2), (1040, 1, 3), (2000, 100, 6), (4100, 205, 7), (8192, 1, 2),
                                             (16384, 2, 3), (16400, 1, 6), (32768, 16, 7)])
def test_generation_at_the_lines(cuda, speo, oracle, n, subs, strategy):
    """Either side of the lines between a wave and 16 lanes a row, and between the search
    in the rows' own launch (row blocks x members <= 2^22) and a launch of its own."""
    test_generation_finds_best(cuda, speo, oracle, n, subs, 13, strategy)

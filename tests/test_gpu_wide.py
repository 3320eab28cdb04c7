"""The tile kernel of wide problems (more than 128 columns): its values equal the
64-row kernel's bit for bit (same MFMA chains, same sums) at the edges of its
row blocks, K stages and column chunks, with rows padded by NaN, and the
components of a composition in one launch equal one launch each."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _problem(speo, objs, D, seed, rate=None):
    rng = np.random.default_rng(seed)
    o = np.float32(rng.uniform(-80, 80, (len(objs), D))).astype(np.float64)
    M = np.stack([np.linalg.qr(rng.standard_normal((D, D)))[0] for _ in objs])
    sigma = [10.0 * (c + 1) for c in range(len(objs))]
    return speo.Problem(objs, o, M, sigma=sigma, bias=[100.0 * c for c in range(len(objs))], rate=rate)


def _rows(n, D, ld, cuda):
    import torch
    X = torch.full((n, ld), float("nan"), device=cuda)
    X[:, :D] = torch.rand((n, D), device=cuda, generator=torch.Generator(cuda).manual_seed(n)) * 200 - 100
    return X


# FP32 takes the tile kernel from 160 blocks of 128 rows x 256 columns on
@pytest.mark.parametrize("D,ld,n,prec", [(129, 132, 20481, 0), (160, 160, 21000, 0), (257, 260, 11009, 0),
                                         (1000, 1000, 5249, 0), (1023, 1024, 5120, 0), (129, 132, 1025, 1),
                                         (255, 256, 1151, 3), (257, 300, 1153, 2), (1001, 1004, 1024, 5),
                                         (513, 516, 1279, 4)])
@pytest.mark.parametrize("obj,rate", [(2, 1.0), (6, 0.05)])
def test_tile_kernel_equals_64_row_kernel(cuda, speo, D, ld, n, prec, obj, rate):
    import torch
    prob = _problem(speo, [obj], D, D, rate=[rate])
    X = _rows(n, D, ld, cuda)
    got = {}
    for on in (1, 0):
        prev, before = speo.wide_eval(on)
        f = torch.zeros(n, device=cuda)
        print(f"D={D} n={n} prec={prec} obj={obj} tile kernel {on}", flush=True)
        speo.evaluate(prob, X, f, precision=prec, ld=ld)
        torch.cuda.synchronize()
        assert speo.wide_eval(prev)[1] - before == on
        got[on] = f.cpu().numpy()
    assert np.isfinite(got[1]).all()
    np.testing.assert_array_equal(got[1], got[0])
    prob.close()


@pytest.mark.parametrize("prec", [0, 1, 3])
def test_batched_components_equal_one_launch_each(cuda, speo, prec):
    """speo_evaluate runs a composition's components in one launch;
    speo_evaluate_noalloc's fixed workspace (2^20 floats) is too small for
    that here and takes them one by one."""
    import torch
    D, n = 260, 22016
    prob = _problem(speo, [1, 2, 3, 3, 2, 1, 7], D, 11)
    X = _rows(n, D, D, cuda)
    a, b = torch.zeros(n, device=cuda), torch.zeros(n, device=cuda)
    chunks = -(-D // 128)
    assert n * (2 * chunks + 7) <= 2 ** 20 < 7 * n * (2 * chunks + 1)
    speo.evaluate(prob, X, a, precision=prec)
    speo.evaluate_noalloc(prob, X, b, precision=prec)
    np.testing.assert_array_equal(a.cpu().numpy(), b.cpu().numpy())
    prob.close()


@pytest.mark.parametrize("prec", range(6))
@pytest.mark.parametrize("n,D,extra,shift", [(5, 129, 0, 0), (700, 301, 0, 0), (3000, 515, 0, 0), (3000, 200, 1, 0),
                                             (1500, 256, 0, 1), (9000, 131, 2, 3)])
def test_unaligned_rows_equal_aligned(cuda, speo, n, D, extra, shift, prec):
    """Rows with a stride or a start off 16 bytes, copied first, against the same rows
    aligned (the components' values, single objectives: bit for bit) and against the
    workspace without room for the copy."""
    import torch
    print(f"n {n} D {D} stride +{extra} start +{shift} precision {prec}", flush=True)
    rng = np.random.default_rng([n, D])
    ld, lda = D + extra, (D + 3) // 4 * 4
    X = rng.uniform(-100, 100, (n, D)).astype(np.float32)
    flat = torch.full((n * ld + 8,), float("nan"), device=cuda)
    Xu = flat[shift:shift + n * ld].view(n, ld)
    Xu[:, :D] = torch.from_numpy(X).to(cuda)
    Xa = torch.zeros((n, lda), device=cuda)
    Xa[:, :D] = torch.from_numpy(X).to(cuda)
    for obj in (speo.OBJ_RASTRIGIN, speo.OBJ_DISCUS):
        p = speo.Problem([obj], rng.uniform(-80, 80, (1, D)), np.linalg.qr(rng.standard_normal((D, D)))[0][None])
        f, g, h = (torch.zeros(n, device=cuda) for _ in range(3))
        speo.evaluate(p, Xu, f, precision=prec, ld=ld)
        speo.evaluate(p, Xa, g, precision=prec, ld=lda)
        m = min(n, 2 ** 20 // (2 * ((D + 127) // 128)))
        speo.evaluate_noalloc(p, Xu, h, precision=prec, ld=ld, n=m)
        torch.cuda.synchronize()
        assert torch.isfinite(f).all()
        np.testing.assert_array_equal(f.cpu().numpy(), g.cpu().numpy())
        if m == n:  # (the same rows per block)
            np.testing.assert_array_equal(h.cpu().numpy(), g.cpu().numpy())
        p.close()


@pytest.mark.parametrize("D,start,ld,n,prec", [(132, 64, 196, 20481, 0), (232, 280, 512, 1031, 3), (260, 4, 264, 1153, 1),
                                               (131, 24, 156, 1025, 5)])
def test_column_slices_equal_whole_rows(cuda, speo, D, start, ld, n, prec):
    """Rows that are the last columns of a wider matrix: nothing of the caller's lies
    behind the last row's last column (D = 131: one column of padding)."""
    import torch
    prob = _problem(speo, [2], D, D)
    X = _rows(n, D, D + (-D) % 4, cuda)
    parent = torch.full((n, ld), float("nan"), device=cuda)
    parent[:, start:start + D] = X[:, :D]
    f, g = torch.zeros(n, device=cuda), torch.zeros(n, device=cuda)
    print(f"D={D} columns {start}.. of {ld} n={n} prec={prec}", flush=True)
    before = speo.wide_eval(-1)[1]
    speo.evaluate(prob, parent[:, start:], f, precision=prec, ld=ld, n=n)
    speo.evaluate(prob, X, g, precision=prec, ld=X.shape[1])
    torch.cuda.synchronize()
    assert speo.wide_eval(-1)[1] == before + 2
    assert torch.isfinite(f).all()
    np.testing.assert_array_equal(f.cpu().numpy(), g.cpu().numpy())
    prob.close()


def test_stride_beyond_31_bit_offsets(cuda, speo):
    """A tile of 128 rows 2^22 floats apart does not fit 31-bit byte offsets: the 64-row
    kernel takes such rows, with the values of the same rows side by side."""
    import torch
    D, n, ld = 160, 1030, 2 ** 22
    prob = _problem(speo, [2], D, D)
    X = _rows(n, D, D, cuda)
    far = torch.empty((n, ld), device=cuda)
    far[:, :D] = X
    f, g = torch.zeros(n, device=cuda), torch.zeros(n, device=cuda)
    print(f"D={D} n={n} ld={ld}", flush=True)
    speo.evaluate(prob, far, f, precision=speo.PREC_BF16, ld=ld)
    speo.evaluate(prob, X, g, precision=speo.PREC_BF16)
    torch.cuda.synchronize()
    np.testing.assert_array_equal(f.cpu().numpy(), g.cpu().numpy())
    prob.close()


@pytest.mark.parametrize("objs", [[2], [1, 2, 3]])
def test_odd_rows_under_capture_after_aligned_ones(cuda, speo, objs):
    """An evaluation that a first call on aligned rows has prepared can be captured for
    rows of an odd stride (they are not copied then), and a captured evaluation of
    aligned rows outlives a later call on odd ones."""
    import torch
    D, n = 301, 700
    prob = _problem(speo, objs, D, 5)
    Xo = _rows(n, D, D, cuda)
    Xa = torch.zeros((n, 304), device=cuda)
    Xa[:, :D] = Xo
    fo, fa, g, h = (torch.zeros(n, device=cuda) for _ in range(4))
    s = torch.cuda.Stream()
    with torch.cuda.stream(s):
        speo.evaluate(prob, Xa, h, stream=s)
        s.synchronize()
        graphs = []
        for X, f in ((Xo, fo), (Xa, fa)):
            graph = torch.cuda.CUDAGraph()
            with torch.cuda.graph(graph, stream=s):
                speo.evaluate(prob, X, f, stream=s)
            graphs.append(graph)
    torch.cuda.synchronize()
    for rep in range(4):
        print(f"replay {rep}", flush=True)
        X = _rows(n, D, D, cuda) * (1.0 - 0.125 * rep)
        Xo.copy_(X)
        Xa[:, :D] = X
        for graph in graphs:
            graph.replay()
        torch.cuda.synchronize()
        speo.evaluate(prob, Xo, g)  # eager, with the copy
        speo.evaluate(prob, Xa, h)
        torch.cuda.synchronize()
        np.testing.assert_array_equal(fo.cpu().numpy(), g.cpu().numpy())
        np.testing.assert_array_equal(fa.cpu().numpy(), h.cpu().numpy())
    del graphs
    prob.close()

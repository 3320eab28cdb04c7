"""A plain engine's run of several generations (one launch a generation, the last
selection after it, donors drawn ahead) leaves what its separate generate,
evaluate and select launches leave: population, fitness, the last trials and
their fitness, bit for bit.  Odd and even lengths, the 64-generation limit of the
donors drawn at once, migrations inside a run, eager and replayed."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _problems(speo, dims):
    rng = np.random.default_rng(5)
    out = []
    for D, objs in dims:
        o = np.float32(rng.uniform(-80, 80, (len(objs), D))).astype(np.float64)
        M = np.stack([np.linalg.qr(rng.standard_normal((D, D)))[0] for _ in objs])
        out.append(speo.Problem(objs, o, M, sigma=[10.0 * (c + 1) for c in range(len(objs))],
                                bias=[100.0 * c for c in range(len(objs))]))
    return out


@pytest.mark.parametrize("lengths,interval,graph,dims", [
    ((1, 2, 3), 0, 0, [(10, [2]), (7, [3])]),
    ((1, 1, 4), 2, 0, [(10, [2]), (128, [1])]),
    ((64, 1), 0, 1, [(9, [3]), (30, [1, 2])]),
    ((65, 65), 0, 0, [(9, [3]), (30, [1, 2])]),
    ((130, 130), 50, 1, [(5, [2]), (33, [5])]),
    ((2, 3), 2, 0, [(129, [2]), (40, [3])]),
])
def test_run_equals_separate_launches(cuda, speo, lengths, interval, graph, dims):
    probs = _problems(speo, dims)
    kw = dict(seed=3, interval=interval, migration_size=2 if interval else 0, mode=speo.MODE_PLAIN,
              rows_per_block=32)
    sizes, which = [31, 64, 100, 8], [0, 1, 0, 1]
    a = speo.Engine(probs, sizes, which, use_graph=bool(graph), **kw)
    b = speo.Engine(probs, sizes, which, use_graph=False, **kw)
    for L in lengths:
        print(f"generations {L} interval {interval} graph {graph} dims {dims}", flush=True)
        a.run(L)
        b.profile(L)
        for x, y in zip(a.read() + a.read_trials(), b.read() + b.read_trials()):
            np.testing.assert_array_equal(x, y)
    assert a.best()[1].tolist() == b.best()[1].tolist()
    for o in [a, b] + probs:
        o.close()


@pytest.mark.parametrize("sizes,k", [([4100, 8, 4097], 4), ([63, 64, 65, 130], 3), ([1000, 257], 128)])
def test_migration_ranks(cuda, speo, oracle, sizes, k):
    """Migration by rank against the oracle: more rows than one LDS pass, edges of a
    block's rows, half an island moving; ties, both zeros, infinities and NaN."""
    print(f"sizes {sizes} migrants {k}", flush=True)
    probs = _problems(speo, [(6, [2])])
    kw = dict(seed=3, mode=speo.MODE_PLAIN, rows_per_block=32)
    which = [0] * len(sizes)
    n = sum(sizes)
    rng = np.random.default_rng(n)
    f = rng.integers(-3, 3, n).astype(np.float32)  # trials never beat values this low; many ties
    f[rng.random(n) < 0.1] = -0.0
    f[rng.random(n) < 0.1] = np.nan
    f[rng.random(n) < 0.05] = -np.inf
    out = []
    for interval in (0, 1):
        e = speo.Engine(probs, sizes, which, interval=interval, migration_size=min(k, min(sizes) // 2), **kw)
        X, _ = e.read()
        e.write(X, f)
        e.run(1)
        out.append(e.read())
        e.close()
    X, f1 = out[0]
    off = np.concatenate([[0], np.cumsum(sizes)]).astype(np.int32)
    dst = np.array([(i + 1) % len(sizes) for i in range(len(sizes))], np.int32)
    Xo, fo = oracle.migrate_ring(X, f1, X.shape[1], off, np.full(len(sizes), 6, np.int32), dst,
                                 min(k, min(sizes) // 2))
    np.testing.assert_array_equal(out[1][1], fo)
    np.testing.assert_array_equal(out[1][0], Xo)
    for p in probs:
        p.close()


@pytest.mark.parametrize("mode", ["PLAIN", "FUSED"])
@pytest.mark.parametrize("islands,rows,D,interval", [(1024, 1024, 10, 0), (512, 1024, 60, 2), (4, 100, 5, 0)])
def test_donor_memory_in_proportion(cuda, speo, mode, islands, rows, D, interval):
    """An engine's device memory beyond its three population arrays: at most one more of
    them, or 64 MiB, for the donors drawn ahead, none past a migration point, and the
    tables and fitness arrays."""
    import torch
    prob, = _problems(speo, [(D, [2])])
    torch.cuda.synchronize()
    free0 = torch.cuda.mem_get_info()[0]
    e = speo.Engine([prob], [rows] * islands, [0] * islands, mode=getattr(speo, "MODE_" + mode), seed=3,
                    rows_per_block=32, interval=interval, migration_size=2 if interval else 0)
    taken = free0 - torch.cuda.mem_get_info()[0]
    print(f"{mode} {islands} x {rows} D {D}: {taken / 2 ** 20:.0f} MiB", flush=True)
    R = islands * rows
    population = 4 * R * ((D + 3) // 4 * 4)
    donors = 16 * R * interval if interval else min(16 * R * 64, max(population, 64 << 20))
    # per row: four fitness values, the row's island, a share of two tile tables (64 bytes
    # a tile of at least 16 rows); 32 MiB for what the allocator rounds up
    assert taken < 3 * population + donors + R * (16 + 4 + 8) + (32 << 20)
    e.run(5)
    e.sync()
    e.close()
    prob.close()


def test_row_tile_chosen_for_the_kernel_that_runs(cuda, speo, tmp_path, monkeypatch):
    """rows_per_block = 0: a plain engine's tile is timed by the fused launches that its
    runs consist of, under a name of its own; engines whose generations are separate
    launches keep the other.  Stored choices are taken, and change no result."""
    cache = tmp_path / "tune.txt"
    monkeypatch.setenv("SPEO_TUNE_CACHE", str(cache))
    probs = _problems(speo, [(21, [2])])
    kw = dict(seed=3, mode=speo.MODE_PLAIN)
    shape = "m0:p0:n3:21/64*3"
    cache.write_text(f"rt:{shape} 64\n")  # timed by the evaluation kernel, under the earlier name
    a = speo.Engine(probs, [50, 51, 52], [0] * 3, **kw)
    b = speo.Engine(probs, [50, 51, 52], [0] * 3, **dict(kw, rows_per_block=16))
    assert [ln.split()[0] for ln in cache.read_text().splitlines()] == [f"rt:{shape}", f"rt_plain:{shape}"]
    speo.Engine(probs, [48, 44, 52], [0] * 3, strategy=6, **kw).close()
    assert len(cache.read_text().splitlines()) == 2
    for e in (a, b):
        e.run(9)
    for x, y in zip(a.read() + a.read_trials(), b.read() + b.read_trials()):
        np.testing.assert_array_equal(x, y)
    for o in [a, b] + probs:
        o.close()
    cache.write_text("rt_plain:m0:p0:n3:22/64*3 64\n")
    p22 = _problems(speo, [(22, [2])])
    e = speo.Engine(p22, [50, 51, 52], [0] * 3, **kw)
    assert e.stats()["rows_per_block"] == 64
    e.close()
    p22[0].close()

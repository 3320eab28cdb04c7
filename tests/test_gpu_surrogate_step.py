"""Screened generations: the one-kernel screening (donors drawn ahead, candidates
made by all lanes) gives the trials of the written-out candidates, and the
evaluation's own append and selection leave the archive and population that the
trials and their values say.  Widths of one group of four columns and of a full
network tile, islands off the 32-row tile, more tiles than one draw covers."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _engine(speo, D, sizes, C, steps=5):
    rng = np.random.default_rng(D)
    probs = []
    for obj in (2, 1):
        o = np.float32(rng.uniform(-80, 80, (1, D))).astype(np.float64)
        M = np.linalg.qr(rng.standard_normal((D, D)))[0][None]
        probs.append(speo.Problem([obj], o, M))
    e = speo.Engine(probs, sizes, [i % 2 for i in range(len(sizes))], F=0.5, CR=0.9, seed=11, mode=speo.MODE_PLAIN,
                    rows_per_block=32, surrogate_candidates=C, surrogate_train_interval=4, surrogate_archive=8192,
                    surrogate_steps=steps, surrogate_batch=256, surrogate_lr=1e-3, surrogate_rho_min=-1.5)
    return probs, e


@pytest.mark.parametrize("D,sizes,C", [(4, [300, 257], 3), (30, [31, 65, 600, 512], 5), (128, [333, 512], 8),
                                       (100, [4000, 4100, 2000, 2100], 32)])
def test_screening_and_append(cuda, speo, D, sizes, C):
    ends = []
    for dump_first in (False, True):  # True: candidates written out, the pick copied
        probs, e = _engine(speo, D, sizes, C)
        if dump_first:
            e.surrogate_dump(0, C, 8192)
        for g in range(6):  # the networks screen from generation 4 on
            print(f"D {D} sizes {sizes} candidates {C} written {dump_first} generation {g}", flush=True)
            X0, f0 = e.read()
            e.run(1)
            U, fU = e.read_trials()
            X, f = e.read()
            acc = fU < f0
            np.testing.assert_array_equal(f, np.where(acc, fU, f0))
            np.testing.assert_array_equal(X, np.where(acc[:, None], U, X0))
        assert e.stats()["surrogate_rounds"] == 1
        if dump_first:
            row0 = np.concatenate([[0], np.cumsum(sizes)])
            for p in (0, 1):
                q = np.concatenate([np.arange(row0[i], row0[i + 1]) for i in range(len(sizes)) if i % 2 == p])
                _, _, _, AX, Ay, head, _ = e.surrogate_dump(p, C, 8192)
                slots = (head - len(q) + np.arange(len(q))) % 8192
                np.testing.assert_array_equal(AX[slots, :D], U[q])
                assert not AX[slots, D:].any()
                # log1pf within 2 ulp
                np.testing.assert_allclose(Ay[slots], np.log1p(np.maximum(fU[q].astype(np.float64), 0)), rtol=3e-7)
        ends.append((X, f, U, fU))
        e.close()
        for p in probs:
            p.close()
    for a, b in zip(*ends):
        np.testing.assert_array_equal(a, b)


def test_profile_of_a_screened_engine(cuda, speo):
    probs, e = _engine(speo, 30, [64, 64], 3)
    ms = e.profile(2)
    assert ms["generate"] > 0 and ms["select"] > 0
    e.close()
    for p in probs:
        p.close()

"""What a user of this framework has it do, as measurable cases.

A case is a dict of plain values; ``kind`` says which public entry points a
pass goes through:

  evolve     an island engine: some generations, then each island's best
             (what a program that follows a run's convergence calls)
  surrogate  the same with the learned screen: one training round per pass
  evaluate   objective values of a batch of rows (FP32 result)
  verify     the FP64 values of a batch of rows
  dropin     one generation cycle through the five drop-in C entry points
"""
import math
import sys
from ctypes import byref, c_void_p
from pathlib import Path

import numpy as np
import torch

_PKG = str(Path(__file__).resolve().parent.parent / "speo-gpu-single-control_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

import speo_de as S  # noqa: E402

LO, HI = -100.0, 100.0
PRECISIONS = {name: code for code, name in S.PREC_NAMES.items()}
MODES = {"plain": S.MODE_PLAIN, "fused": S.MODE_FUSED, "epoch": S.MODE_EPOCH}

# CEC2014's input rates of the objectives (1 where not listed).
RATES = {S.OBJ_RASTRIGIN: 0.0512, S.OBJ_HAPPYCAT: 0.05, S.OBJ_HGBAT: 0.05, S.OBJ_SCHWEFEL: 10.0,
         S.OBJ_ROSENBROCK: 0.02048, S.OBJ_WEIERSTRASS: 0.005, S.OBJ_GRIEWANK: 6.0,
         S.OBJ_KATSUURA: 0.05, S.OBJ_GRIE_ROSEN: 0.05}
# The drop-in call's function numbers that are one objective or one hybrid.
FUNCTIONS = {1: S.OBJ_ELLIPTIC, 2: S.OBJ_BENT_CIGAR, 3: S.OBJ_DISCUS, 4: S.OBJ_ROSENBROCK,
             5: S.OBJ_ACKLEY, 6: S.OBJ_WEIERSTRASS, 7: S.OBJ_GRIEWANK, 9: S.OBJ_RASTRIGIN,
             12: S.OBJ_KATSUURA, 13: S.OBJ_HAPPYCAT, 14: S.OBJ_HGBAT, 15: S.OBJ_GRIE_ROSEN,
             16: S.OBJ_ESCAFFER6, 17: S.OBJ_HYBRID_1, 18: S.OBJ_HYBRID_2, 19: S.OBJ_HYBRID_3,
             20: S.OBJ_HYBRID_4, 21: S.OBJ_HYBRID_5, 22: S.OBJ_HYBRID_6}
FUSED_OBJECTIVES = (S.OBJ_ELLIPTIC, S.OBJ_RASTRIGIN, S.OBJ_ACKLEY, S.OBJ_BENT_CIGAR, S.OBJ_DISCUS,
                    S.OBJ_HAPPYCAT, S.OBJ_HGBAT)
FP64_OBJECTIVES = (S.OBJ_ROSENBROCK, S.OBJ_WEIERSTRASS, S.OBJ_GRIEWANK, S.OBJ_KATSUURA,
                   S.OBJ_GRIE_ROSEN, S.OBJ_ESCAFFER6, S.OBJ_HYBRID_1, S.OBJ_HYBRID_2, S.OBJ_HYBRID_3,
                   S.OBJ_HYBRID_4, S.OBJ_HYBRID_5, S.OBJ_HYBRID_6)
# Segment shares, objectives and rates of the hybrid functions.
HYBRIDS = {
    S.OBJ_HYBRID_1: ((0.3, 0.3, 0.4), (S.OBJ_SCHWEFEL, S.OBJ_RASTRIGIN, S.OBJ_ELLIPTIC),
                     (10.0, 0.0512, 1.0)),
    S.OBJ_HYBRID_2: ((0.3, 0.3, 0.4), (S.OBJ_BENT_CIGAR, S.OBJ_HGBAT, S.OBJ_RASTRIGIN),
                     (1.0, 0.05, 0.0512)),
    S.OBJ_HYBRID_3: ((0.2, 0.2, 0.3, 0.3),
                     (S.OBJ_GRIEWANK, S.OBJ_WEIERSTRASS, S.OBJ_ROSENBROCK, S.OBJ_ESCAFFER6),
                     (6.0, 0.005, 0.02048, 1.0)),
    S.OBJ_HYBRID_4: ((0.2, 0.2, 0.3, 0.3),
                     (S.OBJ_HGBAT, S.OBJ_DISCUS, S.OBJ_GRIE_ROSEN, S.OBJ_RASTRIGIN),
                     (0.05, 1.0, 0.05, 0.0512)),
    S.OBJ_HYBRID_5: ((0.1, 0.2, 0.2, 0.2, 0.3),
                     (S.OBJ_ESCAFFER6, S.OBJ_HGBAT, S.OBJ_ROSENBROCK, S.OBJ_SCHWEFEL, S.OBJ_ELLIPTIC),
                     (1.0, 0.05, 0.02048, 10.0, 1.0)),
    S.OBJ_HYBRID_6: ((0.1, 0.2, 0.2, 0.2, 0.3),
                     (S.OBJ_KATSUURA, S.OBJ_HAPPYCAT, S.OBJ_GRIE_ROSEN, S.OBJ_SCHWEFEL, S.OBJ_ACKLEY),
                     (0.05, 0.05, 0.05, 10.0, 1.0)),
}


def listed():
    return [
        # The smallest run: one island of the classic NP = 100, D = 10, each
        # generation launched by itself.  Launches and the read of the best
        # count here.
        dict(name="one_island_d10", kind="evolve", mode="plain", graph=False, islands=1, rows=100,
             dims="10", objectives="2", precision="fp32", interval=0, generations=10, tile=0),
        # The benchmark's own run: 64 islands x 128, D = 100, one migration
        # interval of the batched engine under graphs.
        dict(name="islands_64x128_d100", kind="evolve", mode="epoch", graph=True, islands=64, rows=128,
             dims="100", objectives="1,2,3", precision="fp32", interval=50, generations=50, tile=0),
        # Uneven islands (D 10 to 100, NP 50 to 512), one launch a generation.
        dict(name="uneven_256_islands", kind="evolve", mode="fused", graph=True, islands=256, rows=0,
             dims="10,30,50,100", objectives="1,2,3", precision="fp32", interval=25, generations=25,
             tile=0),
        # The large-dimension study as a run: 8 islands x 2048 rows, D = 1000,
        # a composition of three functions, split-BF16 rotation.
        dict(name="islands_8x2048_d1000", kind="evolve", mode="fused", graph=False, islands=8, rows=2048,
             dims="1000", objectives="c1,2,3", precision="bf16x3", interval=50, generations=2, tile=64),
        # Surrogate-assisted run, 32 islands x 256, D = 100: ten screened
        # generations and the training round that follows them.
        dict(name="surrogate_32x256_d100", kind="surrogate", islands=32, rows=256, dim=100,
             precision="bf16x3", candidates=8, interval=10, archive=65536, steps=40, batch=1024),
        # The smallest evaluation call: one small population.
        dict(name="eval_100x10_fp32", kind="evaluate", n=100, dim=10, objectives="3", precision="fp32"),
        # An ordinary batch at the benchmark's dimension.
        dict(name="eval_8192x100_fp32", kind="evaluate", n=8192, dim=100, objectives="2", precision="fp32"),
        # The precision study's batch: 16,384 rows of a three-function
        # composition at D = 1000, in FP32 and with the plain 16-bit rotation.
        dict(name="eval_16384x1000_fp32", kind="evaluate", n=16384, dim=1000, objectives="1,2,3",
             precision="fp32"),
        dict(name="eval_16384x1000_bf16", kind="evaluate", n=16384, dim=1000, objectives="1,2,3",
             precision="bf16"),
        # A CEC2014 composition (F26) on the published runs' population:
        # objectives that need FP64 throughout.
        dict(name="eval_cec_f26_4096x100", kind="evaluate", n=4096, dim=100, objectives="8,6,1,10,11",
             precision="fp32"),
        # FP64 values of the points of a precision study.
        dict(name="verify_2048x250", kind="verify", n=2048, dim=250, objectives="1,2,3"),
        # A reference host's generation: the drop-in calls on its default
        # island of 1024 rows.
        dict(name="dropin_f9_1024x100", kind="dropin", n=1024, dim=100, function=9, subislands=1, strategy=4),
    ]


def _spread(rng, lo, hi):
    """A whole number of [lo, hi], even over its logarithm."""
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(("evolve", "evolve", "evolve_wide", "surrogate", "evaluate", "evaluate", "evaluate_wide",
                       "evaluate_fp64", "verify", "dropin"))
    if kind == "evolve":
        # up to the uneven batch's 72,000 rows; any of the three modes
        mode = rng.choice(("plain", "fused", "epoch"))
        islands, rows = _spread(rng, 1, 128), _spread(rng, 16, 512)
        dims = ",".join(str(_spread(rng, 5, 128)) for _ in range(rng.randint(1, 3)))
        objectives = ",".join(str(rng.choice((1, 2, 3, 4, 5))) for _ in range(rng.randint(1, 3)))
        return dict(kind="evolve", mode=mode, graph=rng.random() < 0.6, islands=islands, rows=rows,
                    dims=dims, objectives=objectives,
                    precision=rng.choice(("fp32", "fp32", "bf16x3", "bf16", "fp16x3")),
                    interval=rng.choice((0, 10, 25)), generations=_spread(rng, 5, 40), tile=0)
    if kind == "evolve_wide":
        return dict(kind="evolve", mode=rng.choice(("plain", "fused")), graph=False,
                    islands=rng.randint(1, 8), rows=_spread(rng, 64, 2048),
                    dims=str(_spread(rng, 129, 1000)), objectives=rng.choice(("1", "2", "3", "c1,2", "c1,2,3")),
                    precision=rng.choice(("fp32", "bf16", "bf16x3", "fp16x3")), interval=50,
                    generations=rng.randint(1, 2), tile=rng.choice((16, 32, 64)))
    if kind == "surrogate":
        return dict(kind="surrogate", islands=2 * rng.randint(4, 16), rows=rng.randint(64, 256),
                    dim=_spread(rng, 20, 100), precision=rng.choice(("fp32", "bf16x3")),
                    candidates=rng.randint(2, 8), interval=10, archive=16384,
                    steps=rng.randint(10, 40), batch=rng.choice((256, 512, 1024)))
    if kind == "evaluate":
        return dict(kind="evaluate", n=_spread(rng, 1, 65536), dim=_spread(rng, 2, 128),
                    objectives=_fused_objectives(rng), precision=_any_precision(rng))
    if kind == "evaluate_wide":
        return dict(kind="evaluate", n=_spread(rng, 64, 16384), dim=_spread(rng, 129, 1000),
                    objectives=_fused_objectives(rng), precision=_any_precision(rng))
    if kind == "evaluate_fp64":
        count = rng.choice((1, 1, 3, 5))
        objectives = [rng.choice(FP64_OBJECTIVES)] + [rng.choice(FUSED_OBJECTIVES + FP64_OBJECTIVES)
                                                      for _ in range(count - 1)]
        return dict(kind="evaluate", n=_spread(rng, 1, 8192), dim=_spread(rng, 20, 128),
                    objectives=",".join(map(str, objectives)), precision="fp32")
    if kind == "verify":
        return dict(kind="verify", n=_spread(rng, 1, 2048), dim=_spread(rng, 2, 250),
                    objectives=_fused_objectives(rng))
    subislands = rng.choice((1, 1, 4, 16))
    return dict(kind="dropin", n=16 * subislands * _spread(rng, 1, 4096 // (16 * subislands)),
                dim=_spread(rng, 20, 128), function=rng.choice(sorted(FUNCTIONS)), subislands=subislands,
                strategy=rng.choice((4, 4, 4, 0, 1, 2, 3, 5, 6, 7, 8)))


def _fused_objectives(rng):
    return ",".join(str(rng.choice(FUSED_OBJECTIVES)) for _ in range(rng.choice((1, 1, 3))))


def _any_precision(rng):
    return rng.choice(("fp32", "fp32", "bf16", "fp16", "bf16x3", "fp16x3", "bf16x6"))


# --------------------------------------------------------------- problem data

def _numbers(text):
    return [int(v) for v in text.split(",")]


def _rotation(rng, dim):
    """A Haar-random rotation: Q of a Gaussian matrix, signs fixed by R's diagonal."""
    q, r = np.linalg.qr(rng.standard_normal((dim, dim)))
    return q * np.where(np.diag(r) < 0, -1.0, 1.0)


def _data(seed, objectives, dim):
    """Shift, rotation, rate, sigma, bias, lambda and shuffle of a problem."""
    rng = np.random.default_rng([seed, dim, len(objectives)])
    nc = len(objectives)
    d = {"objectives": objectives, "dim": dim}
    d["shift"] = np.float32(rng.uniform(-80, 80, (nc, dim))).astype(np.float64)
    d["rotation"] = np.stack([_rotation(rng, dim) for _ in range(nc)])
    d["shuffle"] = np.stack([rng.permutation(dim) + 1 for _ in range(nc)]).astype(np.int32)
    d["rate"] = np.array([RATES.get(o, 1.0) for o in objectives])
    d["sigma"] = np.array([10.0 * (c + 1) for c in range(nc)])
    d["bias"] = np.array([100.0 * c for c in range(nc)]) if nc > 1 else np.zeros(1)
    # the compositions scale their objectives to a common range
    d["lam"] = np.array([1e-6 if o in (S.OBJ_ELLIPTIC, S.OBJ_BENT_CIGAR, S.OBJ_DISCUS) else 1.0
                         for o in objectives]) if nc > 1 else np.ones(1)
    return d


def _problem(d):
    hybrid = any(o in HYBRIDS for o in d["objectives"])
    return S.Problem(d["objectives"], d["shift"], d["rotation"], sigma=d["sigma"], bias=d["bias"],
                     lam=d["lam"], rate=d["rate"], shuffle=d["shuffle"] if hybrid else None)


def _rows(seed, n, dim):
    g = torch.Generator(device="cuda").manual_seed(seed)
    return torch.rand((n, dim), generator=g, device="cuda", dtype=torch.float32) * (HI - LO) + LO


# ------------------------------------------------------------------- prepare

def _islands(case, seed):
    """(problems, island sizes, island -> problem) of an evolve case."""
    composed = case["objectives"].startswith("c")
    objectives = _numbers(case["objectives"].lstrip("c"))
    dims = _numbers(case["dims"])
    rng = np.random.default_rng(case["islands"])  # the shapes belong to the case, the data to the seed
    index, problems, which, sizes = {}, [], [], []
    for i in range(case["islands"]):
        dim = dims[int(rng.integers(len(dims)))]
        key = (dim, -1 if composed else i % len(objectives))
        if key not in index:
            index[key] = len(problems)
            objs = objectives if composed else [objectives[key[1]]]
            d = _data(seed * 1000 + len(problems), objs, dim)
            if composed:
                d["lam"] = np.ones(len(objs))
            else:
                d["rate"] = np.ones(1)
            problems.append(_problem(d))
        which.append(index[key])
        sizes.append(case["rows"] or int(rng.integers(50, 513)))
    return problems, sizes, which


def prepare(case, seed):
    state = {"case": case}
    if case["kind"] == "evolve":
        problems, sizes, which = _islands(case, seed)
        engine = S.Engine(problems, sizes, which, F=0.5, CR=0.9, lo=LO, hi=HI, seed=seed,
                          interval=case["interval"], migration_size=2 if case["interval"] else 0,
                          precision=PRECISIONS[case["precision"]], mode=MODES[case["mode"]],
                          use_graph=case["graph"], rows_per_block=case["tile"])
        engine.prepare(case["generations"])
        state.update(engine=engine, problems=problems, views={})
    elif case["kind"] == "surrogate":
        problems = [_problem(_data(seed * 1000 + k, [obj], case["dim"]))
                    for k, obj in enumerate((S.OBJ_RASTRIGIN, S.OBJ_ELLIPTIC))]
        # The threshold below every correlation: both networks screen every
        # generation, as they do in the part of a run where they help.
        engine = S.Engine(problems, [case["rows"]] * case["islands"],
                          [i % 2 for i in range(case["islands"])], F=0.5, CR=0.9, seed=seed, interval=50,
                          migration_size=2, precision=PRECISIONS[case["precision"]], mode=S.MODE_PLAIN,
                          use_graph=True, rows_per_block=32, surrogate_candidates=case["candidates"],
                          surrogate_train_interval=case["interval"], surrogate_archive=case["archive"],
                          surrogate_steps=case["steps"], surrogate_batch=case["batch"],
                          surrogate_lr=1e-3, surrogate_rho_min=-1.5)
        # full archives: from here on a round is one graph
        per_generation = case["rows"] * case["islands"] // 2
        rounds = -(-case["archive"] // per_generation // case["interval"]) + 1
        engine.run(rounds * case["interval"])
        engine.sync()
        state.update(engine=engine, problems=problems, views={})
    elif case["kind"] in ("evaluate", "verify"):
        state["problem"] = _problem(_data(seed, _numbers(case["objectives"]), case["dim"]))
        state["X"] = _rows(seed, case["n"], case["dim"])
        state["f"] = torch.zeros(case["n"], device="cuda",
                                 dtype=torch.float64 if case["kind"] == "verify" else torch.float32)
    else:
        _prepare_dropin(case, seed, state)
    return state


def _prepare_dropin(case, seed, state):
    """The device buffers of a reference host: rows padded to a power of two,
    M transposed and row-padded, one DEInfo per sub-island."""
    n, dim, subs = case["n"], case["dim"], case["subislands"]
    L = S.lib()
    ld = L.SPEO_NextPow2Dim(dim)
    d = _data(seed, [FUNCTIONS[case["function"]]], dim)
    shift = np.zeros(ld, np.float32)
    shift[:dim] = d["shift"][0]
    rotation = np.zeros((ld, dim), np.float32)
    rotation[:dim] = d["rotation"][0].T
    shuffle = np.zeros(ld, np.int32)
    shuffle[:dim] = d["shuffle"][0]
    perm = np.random.default_rng([seed, n]).permutation(n).astype(np.int32)
    info = np.frombuffer(S.de_info_bytes([0.9] * subs, 0.5, case["strategy"]), np.uint8).copy()
    on_gpu = lambda a: torch.from_numpy(a).cuda()  # noqa: E731
    buf = dict(pop=torch.zeros((n, ld), device="cuda"), cand=torch.zeros((n, ld), device="cuda"),
               rotated=torch.zeros((n, ld), device="cuda"), fpop=torch.zeros(n, device="cuda"),
               fcand=torch.zeros(n, device="cuda"), best=torch.zeros(subs, dtype=torch.int32, device="cuda"),
               shift=on_gpu(shift), rotation=on_gpu(rotation), shuffle=on_gpu(shuffle), perm=on_gpu(perm),
               info=on_gpu(info), sigma=torch.full((1,), 10.0, device="cuda"))
    state["buf"] = buf
    state["P"] = S.GPU_Population(buf["pop"].data_ptr(), buf["fpop"].data_ptr())
    state["C"] = S.GPU_Population(buf["cand"].data_ptr(), buf["fcand"].data_ptr())
    state["island"] = S.GPU_IslandInfo(n, subs, buf["perm"].data_ptr())
    state["rand"] = S.SPEO_RandState()
    state["pi"] = S.ProblemInfo(dim, case["function"], 1, 10000, seed, 0, 0, HI, LO)
    S.check(L.API_Initilize(state["P"], byref(state["rand"]), state["island"], state["pi"]))
    _dropin_evaluate(state, "pop", "fpop")
    S.check(L.API_CheckCUDAError())


def _dropin_evaluate(state, rows, values):
    b, case = state["buf"], state["case"]
    ptr = lambda name: c_void_p(b[name].data_ptr())  # noqa: E731
    S.lib().API_evaluateFitness(ptr(values), None, ptr("rotated"), ptr(rows), ptr("shift"), ptr("rotation"),
                                ptr("shuffle"), None, None, ptr("sigma"), case["n"], case["dim"], 0.0,
                                case["function"])


# ----------------------------------------------------------------------- run

class _DeviceArray:
    """`count` floats of an engine's memory; keeps the engine while a tensor looks at them."""

    def __init__(self, engine, pointer, count):
        self.engine = engine
        self.__cuda_array_interface__ = {"shape": (count,), "typestr": "<f4", "data": (pointer, False),
                                         "version": 3}


def _population(state):
    """The engine's device rows and fitness (its own buffers)."""
    e = state["engine"]
    X, f = c_void_p(), c_void_p()
    S.check(S.lib().speo_engine_buffers(e.handle, byref(X), byref(f), None, None, None))
    if "elements" not in state:
        ld = np.zeros(e.num_islands, np.int32)
        S.check(S.lib().speo_engine_buffers(e.handle, None, None, None, None, ld.ctypes.data_as(c_void_p)))
        state["elements"] = int((ld.astype(np.int64) * e.island_size).sum())
    views = state["views"]
    for pointer, count in ((X.value, state["elements"]), (f.value, e.total_rows)):
        if pointer not in views:
            views[pointer] = torch.as_tensor(_DeviceArray(e, pointer, count), device="cuda")
    return views[X.value], views[f.value]


def run(state):
    case = state["case"]
    if case["kind"] in ("evolve", "surrogate"):
        e = state["engine"]
        e.run(case["generations"] if case["kind"] == "evolve" else case["interval"])
        rows, f32, f64 = e.best()
        return {"best_row": rows, "best_f32": f32, "best_f64": f64, "population": _population(state)}
    if case["kind"] == "evaluate":
        S.evaluate(state["problem"], state["X"], state["f"], precision=PRECISIONS[case["precision"]])
        return state["f"]
    if case["kind"] == "verify":
        S.evaluate_f64(state["problem"], state["X"], state["f"])
        return state["f"]
    L, b = S.lib(), state["buf"]
    S.check(L.API_DE_GenerateNewPopulation(state["C"], state["P"], c_void_p(b["best"].data_ptr()),
                                           state["island"], c_void_p(b["info"].data_ptr()),
                                           byref(state["rand"]), state["pi"]))
    _dropin_evaluate(state, "cand", "fcand")
    S.check(L.API_DE_SelectSurvival(state["P"], state["C"], state["island"], state["pi"]))
    return [b[k] for k in ("pop", "fpop", "cand", "fcand", "best")]


# ---------------------------------------------------------------------- work

def work(case):
    kind = case["kind"]
    if kind in ("evaluate", "verify"):
        n, d, nc = case["n"], case["dim"], len(_numbers(case["objectives"]))
        out, m = (8, 8) if kind == "verify" else (4, 4)
        return {"bytes": 4.0 * n * d + out * n + nc * m * d * (d + 1), "flops": 2.0 * n * d * d * nc}
    if kind == "dropin":
        n, d = case["n"], case["dim"]
        # the population read and written, the candidates written, the fitness arrays
        return {"bytes": 4.0 * (3 * n * d + 3 * n + d * (d + 1)), "flops": 2.0 * n * d * d}
    if kind == "surrogate":
        rows, d, g = case["islands"] * case["rows"], case["dim"], case["interval"]
        weights = d * 256 + 256 * 256 + 256
        flops = g * rows * (2.0 * d * d + case["candidates"] * 2.0 * weights)
        flops += 2 * case["steps"] * case["batch"] * 6.0 * weights
        # population in and out, the archive rows the round writes and its minibatches read
        nbytes = 4.0 * (2 * rows * (d + 1) + g * rows * (d + 1) + 2 * case["steps"] * case["batch"] * (d + 1))
        return {"bytes": nbytes, "flops": flops}
    dims = _numbers(case["dims"])
    composed = case["objectives"].startswith("c")
    nc = len(_numbers(case["objectives"].lstrip("c"))) if composed else 1
    np_mean = case["rows"] or 281
    rows = case["islands"] * np_mean
    d1, d2 = sum(dims) / len(dims), sum(d * d for d in dims) / len(dims)
    return {"bytes": 4.0 * (2 * rows * (d1 + 1) + nc * sum(d * (d + 1) for d in dims)),
            "flops": 2.0 * case["generations"] * rows * d2 * nc}


# --------------------------------------------------------------------- exact

def exact(case, seed):
    """The objective values in FP64 with plain torch (evaluations only)."""
    if case["kind"] not in ("evaluate", "verify"):
        return None
    d = _data(seed, _numbers(case["objectives"]), case["dim"])
    x = _rows(seed, case["n"], case["dim"]).double()
    at = lambda a: torch.from_numpy(np.ascontiguousarray(a)).cuda()  # noqa: E731
    fits, logw = [], []
    for c, objective in enumerate(d["objectives"]):
        v = x - at(d["shift"][c])
        z = (v * float(d["rate"][c])) @ at(d["rotation"][c].T)
        if objective in HYBRIDS:
            g = _hybrid(objective, z[:, at(d["shuffle"][c].astype(np.int64) - 1)])
        else:
            g = _objective(objective, z)
        fits.append(float(d["lam"][c]) * g + float(d["bias"][c]))
        d2 = (v * v).sum(1)
        logw.append(-0.5 * torch.log(d2) - d2 / (2.0 * case["dim"] * float(d["sigma"][c]) ** 2))
    if len(fits) == 1:
        return fits[0]
    return (torch.softmax(torch.stack(logw), 0) * torch.stack(fits)).sum(0)


def _hybrid(objective, z):
    shares, objectives, rates = HYBRIDS[objective]
    dim, start, total = z.shape[1], 0, 0.0
    for k, (obj, rate) in enumerate(zip(objectives, rates)):
        end = dim if k + 1 == len(objectives) else start + math.ceil(shares[k] * dim)
        total = total + _objective(obj, z[:, start:end] * rate)
        start = end
    return total


def _objective(obj, z):
    n = z.shape[1]
    j = torch.arange(n, device=z.device, dtype=torch.float64)
    pi = math.pi
    if obj == S.OBJ_ELLIPTIC:
        return (10.0 ** (6.0 * j / (n - 1)) * z * z).sum(1)
    if obj == S.OBJ_BENT_CIGAR:
        return z[:, 0] ** 2 + 1e6 * (z[:, 1:] ** 2).sum(1)
    if obj == S.OBJ_DISCUS:
        return 1e6 * z[:, 0] ** 2 + (z[:, 1:] ** 2).sum(1)
    if obj == S.OBJ_RASTRIGIN:
        return (z * z - 10.0 * torch.cos(2 * pi * z) + 10.0).sum(1)
    if obj == S.OBJ_ACKLEY:
        return (-20.0 * torch.exp(-0.2 * torch.sqrt((z * z).mean(1))) - torch.exp(torch.cos(2 * pi * z).mean(1))
                + 20.0 + math.e)
    if obj in (S.OBJ_HAPPYCAT, S.OBJ_HGBAT):
        u = z - 1.0
        r2, s = (u * u).sum(1), u.sum(1)
        head = (r2 - n).abs() ** 0.25 if obj == S.OBJ_HAPPYCAT else (r2 * r2 - s * s).abs() ** 0.5
        return head + (0.5 * r2 + s) / n + 0.5
    if obj == S.OBJ_SCHWEFEL:
        v = z + 420.9687462275036
        a = v.abs()
        m = 500.0 - torch.fmod(a, 500.0)
        inside = v * torch.sin(torch.sqrt(a))
        outside = torch.sign(v) * m * torch.sin(torch.sqrt(m)) - ((a - 500.0) / 100.0) ** 2 / n
        return 418.9828872724338 * n - torch.where(a <= 500.0, inside, outside).sum(1)
    if obj == S.OBJ_ROSENBROCK:
        y = z + 1.0
        return (100.0 * (y[:, :-1] ** 2 - y[:, 1:]) ** 2 + (y[:, :-1] - 1.0) ** 2).sum(1)
    if obj == S.OBJ_WEIERSTRASS:
        total, c = 0.0, 0.0
        for k in range(21):
            total = total + 0.5 ** k * torch.cos(2 * pi * 3.0 ** k * (z + 0.5)).sum(1)
            c += 0.5 ** k * math.cos(2 * pi * 3.0 ** k * 0.5)
        return total - n * c
    if obj == S.OBJ_GRIEWANK:
        return 1.0 + (z * z).sum(1) / 4000.0 - torch.cos(z / torch.sqrt(1.0 + j)).prod(1)
    if obj == S.OBJ_KATSUURA:
        t = 0.0
        for k in range(1, 33):
            v = z * 2.0 ** k
            t = t + (v - torch.floor(v + 0.5)).abs() / 2.0 ** k
        return 10.0 / n ** 2 * ((1.0 + (j + 1.0) * t) ** (10.0 / n ** 1.2)).prod(1) - 10.0 / n ** 2
    if obj == S.OBJ_GRIE_ROSEN:
        y = z + 1.0
        y1 = torch.roll(y, -1, 1)
        t = 100.0 * (y * y - y1) ** 2 + (y - 1.0) ** 2
        return (t * t / 4000.0 - torch.cos(t) + 1.0).sum(1)
    if obj == S.OBJ_ESCAFFER6:
        r2 = z * z if n == 1 else z * z + torch.roll(z, -1, 1) ** 2
        return (0.5 + (torch.sin(torch.sqrt(r2)) ** 2 - 0.5) / (1.0 + 0.001 * r2) ** 2).sum(1)
    raise ValueError(f"objective {obj}")

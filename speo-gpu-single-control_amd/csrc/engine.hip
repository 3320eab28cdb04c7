// engine.hip -- the island engine: islands of uneven size and dimension in one
// GPU's HBM, evolved by DE/rand/1/bin with ring migration.
//
// Reference counterparts: the generation loop of IslandEA::Execute
// (src/island_EA.cc:78-113), DE_CUDA::Run (CUDA_EA_library/DE_CUDA.cc:200-216),
// EA_CUDA::FindBestIndividual (EA_CUDA.cc:104-120) and the MPI migration of
// src/migrate.cc:46-144, which here becomes a ring among islands in HBM.
//
// One kernel, k_generation, covers the four per-generation roles over a table
// of (island, row tile) work items, so every launch spans all islands:
//   kModeGen     trials U <- X
//   kModeEval    f(U) through the MFMA evaluation
//   kModeSelect  X, fX <- U, fU where fU < fX
//   kModeFused   select(g-1) + generate(g) + evaluate(g) in one launch.
// A plain engine runs its generations as fused launches and one selection
// after the last; the three separate roles serve sub-islands, the surrogate,
// problems of the generic kernel and the per-role profile.
// Evaluation inside this kernel is for rows of at most 128 columns; when an
// island is wider, kModeFusedGen makes the generation's trials and the launches
// of engine_wide.hip evaluate them.
// The fused mode needs no grid-wide barrier: the selection of generation g-1
// is not applied before the donors are read; instead a donor row r is read as
// U_prev[r] when fU_prev[r] < fX_prev[r] and as X[r] otherwise, and X[r] is
// only written for accepted rows (which nobody reads as X), while U and the
// fitness arrays are double-buffered.  The result equals the plain engine's.
#pragma clang fp contract(off)

#include <sys/stat.h>

#include <chrono>
#include <algorithm>
#include <cstdlib>
#include <fstream>
#include <sstream>
#include <map>
#include <memory>
#include <mutex>
#include <tuple>
#include <vector>

#include "engine.h"
#include "eval.h"
#include "surrogate.h"
#include "wide_core.h"

namespace speo {

enum GenMode { kModeGen = 0, kModeEval = 1, kModeSelect = 2, kModeFused = 3, kModeFusedGen = 4 };

// A block's work item: rows [row0, row0 + nrows) of an island, with a copy of
// the island's descriptor (immutable after set-up), so a block reads its work
// in one round trip instead of two dependent ones.
struct TileDesc {
    IslandDesc I;
    int island, row0, nrows;
    uint32_t inv_ng;  // group_inverse(I.dim)
};

// A screened generation's appends (C > 0): the evaluation writes the trials and
// log(1 + f) to the archive and applies the selection itself.
struct AppendArgs {
    float *AX, *Ay;     // [problem][cap][Kp], [problem][cap]; AX null: evaluation only
    const int *qrel;    // [island] first target's place among its problem's
    const int *head;    // [problem] first slot of the generation
    int cap, Kp;
};

struct GenerationArgs {
    const IslandDesc *isl;
    const TileDesc *tiles;
    const FusedProblem *probs;
    float *X;
    const float *fX_prev;
    float *fX_new;
    const float *U_prev;
    float *fU_prev;
    float *U_new;
    float *fU_new;
    const float *eval_src;
    float *eval_out;
    float lo, hi;
    uint64_t seed;
    const uint32_t *gen_base;
    uint32_t gen_offset;
    const int4 *donors;  // [row] {r0, r1, r2, j_rand} of the generation (epoch_donors)
    int pending;         // fused modes: trials of the previous generation await selection
    int clear_trials;
    int composed;        // an island's problem has more than one component
    AppendArgs append;
};

// Rows per block of the launches that only make trials or select: they depend on
// no arithmetic of the evaluation's tile, and small tiles fill the chip (16,384
// rows of D = 1000: trials 85 us at 64 rows a block, 55 us at 16).
constexpr int kTrialRows = 16;

constexpr int kTLD = kSmallD;  // widest dimension this kernel evaluates

// LDS of one block: [trial rows RT x kTS] [gval kMaxComp x RT] [scratch of the
// GEMM and the row reduction, before them the parents' table].  Generations
// without evaluation hold the table alone.
template <int RT> constexpr int parent_table_bytes() { return RT * (4 * 8 + 4); }
template <int RT, int PREC>
constexpr int generation_lds_bytes() {
    return RT * kTS * 4 + kMaxComp * RT * 4 +
           std::max(small_scratch_bytes<RT>(Prec<PREC>::parts) + 10 * RT * 4, parent_table_bytes<RT>());
}

__device__ __forceinline__ float4 ld4(const float *p) { return *reinterpret_cast<const float4 *>(p); }
__device__ __forceinline__ void st4(float *p, float4 v) { *reinterpret_cast<float4 *>(p) = v; }
__device__ __forceinline__ float comp4(const float4 &v, int q) {
    return q == 0 ? v.x : (q == 1 ? v.y : (q == 2 ? v.z : v.w));
}

// What bounds the fused kernel: the chain of a block's phases (a D = 100 block of
// 32 rows takes about 19 us) and the last blocks behind it, not the chip's issue
// rates: over a 34 us launch of the uneven islands vector instructions issue in 35 %
// of the SIMD units' cycles (18 wide integer multiplies per four coordinates of
// the crossover, at a quarter of the rate, among them), the matrix pipe is busy
// for 11 %, and 2.9 of the four waves that fit a unit are there.  So every lane makes trials (items of a row and
// four coordinates, where 16 lanes a row left 13 idle at D = 10), the parents of
// a row are found once, not by 16 lanes, a generation's donors are drawn ahead
// of it, one row per lane (k_epoch_donors), and blocks start at different
// column classes.  256 uneven islands, D 10..100, one generation: 62 us with
// donors drawn here, 49 without, 40 with the evaluation's registers at four
// waves a SIMD unit, 33 with the items and classes.
// Row tile 32 is held to four waves a SIMD unit (128 registers, no spills); with
// the composition's code to three.  The other row tiles keep the compiler's
// allocation.
template <int RT, int PREC, int MODE, bool COMP>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(RT == 32 ? (COMP ? 3 : 4) : 1))) void k_generation(
    GenerationArgs a) {
    extern __shared__ __align__(16) char lds[];
    const TileDesc t = a.tiles[blockIdx.x];
    const IslandDesc I = t.I;
    const int tid = threadIdx.x;

    if constexpr (MODE == kModeSelect) {
        // 16 lanes per row: trials (U_prev, fU_prev) into (X, fX_new).
        for (int pass = 0; pass < RT / 16; ++pass) {
            const int lr = pass * 16 + (tid >> 4), l = tid & 15;
            if (lr >= t.nrows) continue;
            const int li = t.row0 + lr, gr = I.row_off + li;
            const float fu = a.fU_prev[gr], fx = a.fX_prev[gr];
            const bool acc = fu < fx;
            if (acc) {
                const float *u = a.U_prev + I.elem_off + (size_t)li * I.ld;
                float *x = a.X + I.elem_off + (size_t)li * I.ld;
                for (int g = l; g < (I.ld >> 2); g += 16) st4(x + 4 * g, ld4(u + 4 * g));
            }
            if (l == 0) {
                a.fX_new[gr] = acc ? fu : fx;
                if (a.clear_trials) a.fU_prev[gr] = INFINITY;
            }
        }
        return;
    }

    constexpr bool FUSED = MODE == kModeFused || MODE == kModeFusedGen;
    constexpr bool lds_trial = MODE == kModeFused || MODE == kModeEval;
    float *trial = reinterpret_cast<float *>(lds);
    float *gval = trial + RT * kTS;
    char *gemm_lds = lds_trial ? reinterpret_cast<char *>(gval + kMaxComp * RT) : lds;

    // The first component's rotation does not depend on the rows: its operands
    // are requested before them.
    constexpr bool EVAL = MODE == kModeEval || MODE == kModeFused;
    constexpr bool AHEAD = EVAL && Prec<PREC>::parts == 0;
    const FusedProblem *P = a.probs + I.problem;
    if (MODE == kModeEval && P->generic) return;  // the generic kernel evaluates this island
    SmallB B;

    const int ng = (I.dim + 3) >> 2;  // groups of four coordinates
    // row and group of item e < RT * ng
    auto item_row = [&](int e) { return t.inv_ng ? (int)__umulhi((uint32_t)e, t.inv_ng) : e / ng; };

    if constexpr (MODE == kModeGen || FUSED) {
        const uint32_t gen = (a.gen_base ? *a.gen_base : 0u) + a.gen_offset;
        const uint32_t crt = cr_threshold(I.CR);
        // Four threads a row find its parents: the donors' rows and its own,
        // each where the pending selection left it.
        const float **src = reinterpret_cast<const float **>(gemm_lds);  // [RT][4]
        int *own = reinterpret_cast<int *>(src + 4 * RT);                // [RT] j_rand, bit 31: own trial accepted
        if (tid < 4 * t.nrows) {
            const int lr = tid >> 2, j = tid & 3, li = t.row0 + lr, gr = I.row_off + li;
            const int4 d = a.donors[gr];
            const int r = j == 0 ? d.x : j == 1 ? d.y : j == 2 ? d.z : li;
            bool acc = false;
            if (FUSED) {
                const float fx = a.fX_prev[I.row_off + r];
                const float fu = a.pending ? a.fU_prev[I.row_off + r] : INFINITY;
                acc = fu < fx;
                if (j == 3) a.fX_new[gr] = acc ? fu : fx;
            }
            src[tid] = (acc ? a.U_prev : a.X) + I.elem_off + (size_t)r * I.ld;
            if (j == 3) own[lr] = d.w | (acc ? (int)0x80000000 : 0);
        }
        __syncthreads();
        float *U_new = a.U_new + I.elem_off + (size_t)t.row0 * I.ld;
        float *X = a.X + I.elem_off + (size_t)t.row0 * I.ld;
        // Items of (row, group of four coordinates), two at a time: the loads
        // of both are in flight together.
        struct Item {
            bool valid, acc;
            int lr, g, jr;
            float4 e0, e1, e2, xo;
        };
        auto load = [&](int e) {
            Item c;
            c.valid = e < t.nrows * ng;
            if (!c.valid) return c;
            c.lr = item_row(e);
            c.g = e - c.lr * ng;
            const int o = own[c.lr];
            c.jr = o & 0x7fffffff;
            c.acc = o < 0;
            c.e0 = ld4(src[4 * c.lr + 0] + 4 * c.g);
            c.e1 = ld4(src[4 * c.lr + 1] + 4 * c.g);
            c.e2 = ld4(src[4 * c.lr + 2] + 4 * c.g);
            c.xo = ld4(src[4 * c.lr + 3] + 4 * c.g);
            return c;
        };
        auto make = [&](const Item &c) {
            const U4 w = philox_block(a.seed, (uint32_t)c.g, (uint32_t)(I.row_off + t.row0 + c.lr), gen,
                                      kPurposeCross);
            float v[4];
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const int j = 4 * c.g + q;
                const bool take = (j == c.jr) || cross_take(word(w, q), crt);
                const float m = take ? fmaf(I.F, comp4(c.e1, q) - comp4(c.e2, q), comp4(c.e0, q))
                                     : comp4(c.xo, q);
                v[q] = j < I.dim ? check_bound(m, a.lo, a.hi) : 0.f;
            }
            const float4 out{v[0], v[1], v[2], v[3]};
            st4(U_new + c.lr * I.ld + 4 * c.g, out);
            if (lds_trial) st4(trial + c.lr * kTS + 4 * c.g, out);
            if (FUSED && c.acc) st4(X + c.lr * I.ld + 4 * c.g, c.xo);
        };
        for (int e = tid; e < t.nrows * ng; e += 512) {
            const Item A = load(e), B = load(e + 256);
            make(A);
            if (B.valid) make(B);
        }
        if (lds_trial)  // rows past the tile's
            for (int e = t.nrows * ng + tid; e < RT * ng; e += 256) {
                const int lr = item_row(e);
                st4(trial + lr * kTS + 4 * (e - lr * ng), float4{0.f, 0.f, 0.f, 0.f});
            }
        if constexpr (EVAL) __syncthreads();  // the parents' table lies where the evaluation's scratch does
    }

    if constexpr (MODE == kModeEval || MODE == kModeFused) {
        const int ncomp = COMP ? P->ncomp : 1, dim = I.dim, cls = column_class();
        if (MODE == kModeEval) {
            // stage the rows to evaluate into the LDS tile (zero rows past nrows)
            const float *srcp = a.eval_src + I.elem_off + (size_t)t.row0 * I.ld;
            for (int e = tid; e < RT * ng; e += 256) {
                const int r = item_row(e), g = e - r * ng;
                st4(trial + r * kTS + 4 * g,
                    r < t.nrows ? ld4(srcp + (size_t)r * I.ld + 4 * g) : float4{0.f, 0.f, 0.f, 0.f});
            }
        }
        if constexpr (AHEAD) {
            B.load(P->comp[0], dim, cls);
            B.stage(gemm_lds);
        }
        __syncthreads();
        for (int c = 0; c < ncomp; ++c) {
            const CompDev comp = P->comp[c];
            float *red = reinterpret_cast<float *>(gemm_lds + small_scratch_bytes<RT>(Prec<PREC>::parts));
            float *o1 = red + 8 * RT, *o2 = o1 + RT;
            float s1[RT / 16][4], s2[RT / 16][4];
            if constexpr (AHEAD) {
                if (c > 0) {  // (the reduction's barriers lie between this and the last K loop)
                    B.load(comp, dim, cls);
                    B.stage(gemm_lds);
                    __syncthreads();
                }
                gemm_small_f32<RT>(comp, B, trial, dim, cls, gemm_lds, s1, s2);
            } else {
                gemm_small<RT, PREC>(comp, trial, dim, cls, gemm_lds, s1, s2);
            }
            reduce_rows_small<RT>(s1, s2, cls, red, o1, o2);
            if (tid < t.nrows) gval[c * RT + tid] = finish_objective_ext(comp.objective, o1[tid], o2[tid], dim);
            if (comp.heavy.j >= 0) {
                // the heavy column's FP64 term, one wave per row
                __syncthreads();
                const int wave = tid >> 6, lane = tid & 63;
                heavy_rows(comp.heavy, dim, wave, 4, t.nrows, lane, [&](int r) { return trial + r * kTS; },
                           [&](int r, double h) {
                               if (lane == 0) gval[c * RT + r] = with_heavy(gval[c * RT + r], (float)h);
                           });
                __syncthreads();
            }
        }
        if (tid < t.nrows) {
            float f;
            if (!COMP || ncomp == 1) {
                f = fmaf(P->lambda[0], gval[tid], P->bias[0]);
            } else {
                // cf_cal weights (CEC2014.cc:1481-1519) in the log domain.
                const float *x = trial + tid * kTS;
                // (components at distance 0 share the weight equally, as
                // cf_cal's w = 1e99 each)
                float lw[kMaxComp], lwmax = -INFINITY;
                bool zero[kMaxComp];
                bool any_zero = false;
                for (int c = 0; c < ncomp; ++c) {
                    const float *o = P->comp[c].shift;
                    float d = 0.f;
                    for (int j = 0; j < dim; ++j) {
                        const float v = x[j] - o[j];
                        d = fmaf(v, v, d);
                    }
                    zero[c] = d == 0.f;
                    any_zero = any_zero || zero[c];
                    const float s = P->sigma[c];
                    lw[c] = -0.5f * logf(d) - d / (2.0f * (float)dim * s * s);
                    lwmax = fmaxf(lwmax, lw[c]);
                }
                float wsum = 0.f, acc = 0.f;
                for (int c = 0; c < ncomp; ++c) {
                    const float w = any_zero ? (zero[c] ? 1.f : 0.f) : expf(lw[c] - lwmax);
                    wsum += w;
                    acc = fmaf(w, fmaf(P->lambda[c], gval[c * RT + tid], P->bias[c]), acc);
                }
                f = acc / wsum;
            }
            float *out = MODE == kModeEval ? a.eval_out : a.fU_new;
            out[I.row_off + t.row0 + tid] = f;
            if (MODE == kModeEval && a.append.AX) {
                const int gr = I.row_off + t.row0 + tid;
                const float fx = a.fX_new[gr];
                const size_t slot = (size_t)I.problem * a.append.cap +
                                    (size_t)(((int64_t)a.append.head[I.problem] + a.append.qrel[t.island] + t.row0 +
                                              tid) % a.append.cap);
                if (f < fx) a.fX_new[gr] = f;
                a.append.Ay[slot] = log1pf(fmaxf(f, 0.f));
                reinterpret_cast<int64_t *>(gemm_lds)[tid] = (int64_t)slot * 2 + (f < fx ? 1 : 0);
            }
        }
        if (MODE == kModeEval && a.append.AX) {
            // the rows to the archive (zeros past the dimension), accepted ones
            // also to the population
            __syncthreads();
            const int64_t *slots = reinterpret_cast<const int64_t *>(gemm_lds);
            float *X = a.X + I.elem_off + (size_t)t.row0 * I.ld;
            const int kg = a.append.Kp >> 2;
            for (int e = tid; e < t.nrows * kg; e += 256) {
                const int r = e / kg, g = e - r * kg;
                const int64_t sl = slots[r];
                const float4 v = g < ng ? ld4(trial + r * kTS + 4 * g) : float4{0.f, 0.f, 0.f, 0.f};
                st4(a.append.AX + (size_t)(sl >> 1) * a.append.Kp + 4 * g, v);
                if ((sl & 1) && g < ng) st4(X + r * I.ld + 4 * g, v);
            }
        }
    }
}

__global__ void k_fill(float *p, int n, float v) {
    for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) p[i] = v;
}
__global__ void k_add_u32(uint32_t *p, uint32_t v) {
    if (threadIdx.x == 0 && blockIdx.x == 0) p[0] += v;
}
// ------------------------------------------------------------------ launch

template <int RT, int PREC, int MODE, bool COMP>
static int launch_generation(const GenerationArgs &a, int ntiles, hipStream_t s) {
    const int lds = MODE == kModeEval || MODE == kModeFused ? generation_lds_bytes<RT, PREC>()
                    : MODE == kModeSelect                     ? 0
                                                              : parent_table_bytes<RT>();
    static std::once_flag once;
    std::call_once(once, [] {
        (void)hipFuncSetAttribute(reinterpret_cast<const void *>(&k_generation<RT, PREC, MODE, COMP>),
                                  hipFuncAttributeMaxDynamicSharedMemorySize,
                                  generation_lds_bytes<RT, PREC>());
    });
    hipLaunchKernelGGL((k_generation<RT, PREC, MODE, COMP>), dim3(ntiles), dim3(256), lds, s, a);
    return check_launch("k_generation");
}

template <int RT, int PREC, int MODE>
static int launch_values(const GenerationArgs &a, int ntiles, hipStream_t s) {
    return a.composed ? launch_generation<RT, PREC, MODE, true>(a, ntiles, s)
                      : launch_generation<RT, PREC, MODE, false>(a, ntiles, s);
}

template <int RT, int PREC>
static int launch_mode(int mode, const GenerationArgs &a, int ntiles, hipStream_t s) {
    return mode == kModeEval ? launch_values<RT, PREC, kModeEval>(a, ntiles, s)
                             : launch_values<RT, PREC, kModeFused>(a, ntiles, s);
}

template <int RT>
static int launch_prec(int prec, int mode, const GenerationArgs &a, int ntiles, hipStream_t s) {
    switch (prec) {
    case SPEO_PREC_FP32: return launch_mode<RT, SPEO_PREC_FP32>(mode, a, ntiles, s);
    case SPEO_PREC_BF16: return launch_mode<RT, SPEO_PREC_BF16>(mode, a, ntiles, s);
    case SPEO_PREC_FP16: return launch_mode<RT, SPEO_PREC_FP16>(mode, a, ntiles, s);
    case SPEO_PREC_BF16X3: return launch_mode<RT, SPEO_PREC_BF16X3>(mode, a, ntiles, s);
    case SPEO_PREC_FP16X3: return launch_mode<RT, SPEO_PREC_FP16X3>(mode, a, ntiles, s);
    case SPEO_PREC_BF16X6: return launch_mode<RT, SPEO_PREC_BF16X6>(mode, a, ntiles, s);
    default: return set_error(SPEO_ERR_ARG, "unknown precision");
    }
}

// kModeEval and kModeFused, tiles of rt rows.
static int launch_any(int rt, int prec, int mode, const GenerationArgs &a, int ntiles,
                      hipStream_t s) {
    switch (rt) {
    case 16: return launch_prec<16>(prec, mode, a, ntiles, s);
    case 32: return launch_prec<32>(prec, mode, a, ntiles, s);
    case 64: return launch_prec<64>(prec, mode, a, ntiles, s);
    default: return set_error(SPEO_ERR_ARG, "rows_per_block must be 16, 32 or 64");
    }
}

// The roles without evaluation, tiles of kTrialRows.
static int launch_trials(int mode, const GenerationArgs &a, int ntiles, hipStream_t s) {
    constexpr int RT = kTrialRows, FP32 = SPEO_PREC_FP32;
    switch (mode) {
    case kModeGen: return launch_generation<RT, FP32, kModeGen, false>(a, ntiles, s);
    case kModeSelect: return launch_generation<RT, FP32, kModeSelect, false>(a, ntiles, s);
    default: return launch_generation<RT, FP32, kModeFusedGen, false>(a, ntiles, s);
    }
}

// ------------------------------------------------------------ tuning cache
//
// The autotuner's choices, persisted across processes: one "key value" line
// per choice in $SPEO_TUNE_CACHE (empty: no file), else
// $HOME/.cache/speo_de/autotune-v1.txt.  Keys name the mode, the precision
// and every island's (dimension, NP rounded up to a power of two).

namespace {
std::mutex g_tune_mu;

std::string tune_path() {
    if (const char *e = std::getenv("SPEO_TUNE_CACHE")) return e;
    const char *h = std::getenv("HOME");
    return h ? std::string(h) + "/.cache/speo_de/autotune-v1.txt" : std::string();
}

bool tune_lookup(const std::string &key, int *value) {
    std::lock_guard<std::mutex> lk(g_tune_mu);
    const std::string path = tune_path();
    if (path.empty()) return false;
    std::ifstream f(path);
    std::string k;
    int v = 0;
    bool found = false;
    while (f >> k >> v)
        if (k == key) {
            *value = v;  // the last line for a key wins
            found = true;
        }
    return found;
}

void tune_store(const std::string &key, int value) {
    std::lock_guard<std::mutex> lk(g_tune_mu);
    const std::string path = tune_path();
    if (path.empty()) return;
    for (size_t i = 1; i < path.size(); ++i)  // create the directories on the way
        if (path[i] == '/') (void)::mkdir(path.substr(0, i).c_str(), 0755);
    std::ofstream f(path, std::ios::app);
    if (f) f << key << ' ' << value << '\n';
}
}  // namespace

// ------------------------------------------------------------------ engine

struct Engine {
    hipStream_t stream = nullptr;
    bool own_stream = false;
    speo_engine_config cfg{};
    int I = 0, total_rows = 0, max_dim = 0, max_ld = 0, max_np = 0;
    int64_t total_elems = 0;
    std::vector<IslandDesc> isl;
    std::vector<int> row_off, dst;
    std::vector<speo_problem> problems;
    bool all_small = true;  // every dim <= kTLD
    bool any_generic = false;  // some problem needs the generic kernel (plain mode only)
    // The reference island's sub-islands and DE configuration (plain mode):
    // per island the sub-island count, permutation and DEInfo per sub-island.
    bool configured = false;
    int regroup_events = 0;
    // measured communication (run_fes_timed): migrations (and regroups) run
    // eagerly between synchronisations and their wall time is summed, as the
    // reference's MPI_Wtime brackets around MigrateOut / MigrateIn
    // (island_EA.cc:94-104)
    bool time_comm = false;
    double comm_seconds = 0.0;
    int timed_point(bool mig, bool point);
    std::vector<int> subs_h;
    std::vector<std::vector<int>> perm_h;
    std::vector<std::vector<DEInfo>> info_h;
    std::vector<DEInfo> base_h;
    std::vector<int> doff;           // island -> first DEInfo / best slot
    int *perm_dev = nullptr, *best_sub_dev = nullptr;
    DEInfo *info_dev = nullptr;
    int configure_setup();
    int regroup(bool initial);
    int generate_configured(int gen_offset, hipStream_t s);
    int subislands(int island, int *subs_out, int *perm_out, DEInfo *info_out);
    int eval_generic_islands(const float *src, float *out, hipStream_t s);

    IslandDesc *isl_dev = nullptr;
    int *row_off_dev = nullptr, *dst_dev = nullptr, *best_buf = nullptr, *worst_buf = nullptr;
    int *best_row_dev = nullptr;
    BestOut *best_out = nullptr, *best_out_dev = nullptr;  // pinned host memory and its device address
    double *best_part = nullptr;  // chunk sums of best() when an island is wider than kBestCols
    FusedProblem *probs_dev = nullptr;
    const CompParams **params_tab_dev = nullptr;
    std::map<int, TileDesc *> tiles_dev;  // per rows-per-block
    std::map<int, int> ntiles;
    // islands wider than kTLD (any of them): the evaluation's items, those the
    // tile kernel takes first, then those of rows_chunk; component values
    WideItem *wide_items = nullptr;
    std::vector<FusedProblem> fused;    // probs_dev's contents
    std::vector<void *> narrow_frags;   // M in the tile kernel's order, of problems up to kTLD
    int narrow_fragments(const CompHost &h, const ProblemHost &P, CompDev &c);
    int wide_tile = 0, wide_chunk = 0, wide_ncomp = 1;
    int wide_dim = 0;  // the widest of the tile kernel's items (their shift lies in LDS)
    float *gval = nullptr;
    int build_wide_items();
    int eval_wide_rows(const float *src, float *out, int rt_, hipStream_t s);
    uint32_t *gen_base = nullptr;

    float *X = nullptr, *fX[2] = {nullptr, nullptr}, *U[2] = {nullptr, nullptr};
    float *fU[2] = {nullptr, nullptr};
    bool composed = false;  // a problem has more than one component
    int p = 0;            // fused mode: the buffers of the current fitness and trials
    int pf = 0, pu = 0;   // the same within a plain chunk, where they part (both 0 outside)
    bool pending = false;

    int rt = 32;
    int64_t gens = 0, fes = 0, migrations = 0, graph_launches = 0;

    // learned surrogate (config.surrogate_candidates > 0)
    struct SurrProblem {
        Mlp net;
        int qoff = 0, rows = 0, head = 0;
        int64_t appended = 0;
        bool trained = false;
    };
    int C = 0, Kp = 0, Q = 0;
    std::vector<std::unique_ptr<SurrProblem>> surr;
    SurrRowDesc *srows_dev = nullptr;
    float *cand = nullptr, *pred = nullptr, *rho_dev = nullptr, *AX = nullptr, *Ay = nullptr;
    long long *scored_dev = nullptr;  // candidates scored per problem by the one-kernel screening
    float *Xb = nullptr, *tb = nullptr, *Xh = nullptr, *yh = nullptr, *predh = nullptr;
    float2 *ranks_ws = nullptr;  // Spearman workspace
    int *heads_dev = nullptr;         // the generation's first archive slot per problem (device)
    int *qrel_dev = nullptr;          // [island] first target's place among its problem's
    int4 *drawn = nullptr;            // [target][candidate] donors and j_rand of scored candidates
    uint32_t *round_dev = nullptr;    // training rounds run (device; keys the minibatch draws)
    bool any_trained = false;
    int last_Ce = 1;  // candidates per target in the last surrogate generation
    bool retain_cand = false;  // candidates also written to memory (after a dump request)
    int64_t surr_pred = 0, surr_rounds = 0;
    int surrogate_setup();
    int surrogate_generation(int gen_offset, hipStream_t s);
    int enqueue_surrogate_round(int TI, int mig_pos, hipStream_t s);
    void surrogate_round_host(int TI);
    bool surrogate_round_replayable() const;
    int surrogate_train(hipStream_t s);
    std::map<std::tuple<int, int, int>, hipGraphExec_t> graphs;
    bool graph_failed = false;

    // donors drawn ahead of the generations (engines without sub-islands)
    int4 *donor_buf = nullptr;  // [donor_gens][rows]
    int *row_island_dev = nullptr;
    int donor_gens = 1;
    int donor_setup();
    int draw_ahead(int gen_offset, int L, hipStream_t s);

    // epoch mode: per-island plans, block order, LDS of a launch
    EpochBlock *blocks_dev = nullptr;
    int epoch_lds = 0, epoch_parts = 1, epoch_blocks = 0;
    float *Xnext = nullptr;  // split islands: the population of the next generation
    int ep_par = 0;          // split islands: buffers swapped an odd number of times
    int epoch_setup();
    int epoch_plan_all(int parts, std::vector<EpochPlan> *plans, int *lds);
    int launch_epoch_chunk(int L, hipStream_t s);
    void swap_epoch_buffers();

    ~Engine();
    int create(const speo_engine_config &c, hipStream_t s);
    int upload_tables();
    int build_tiles(int rt_);
    int launch(int mode, int gen_offset, int rt_, hipStream_t s, int clear = 0, bool append = false);
    int enqueue_plain(int L, hipStream_t s);
    int enqueue_chunk(int L, bool migrate, hipStream_t s);
    int finalize_pending(hipStream_t s);
    int migrate(hipStream_t s);
    // dry: capture and instantiate the chunks' graphs, launch nothing (host
    // state is advanced as if launched; prepare() restores it)
    int run(int generations, bool dry = false);
    int prepare(int generations);
    int profile(int generations, double *avg_ms);
    int profile_epoch(int generations, double *avg_ms);
    // when set, launch_epoch_chunk records an event pair around every launch:
    // (role 4 = epoch kernel, role 5 = donor draws, events, generations covered)
    struct ProfEvent {
        int role;
        hipEvent_t a, b;
        int gens;
    };
    std::vector<ProfEvent> *prof = nullptr;
    int prof_begin(int role, int gens, hipStream_t s);
    int prof_end(hipStream_t s);
    int next_chunk(int left, bool *mig) const;
    int autotune();
    // epoch mode: workgroups per island measured over the candidates on
    // throwaway engines of the same configuration (cfg.epoch_parts == 0)
    bool tuning_child = false;
    int tuned_from_cache = 0;  // bit 0: row tile, bit 1: epoch parts
    std::string tune_key(const char *what) const;
    std::string plan_key(const char *what) const;
    bool runs_fused() const;
    int tune_epoch_parts();
    // epoch mode: generations as fused launches instead of an epoch kernel
    bool by_launches = false;
    int tune_launches();
    int time_plan(int parts, bool launches, double *seconds);
    int best(int *row_out, float *f32_out, double *f64_out);
    int read(float *Xo, float *fo);
    int read_rows(const float *src, const float *fsrc, float *Xo, float *fo);
    int write(const float *Xi, const float *fi);
};

Engine::~Engine() {
    if (stream) (void)hipStreamSynchronize(stream);
    for (auto &kv : graphs) (void)hipGraphExecDestroy(kv.second);
    for (auto &kv : tiles_dev) (void)hipFree(kv.second);
    void *bufs[] = {isl_dev, row_off_dev, dst_dev, best_buf, worst_buf, best_row_dev,
                    best_part, probs_dev, params_tab_dev, gen_base,
                    blocks_dev, Xnext, donor_buf, row_island_dev, wide_items, gval,
                    X, fX[0], fX[1], U[0], U[1], fU[0], fU[1], srows_dev, cand, pred, rho_dev, scored_dev,
                    AX, Ay, Xb, tb, Xh, yh, predh, ranks_ws, heads_dev, qrel_dev, drawn, round_dev, perm_dev,
                    best_sub_dev, info_dev};
    for (void *b : bufs) (void)hipFree(b);
    for (void *b : narrow_frags) (void)hipFree(b);
    (void)hipHostFree(best_out);
    if (own_stream && stream) (void)hipStreamDestroy(stream);
}

template <typename T>
static int upload_vec(T **dst, const std::vector<T> &src) {
    SPEO_TRY_HIP(hipMalloc(reinterpret_cast<void **>(dst), sizeof(T) * std::max<size_t>(src.size(), 1)));
    if (!src.empty())
        SPEO_TRY_HIP(hipMemcpy(*dst, src.data(), sizeof(T) * src.size(), hipMemcpyHostToDevice));
    return SPEO_OK;
}

int Engine::build_tiles(int rt_) {
    if (tiles_dev.count(rt_)) return SPEO_OK;
    std::vector<TileDesc> tiles;
    for (int i = 0; i < I; ++i)
        for (int r0 = 0; r0 < isl[(size_t)i].np; r0 += rt_)
            tiles.push_back(TileDesc{isl[(size_t)i], i, r0, std::min(rt_, isl[(size_t)i].np - r0),
                                     group_inverse(isl[(size_t)i].dim)});
    // Heaviest tiles first (rows x dim^2, ties in island order): blocks are
    // dispatched in this order, so with uneven islands the last wave of blocks
    // holds the cheap tiles.  Tiles are independent: the order changes no result.
    auto cost = [&](const TileDesc &t) { return (int64_t)t.nrows * t.I.dim * t.I.dim; };
    std::stable_sort(tiles.begin(), tiles.end(),
                     [&](const TileDesc &x, const TileDesc &y) { return cost(x) > cost(y); });
    TileDesc *d = nullptr;
    SPEO_TRY(upload_vec(&d, tiles));
    tiles_dev[rt_] = d;
    ntiles[rt_] = (int)tiles.size();
    return SPEO_OK;
}

// Items of the wide evaluation: 64-row tiles of every island the fused
// kernels' arithmetic evaluates, each component an item.  Groups of eight tiles
// are listed component by component: workgroup b runs on XCD b mod 8, so a
// tile's components run on one XCD, close in time, and share its rows in that
// L2.  Wider islands first.
int Engine::build_wide_items() {
    std::vector<WideItem> tile, chunk;
    std::vector<int> order((size_t)I);
    for (int i = 0; i < I; ++i) order[(size_t)i] = i;
    std::stable_sort(order.begin(), order.end(),
                     [&](int x, int y) { return isl[(size_t)x].dim > isl[(size_t)y].dim; });
    for (int i : order) {
        const IslandDesc &d = isl[(size_t)i];
        const ProblemHost &P = problems[(size_t)d.problem]->h;
        if (P.generic) continue;
        wide_ncomp = std::max(wide_ncomp, P.ncomp);
        for (int g0 = 0; g0 < d.np; g0 += 8 * kWideRows)
            for (int c = 0; c < P.ncomp; ++c) {
                const bool tiled = rows_wide_applies(fused[(size_t)d.problem].comp[c], d.dim, cfg.precision);
                auto &list = tiled ? tile : chunk;
                if (tiled) wide_dim = std::max(wide_dim, d.dim);
                for (int r0 = g0; r0 < std::min(d.np, g0 + 8 * kWideRows); r0 += kWideRows)
                    list.push_back(WideItem{d.elem_off + (int64_t)r0 * d.ld, d.row_off + r0,
                                            std::min(kWideRows, d.np - r0), d.ld, d.dim, d.problem, c});
            }
    }
    wide_tile = (int)tile.size();
    wide_chunk = (int)chunk.size();
    tile.insert(tile.end(), chunk.begin(), chunk.end());
    SPEO_TRY(upload_vec(&wide_items, tile));
    if (wide_ncomp > 1)
        SPEO_TRY_HIP(hipMalloc(&gval, sizeof(float) * (size_t)wide_ncomp * (size_t)total_rows));
    return SPEO_OK;
}

int Engine::eval_wide_rows(const float *src, float *out, int rt_, hipStream_t s) {
    const WideRowsArgs a{wide_items, probs_dev, src, out, gval, total_rows};
    WideRowsArgs rest = a;
    rest.items = wide_items + wide_tile;
    const int nsplit = 64 / rt_;
    SPEO_TRY(rows_wide(a, wide_tile, wide_dim, cfg.precision, nsplit, s));
    SPEO_TRY(rows_chunk(rest, wide_chunk, cfg.precision, nsplit, s));
    if (wide_ncomp > 1) SPEO_TRY(rows_combine(a, wide_tile + wide_chunk, wide_ncomp, s));
    return SPEO_OK;
}

// A problem keeps its rotations in the tile kernel's order from 129 columns on;
// those of narrower islands beside wider ones belong to the engine, in its precision.
int Engine::narrow_fragments(const CompHost &h, const ProblemHost &P, CompDev &c) {
    const int dim = P.dim;
    const size_t fe = wide_frag_elems(dim);
    const bool f32 = cfg.precision == SPEO_PREC_FP32;
    const bool half = cfg.precision == SPEO_PREC_FP16 || cfg.precision == SPEO_PREC_FP16X3;
    void *frag = nullptr;
    SPEO_TRY_HIP(hipMalloc(&frag, f32 ? 4 * fe : 3 * 2 * fe));
    narrow_frags.push_back(frag);
    uint16_t *part = static_cast<uint16_t *>(frag);
    const uint16_t *src[6] = {h.Mbf[0], h.Mbf[1], h.Mbf[2], h.Mh[0], h.Mh[1], h.Mh[2]};
    uint16_t *dst[6] = {};
    for (int q = 0; q < 3 && !f32; ++q) dst[(half ? 3 : 0) + q] = part + q * fe;
    SPEO_TRY(wide_fragments(h.B32, P.ldb32, src, P.ldm16, dim, f32 ? static_cast<float *>(frag) : nullptr, dst, stream));
    c.wide = frag;
    return SPEO_OK;
}

int Engine::upload_tables() {
    SPEO_TRY(upload_vec(&isl_dev, isl));
    SPEO_TRY(upload_vec(&row_off_dev, row_off));
    SPEO_TRY(upload_vec(&dst_dev, dst));
    fused.resize(problems.size());
    std::vector<const CompParams *> tab(problems.size());
    for (size_t q = 0; q < problems.size(); ++q) {
        const ProblemHost &P = problems[q]->h;
        FusedProblem f{};
        f.ncomp = P.ncomp;
        f.dim = P.dim;
        f.generic = P.generic ? 1 : 0;
        any_generic = any_generic || P.generic;
        composed = composed || P.ncomp > 1;
        for (int c = 0; c < P.ncomp; ++c) {
            f.lambda[c] = (float)P.comp[c].lambda;
            f.bias[c] = (float)P.comp[c].bias;
            f.sigma[c] = (float)P.comp[c].sigma;
            f.comp[c] = P.view(c, cfg.precision);
            if (!all_small && P.dim <= kTLD && !P.generic) SPEO_TRY(narrow_fragments(P.comp[c], P, f.comp[c]));
        }
        fused[q] = f;
        tab[q] = P.params_dev;
    }
    SPEO_TRY(upload_vec(&probs_dev, fused));
    SPEO_TRY(upload_vec(&params_tab_dev, tab));
    const int k = std::max(cfg.migration_size, 1);
    SPEO_TRY_HIP(hipMalloc(&best_buf, sizeof(int) * (size_t)I * k));
    SPEO_TRY_HIP(hipMalloc(&worst_buf, sizeof(int) * (size_t)I * k));
    SPEO_TRY_HIP(hipMalloc(&best_row_dev, sizeof(int) * (size_t)I));
    SPEO_TRY_HIP(hipHostMalloc(reinterpret_cast<void **>(&best_out), sizeof(BestOut) * (size_t)I, hipHostMallocMapped));
    SPEO_TRY_HIP(hipHostGetDevicePointer(reinterpret_cast<void **>(&best_out_dev), best_out, 0));
    if (max_dim > kBestCols)
        SPEO_TRY_HIP(hipMalloc(&best_part, sizeof(double) * 3 * (size_t)I * kMaxComp *
                                               ((size_t)(max_dim + kBestCols - 1) / kBestCols)));
    SPEO_TRY_HIP(hipMalloc(&gen_base, sizeof(uint32_t)));
    SPEO_TRY_HIP(hipMemset(gen_base, 0, sizeof(uint32_t)));
    return SPEO_OK;
}

int Engine::create(const speo_engine_config &c, hipStream_t s) {
    cfg = c;
    if (c.num_islands < 1 || !c.island_size || !c.island_problem || c.num_problems < 1 ||
        !c.problems)
        return set_error(SPEO_ERR_ARG, "speo_engine_create: islands and problems are required");
    if (c.mode != SPEO_MODE_PLAIN && c.mode != SPEO_MODE_FUSED && c.mode != SPEO_MODE_EPOCH)
        return set_error(SPEO_ERR_ARG, "speo_engine_create: unknown mode");
    if (c.precision < SPEO_PREC_FP32 || c.precision > SPEO_PREC_BF16X6)
        return set_error(SPEO_ERR_ARG, "speo_engine_create: unknown precision");
    if (c.migration_size < 0 || c.interval < 0 || !(c.min_bound < c.max_bound))
        return set_error(SPEO_ERR_ARG, "speo_engine_create: bad migration or bounds");
    if (c.rows_per_block != 0 && c.rows_per_block != 16 && c.rows_per_block != 32 &&
        c.rows_per_block != 64)
        return set_error(SPEO_ERR_ARG, "speo_engine_create: rows_per_block must be 0, 16, 32, 64");
    problems.assign(c.problems, c.problems + c.num_problems);
    for (auto *q : problems) {
        if (!q) return set_error(SPEO_ERR_ARG, "speo_engine_create: null problem");
        if (c.precision != SPEO_PREC_FP32 && !q->h.generic)
            for (int k = 0; k < q->h.ncomp; ++k)
                if (q->h.comp[k].unrotated)
                    return set_error(SPEO_ERR_UNSUPPORTED,
                                     "speo_engine_create: a 16-bit rotation precision would round "
                                     "an unrotated component's z; use SPEO_PREC_FP32 for it");
    }
    I = c.num_islands;
    for (int i = 0; i < I; ++i) {
        const int pr = c.island_problem[i];
        if (pr >= 0 && pr < c.num_problems && problems[(size_t)pr]->h.dim > kTLD) all_small = false;
    }
    // When the fused kernel reads its trial rows back from global memory
    // (dim > kTLD), rows start on 128-byte lines so that no cache line holds
    // rows of two tiles (two blocks).
    const int ld_align = all_small ? 4 : 32;
    int64_t eoff = 0;
    row_off.assign((size_t)I + 1, 0);
    for (int i = 0; i < I; ++i) {
        const int np = c.island_size[i], pr = c.island_problem[i];
        if (np < 8 || pr < 0 || pr >= c.num_problems || np < 2 * c.migration_size)
            return set_error(SPEO_ERR_ARG, "speo_engine_create: island size must be >= 8 and "
                                           ">= 2 * migration_size; problem index in range");
        IslandDesc d{};
        d.elem_off = eoff;
        d.row_off = row_off[(size_t)i];
        d.np = np;
        d.dim = problems[(size_t)pr]->h.dim;
        d.ld = round_up(d.dim, ld_align);
        d.problem = pr;
        d.F = c.island_F ? c.island_F[i] : c.F;
        d.CR = c.island_CR ? c.island_CR[i] : c.CR;
        isl.push_back(d);
        eoff += (int64_t)np * d.ld;
        row_off[(size_t)i + 1] = row_off[(size_t)i] + np;
        max_dim = std::max(max_dim, d.dim);
        max_np = std::max(max_np, np);
        max_ld = std::max(max_ld, d.ld);
    }
    total_rows = row_off[(size_t)I];
    total_elems = eoff;
    // Ring per problem: island i sends to the next island (by index) that
    // solves the same problem; islands alone on their problem send nothing.
    dst.assign((size_t)I, -1);
    for (int i = 0; i < I; ++i) {
        for (int k = 1; k < I; ++k) {
            const int j = (i + k) % I;
            if (c.island_problem[j] == c.island_problem[i]) {
                dst[(size_t)i] = j;
                break;
            }
        }
    }
    if (s) {
        stream = s;
    } else {
        SPEO_TRY_HIP(hipStreamCreateWithFlags(&stream, hipStreamNonBlocking));
        own_stream = true;
    }
    SPEO_TRY(upload_tables());
    if (!all_small) SPEO_TRY(build_wide_items());
    if (any_generic && (c.mode != SPEO_MODE_PLAIN || c.surrogate_candidates > 0))
        return set_error(SPEO_ERR_UNSUPPORTED,
                         "speo_engine_create: objectives 9-22 run in SPEO_MODE_PLAIN without the surrogate");
    const size_t E = (size_t)total_elems, R = (size_t)total_rows;
    SPEO_TRY_HIP(hipMalloc(&X, sizeof(float) * E));
    for (int b = 0; b < 2; ++b) {
        SPEO_TRY_HIP(hipMalloc(&U[b], sizeof(float) * E));
        SPEO_TRY_HIP(hipMalloc(&fX[b], sizeof(float) * R));
        SPEO_TRY_HIP(hipMalloc(&fU[b], sizeof(float) * R));
        SPEO_TRY_HIP(hipMemsetAsync(U[b], 0, sizeof(float) * E, stream));
    }
    for (int i = 0; i < I; ++i) {
        const IslandDesc &d = isl[(size_t)i];
        SPEO_TRY(init_population(X + d.elem_off, d.ld, d.np, d.dim, c.min_bound, c.max_bound,
                                 c.seed, (uint32_t)d.row_off, stream));
    }
    for (int b = 0; b < 2; ++b) {
        hipLaunchKernelGGL(k_fill, dim3(256), dim3(256), 0, stream, fU[b], total_rows, INFINITY);
        SPEO_TRY(check_launch("k_fill"));
    }
    configured = c.subisland_size != 0 || c.de_strategy != 0 || c.configure_EA != 0 ||
                 c.regroup_option != 0;
    if (configured) {
        if (c.mode != SPEO_MODE_PLAIN || c.use_graph || c.surrogate_candidates > 0)
            return set_error(SPEO_ERR_UNSUPPORTED, "speo_engine_create: sub-islands, strategies and "
                                                   "regroups run in SPEO_MODE_PLAIN without graphs "
                                                   "or the surrogate");
        if (c.de_strategy < 0 || c.de_strategy > 9 || c.configure_EA < 0 || c.configure_EA > 1 ||
            c.regroup_option < 0 || c.regroup_option > 3 || c.subisland_size < 0 ||
            (c.subisland_size > 0 && c.subisland_size < 4))
            return set_error(SPEO_ERR_ARG, "speo_engine_create: bad sub-island options");
        for (int i = 0; i < I; ++i) {
            const int np = isl[(size_t)i].np;
            if (c.subisland_size > 0 && np % c.subisland_size)
                return set_error(SPEO_ERR_ARG, "speo_engine_create: subisland_size must divide "
                                               "every island size");
            if ((c.regroup_option == SPEO_REGROUP_DYNAMIC_RANDOM ||
                 c.regroup_option == SPEO_REGROUP_DYNAMIC_ORDERED) &&
                ((np & (np - 1)) != 0 || np < 4))
                return set_error(SPEO_ERR_ARG, "speo_engine_create: dynamic regroups need islands "
                                               "of 4 * 2^k rows");
        }
    }
    if (!configured) SPEO_TRY(donor_setup());
    if (c.surrogate_candidates > 0 && c.mode != SPEO_MODE_PLAIN)
        return set_error(SPEO_ERR_UNSUPPORTED, "speo_engine_create: the surrogate runs in "
                                               "SPEO_MODE_PLAIN");
    if (cfg.mode == SPEO_MODE_EPOCH && cfg.epoch_parts == 0 && !tuning_child) {
        SPEO_TRY(tune_epoch_parts());
        if (cfg.epoch_parts > 0) SPEO_TRY(tune_launches());
    }
    if (cfg.mode == SPEO_MODE_EPOCH) SPEO_TRY(epoch_setup());
    rt = c.rows_per_block;
    if (rt == 0) SPEO_TRY(autotune());
    if (c.surrogate_candidates > 0) SPEO_TRY(surrogate_setup());
    if (configured) SPEO_TRY(configure_setup());
    SPEO_TRY(build_tiles(rt));
    SPEO_TRY(build_tiles(kTrialRows));
    // Initial evaluation (island_EA.cc:81 counts it as island_size FEs).
    if (all_small) {
        GenerationArgs a{};
        a.isl = isl_dev;
        a.tiles = tiles_dev[rt];
        a.probs = probs_dev;
        a.eval_src = X;
        a.eval_out = fX[0];
        a.composed = composed;
        SPEO_TRY(launch_any(rt, cfg.precision, kModeEval, a, ntiles[rt], stream));
    } else {
        SPEO_TRY(eval_wide_rows(X, fX[0], rt, stream));
    }
    SPEO_TRY(eval_generic_islands(X, fX[0], stream));
    hipLaunchKernelGGL(k_fill, dim3(256), dim3(256), 0, stream, fX[1], total_rows, INFINITY);
    SPEO_TRY(check_launch("k_fill"));
    fes = total_rows;
    SPEO_TRY_HIP(hipStreamSynchronize(stream));
    return SPEO_OK;
}

// Plans of all islands for `parts` workgroups per island; fails when one
// does not fit.
int Engine::epoch_plan_all(int parts, std::vector<EpochPlan> *plans, int *lds) {
    plans->assign((size_t)I, EpochPlan{});
    *lds = 0;
    for (int i = 0; i < I; ++i) {
        const IslandDesc &d = isl[(size_t)i];
        const EpochPlan p = epoch_plan(d.np, d.dim, parts, precision_parts(cfg.precision));
        if (p.lds_bytes > kEpochLdsMax) return SPEO_ERR_UNSUPPORTED;
        if (parts > 1 && d.np < 16 * parts) return SPEO_ERR_UNSUPPORTED;
        (*plans)[(size_t)i] = p;
        *lds = std::max(*lds, p.lds_bytes);
    }
    return SPEO_OK;
}

// Plans the epoch kernel.  With fewer islands than compute units an island
// is split over `parts` workgroups, one generation per launch
// (cfg.epoch_parts = 0: the largest power of two up to 8 with islands x parts
// <= compute units whose plans fit in LDS; else as configured); otherwise one
// workgroup per island runs whole epochs.  Workgroup b serves island b % I,
// share b / I.
int Engine::epoch_setup() {
    for (int i = 0; i < I; ++i) {
        const ProblemHost &P = problems[(size_t)isl[(size_t)i].problem]->h;
        if (P.ncomp != 1 || P.dim > kSmallD)
            return set_error(SPEO_ERR_UNSUPPORTED, "epoch mode needs single-component objectives "
                                                   "with dim <= 128");
        if (P.view(0, cfg.precision).objective > SPEO_OBJ_ACKLEY)
            return set_error(SPEO_ERR_UNSUPPORTED, "epoch mode: objectives 1-5 only");
        if (isl[(size_t)i].np > 8192)
            return set_error(SPEO_ERR_UNSUPPORTED, "epoch mode: islands of at most 8192 rows");
        // the epoch kernel reads an island's rows as one block of np * 4 ceil(dim / 4) floats
        if (isl[(size_t)i].ld != round_up(P.dim, 4))
            return set_error(SPEO_ERR_UNSUPPORTED, "epoch mode: unexpected population row stride");
    }
    int dev = 0, cus = 0;
    SPEO_TRY_HIP(hipGetDevice(&dev));
    SPEO_TRY_HIP(hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev));
    if (cfg.epoch_parts < 0 || cfg.epoch_parts > kEpochMaxParts ||
        (cfg.epoch_parts & (cfg.epoch_parts - 1)) != 0)
        return set_error(SPEO_ERR_ARG, "epoch_parts must be 0 (automatic), 1, 2, 4 or 8");
    int parts = cfg.epoch_parts;
    if (parts == 0) {
        parts = 1;
        while (parts < kEpochMaxParts && (int64_t)I * parts * 2 <= cus) parts *= 2;
    }
    std::vector<EpochPlan> plans;
    int lds = 0;
    while (epoch_plan_all(parts, &plans, &lds) != SPEO_OK) {
        if (parts == 1) return set_error(SPEO_ERR_UNSUPPORTED, "epoch mode: island too large for one workgroup");
        if (cfg.epoch_parts > 1)
            return set_error(SPEO_ERR_UNSUPPORTED, "epoch mode: islands cannot be split that far");
        parts /= 2;
    }
    epoch_parts = parts;
    epoch_lds = lds;
    epoch_blocks = I * parts;
    std::vector<EpochBlock> blocks((size_t)epoch_blocks);
    for (int b = 0; b < epoch_blocks; ++b) {
        const int i = b % I;
        const IslandDesc &d = isl[(size_t)i];
        const ProblemHost &P = problems[(size_t)d.problem]->h;
        const CompDev c = P.view(0, cfg.precision);
        EpochBlock &e = blocks[(size_t)b];
        e.I = d;
        e.pl = plans[(size_t)i];
        e.share = b / I;
        e.objective = c.objective;
        e.kp32 = c.kp32;
        const uint64_t ng = (uint64_t)(d.dim + 3) / 4;
        e.inv_ng = ng > 1 ? (uint32_t)((0x100000000ull + ng - 1) / ng) : 0u;
        e.crt = cr_threshold(d.CR);
        e.rate = c.rate;
        e.lambda = (float)P.comp[0].lambda;
        e.bias = (float)P.comp[0].bias;
        e.shift = c.shift;
        e.B32s = c.B32s;
        e.colw = c.colw;
        for (int q = 0; q < 3; ++q) e.M16s[q] = c.M16s[q];
        e.heavy = c.heavy;
    }
    SPEO_TRY(upload_vec(&blocks_dev, blocks));
    if (parts > 1) {
        SPEO_TRY_HIP(hipMalloc(&Xnext, sizeof(float) * (size_t)total_elems));
        SPEO_TRY_HIP(hipMemcpy(Xnext, X, sizeof(float) * (size_t)total_elems, hipMemcpyDeviceToDevice));
    }
    return SPEO_OK;
}

// The buffer of donors drawn ahead, 16 bytes a row and generation: at most 64
// generations, none past a migration point (a chunk ends there), and outside
// epoch mode, whose kernel runs a whole chunk from it, no more than the
// population's own bytes or 64 MiB: by then one generation's draw fills the chip.
// A surrogate engine draws its own donors and has one generation for profiles.
int Engine::donor_setup() {
    std::vector<int> row_island((size_t)total_rows);
    for (int i = 0; i < I; ++i)
        for (int r = 0; r < isl[(size_t)i].np; ++r) row_island[(size_t)(isl[(size_t)i].row_off + r)] = i;
    SPEO_TRY(upload_vec(&row_island_dev, row_island));
    int64_t ahead = std::min<int64_t>(64, (int64_t(1) << 26) / total_rows);
    if (cfg.interval > 0 && cfg.migration_size > 0) ahead = std::min<int64_t>(ahead, cfg.interval);
    if (cfg.mode != SPEO_MODE_EPOCH)
        ahead = std::min(ahead, std::max<int64_t>(int64_t(64) << 20, 4 * total_elems) / (16 * (int64_t)total_rows));
    if (cfg.surrogate_candidates > 0) ahead = 1;
    donor_gens = (int)std::max<int64_t>(1, ahead);
    SPEO_TRY_HIP(hipMalloc(&donor_buf, sizeof(int4) * (size_t)donor_gens * (size_t)total_rows));
    return SPEO_OK;
}

void Engine::swap_epoch_buffers() {
    std::swap(X, Xnext);
    std::swap(fX[0], fX[1]);
    ep_par ^= 1;
}

// Chunks of at most donor_gens generations: the donors of the chunk are drawn
// first, then one launch runs the chunk (one workgroup per island) or one
// launch per generation runs it (split islands, swapping the population
// buffers).
int Engine::launch_epoch_chunk(int L, hipStream_t s) {
    if (by_launches) return enqueue_plain(L, s);
    EpochArgs a{};
    a.blocks = blocks_dev;
    a.Xalt = U[1];
    a.U = U[0];
    a.fU = fU[0];
    a.lo = cfg.min_bound;
    a.hi = cfg.max_bound;
    a.seed = cfg.seed;
    a.gen_base = gen_base;
    a.donors = donor_buf;
    a.rows = total_rows;
    for (int g0 = 0; g0 < L; g0 += donor_gens) {
        const int Ls = std::min(donor_gens, L - g0);
        SPEO_TRY(prof_begin(5, Ls, s));
        SPEO_TRY(epoch_donors(isl_dev, row_island_dev, total_rows, Ls, cfg.seed, gen_base,
                              (uint32_t)g0, donor_buf, s));
        SPEO_TRY(prof_end(s));
        if (epoch_parts == 1) {
            a.Xin = X;
            a.Xout = X;
            a.fXin = fX[0];
            a.fXout = fX[0];
            a.gen_offset = (uint32_t)g0;
            a.donor_gen = 0;
            a.L = Ls;
            a.write_trials = 1;
            SPEO_TRY(prof_begin(4, Ls, s));
            SPEO_TRY(launch_epoch(cfg.precision, a, epoch_blocks, epoch_lds, epoch_parts > 1, s));
            SPEO_TRY(prof_end(s));
            continue;
        }
        SPEO_TRY(prof_begin(4, Ls, s));  // one event pair around the sub-chunk's launches
        for (int g = 0; g < Ls; ++g) {
            a.Xin = X;
            a.Xout = Xnext;
            a.fXin = fX[0];
            a.fXout = fX[1];
            a.gen_offset = (uint32_t)(g0 + g);
            a.donor_gen = g;
            a.L = 1;
            a.write_trials = g0 + g == L - 1;
            SPEO_TRY(launch_epoch(cfg.precision, a, epoch_blocks, epoch_lds, epoch_parts > 1, s));
            swap_epoch_buffers();
        }
        SPEO_TRY(prof_end(s));
    }
    return SPEO_OK;
}

int Engine::surrogate_setup() {
    C = cfg.surrogate_candidates;
    const int D = isl[0].dim;
    for (const auto &d : isl)
        if (d.dim != D) return set_error(SPEO_ERR_ARG, "surrogate: all islands must share one dimension");
    if (C > 32 || cfg.num_problems > kMaxSurrProblems || cfg.surrogate_archive < 1024 ||
        cfg.surrogate_batch < 16 || cfg.surrogate_steps < 0 || cfg.surrogate_train_interval < 1 ||
        !(cfg.surrogate_lr > 0.f))
        return set_error(SPEO_ERR_ARG, "surrogate: need <= 32 candidates, <= 16 problems, archive "
                                       ">= 1024, batch >= 16, train interval >= 1, lr > 0");
    Kp = round_up(D, 32);
    std::vector<SurrRowDesc> rows;
    std::vector<int> qrel((size_t)I, 0);
    for (int p = 0; p < cfg.num_problems; ++p) {
        auto sp = std::make_unique<SurrProblem>();
        sp->qoff = (int)rows.size();
        for (int i = 0; i < I; ++i)
            if (isl[(size_t)i].problem == p) {
                qrel[(size_t)i] = (int)rows.size() - sp->qoff;
                for (int li = 0; li < isl[(size_t)i].np; ++li)
                    rows.push_back(SurrRowDesc{isl[(size_t)i].row_off + li, i, p, li});
            }
        sp->rows = (int)rows.size() - sp->qoff;
        if (sp->rows > 0) {
            const int mb = std::max({cfg.surrogate_batch, sp->rows * C, 1024});
            SPEO_TRY(sp->net.alloc(D, mb));
            SPEO_TRY(sp->net.init(cfg.seed ^ (0x9E3779B97F4A7C15ull * (uint64_t)(p + 1)), stream));
        }
        surr.push_back(std::move(sp));
    }
    Q = (int)rows.size();
    SPEO_TRY(upload_vec(&srows_dev, rows));
    const size_t P = (size_t)cfg.num_problems, cap = (size_t)cfg.surrogate_archive;
    SPEO_TRY_HIP(hipMalloc(&cand, sizeof(float) * (size_t)Q * C * Kp));
    SPEO_TRY_HIP(hipMalloc(&pred, sizeof(float) * (size_t)Q * C));
    SPEO_TRY(upload_vec(&rho_dev, std::vector<float>(P, -1.0f)));
    SPEO_TRY(upload_vec(&scored_dev, std::vector<long long>(P, 0)));
    SPEO_TRY_HIP(hipMalloc(&AX, sizeof(float) * P * cap * Kp));
    SPEO_TRY_HIP(hipMalloc(&Ay, sizeof(float) * P * cap));
    SPEO_TRY_HIP(hipMalloc(&Xb, sizeof(float) * (size_t)cfg.surrogate_batch * Kp));
    SPEO_TRY_HIP(hipMalloc(&tb, sizeof(float) * (size_t)cfg.surrogate_batch));
    SPEO_TRY_HIP(hipMalloc(&Xh, sizeof(float) * 1024 * (size_t)Kp));
    SPEO_TRY_HIP(hipMalloc(&yh, sizeof(float) * 1024));
    SPEO_TRY_HIP(hipMalloc(&predh, sizeof(float) * 1024));
    SPEO_TRY_HIP(hipMalloc(&ranks_ws, sizeof(float2) * 4096));
    SPEO_TRY_HIP(hipMalloc(&heads_dev, sizeof(int) * kMaxSurrProblems));
    // (the first generation's pick advances the heads to slot 0)
    std::vector<int> head0(kMaxSurrProblems, 0);
    for (size_t p = 0; p < surr.size(); ++p)
        head0[p] = (cfg.surrogate_archive - surr[p]->rows % cfg.surrogate_archive) % cfg.surrogate_archive;
    SPEO_TRY_HIP(hipMemcpy(heads_dev, head0.data(), sizeof(int) * head0.size(), hipMemcpyHostToDevice));
    SPEO_TRY(upload_vec(&qrel_dev, qrel));
    SPEO_TRY_HIP(hipMalloc(&drawn, sizeof(int4) * (size_t)Q * C));
    SPEO_TRY_HIP(hipMalloc(&round_dev, sizeof(uint32_t)));
    SPEO_TRY_HIP(hipMemset(round_dev, 0, sizeof(uint32_t)));
    return SPEO_OK;
}

// One surrogate-screened generation: C candidates per target (only candidate
// 0 before the first training round), MLP scores, pick, true evaluation of
// the picked trial, archive append, selection.
int Engine::surrogate_generation(int gen_offset, hipStream_t s) {
    const int Ce = any_trained ? C : 1;
    last_Ce = Ce;
    const float rho_min = any_trained ? cfg.surrogate_rho_min : INFINITY;
    const float lo = cfg.min_bound, hi = cfg.max_bound;
    SurrArchive ar{};
    for (size_t p = 0; p < surr.size(); ++p) {
        ar.heads.qoff[p] = surr[p]->qoff;
        ar.heads.rows[p] = surr[p]->rows;
    }
    ar.problems = (int)surr.size();
    ar.cap = cfg.surrogate_archive;
    ar.head_dev = heads_dev;
    if (retain_cand || Kp > kFusedMaxKp) {
        // candidates written to memory, scored, the pick copied
        SPEO_TRY(gen_candidates(isl_dev, srows_dev, Q, Ce, X, lo, hi, cfg.seed, gen_base,
                                (uint32_t)gen_offset, cand, Kp, s));
        if (any_trained) {
            for (auto &sp : surr)
                if (sp->rows > 0)
                    SPEO_TRY(sp->net.infer(cand + (size_t)sp->qoff * Ce * Kp, Kp, sp->rows * Ce,
                                           pred + (size_t)sp->qoff * Ce, s));
            surr_pred += (int64_t)Q * Ce;
        }
        SPEO_TRY(pick_candidates(isl_dev, srows_dev, Q, Ce, cand, Kp, pred, rho_dev, rho_min, U[0], ar, s));
    } else {
        // candidates generated and scored in one kernel per problem, the pick
        // generated again into U: the same trials without the candidate buffer
        if (any_trained) {
            std::vector<Mlp *> nets;
            std::vector<int> qo, nq, pi;
            for (size_t p = 0; p < surr.size(); ++p)
                if (surr[p]->rows > 0) {
                    nets.push_back(&surr[p]->net);
                    qo.push_back(surr[p]->qoff);
                    nq.push_back(surr[p]->rows);
                    pi.push_back((int)p);
                }
            SPEO_TRY(cand_infer(nets.data(), qo.data(), nq.data(), pi.data(), (int)nets.size(), isl_dev,
                                srows_dev, Ce, X, lo, hi, cfg.seed, gen_base, (uint32_t)gen_offset,
                                rho_dev, rho_min, scored_dev, pred, drawn, s));
        }
        SPEO_TRY(pick_regen(isl_dev, srows_dev, Q, Ce, pred, drawn, rho_dev, rho_min, X, lo, hi, cfg.seed,
                            gen_base, (uint32_t)gen_offset, U[0], ar, s));
    }
    for (auto &sp : surr) {  // host copies of the device heads
        sp->head = (int)(((int64_t)sp->head + sp->rows) % cfg.surrogate_archive);
        sp->appended += sp->rows;
    }
    // up to 128 columns the evaluation appends and selects as well
    if (all_small) return launch(kModeEval, gen_offset, rt, s, 0, true);
    SPEO_TRY(launch(kModeEval, gen_offset, rt, s));
    SPEO_TRY(archive_append(isl_dev, srows_dev, Q, U[0], fU[0], AX, Ay, Kp, ar, s));
    return launch(kModeSelect, gen_offset, rt, s);
}

int Engine::surrogate_train(hipStream_t s) {
    const size_t cap = (size_t)cfg.surrogate_archive;
    std::vector<size_t> todo;
    for (size_t p = 0; p < surr.size(); ++p) {
        SurrProblem &sp = *surr[p];
        if (sp.rows == 0) continue;
        const int n_valid = (int)std::min<int64_t>(sp.appended, (int64_t)cap);
        if (n_valid < std::max(cfg.surrogate_batch, 512)) continue;
        SPEO_TRY(mean_std(Ay + p * cap, n_valid, sp.net.stats, s));
        todo.push_back(p);
    }
    auto seed_of = [&](size_t p) { return cfg.seed ^ (0xD1B54A32D192ED03ull * (p + 1)); };
    auto n_valid_of = [&](size_t p) { return (int)std::min<int64_t>(surr[p]->appended, (int64_t)cap); };
    if (!todo.empty() && Kp <= kFusedMaxKp) {
        // every problem's network takes its step in the same two launches
        std::vector<Mlp *> nets;
        std::vector<const float *> ax, ay;
        std::vector<int> nv;
        std::vector<uint64_t> seeds;
        for (size_t p : todo) {
            nets.push_back(&surr[p]->net);
            ax.push_back(AX + p * cap * Kp);
            ay.push_back(Ay + p * cap);
            nv.push_back(n_valid_of(p));
            seeds.push_back(seed_of(p));
        }
        for (int step = 0; step < cfg.surrogate_steps; ++step)
            SPEO_TRY(train_steps(nets.data(), ax.data(), ay.data(), nv.data(), seeds.data(),
                                 (int)todo.size(), round_dev, (uint32_t)step, cfg.surrogate_batch,
                                 cfg.surrogate_lr, step == cfg.surrogate_steps - 1, s));
        for (Mlp *n : nets) SPEO_TRY(add_i32(n->t_dev, cfg.surrogate_steps, s));
    } else {
        for (size_t p : todo)
            for (int step = 0; step < cfg.surrogate_steps; ++step)
                SPEO_TRY(surr[p]->net.train_step(AX + p * cap * Kp, Ay + p * cap, n_valid_of(p),
                                                 seed_of(p), (uint32_t)surr_rounds, (uint32_t)step,
                                                 cfg.surrogate_batch, cfg.surrogate_lr,
                                                 step == cfg.surrogate_steps - 1, Xb, tb, s));
    }
    for (size_t p : todo) {
        SurrProblem &sp = *surr[p];
        if (sp.net.bf16_stale) SPEO_TRY(sp.net.refresh_bf16(s));
        const int H = std::min(1024, n_valid_of(p) / 8);
        SPEO_TRY(gather_holdout(AX + p * cap * Kp, Ay + p * cap, H, Kp, Xh, yh, s));
        SPEO_TRY(sp.net.infer(Xh, Kp, H, predh, s));
        SPEO_TRY(spearman(predh, yh, H, rho_dev + p, ranks_ws, s));
        sp.trained = true;
        any_trained = true;
    }
    ++surr_rounds;
    hipLaunchKernelGGL(k_add_u32, dim3(1), dim3(64), 0, s, round_dev, 1u);
    return check_launch("k_add_u32");
}

int Engine::launch(int mode, int gen_offset, int rt_, hipStream_t s, int clear, bool append) {
    GenerationArgs a{};
    a.isl = isl_dev;
    a.tiles = tiles_dev[rt_];
    a.probs = probs_dev;
    a.X = X;
    a.lo = cfg.min_bound;
    a.hi = cfg.max_bound;
    a.seed = cfg.seed;
    a.gen_base = gen_base;
    a.gen_offset = (uint32_t)gen_offset;
    a.donors = donor_buf ? donor_buf + (size_t)(gen_offset % donor_gens) * (size_t)total_rows : nullptr;
    a.clear_trials = clear;
    a.composed = composed;
    switch (mode) {
    case kModeGen:
        a.U_new = U[0];
        break;
    case kModeEval:
        if (!all_small) return eval_wide_rows(U[0], fU[0], rt_, s);
        a.eval_src = U[0];
        a.eval_out = fU[0];
        if (append) {
            a.fX_new = fX[0];
            a.append = AppendArgs{AX, Ay, qrel_dev, heads_dev, cfg.surrogate_archive, Kp};
        }
        break;
    case kModeSelect:
        if (cfg.mode == SPEO_MODE_FUSED) {  // apply the pending selection
            a.U_prev = U[p];
            a.fU_prev = fU[p];
            a.fX_prev = a.fX_new = fX[p];
        } else {
            a.U_prev = U[0];
            a.fU_prev = fU[0];
            a.fX_prev = fX[pf];
            a.fX_new = fX[0];
        }
        break;
    default: {
        const bool fused = cfg.mode == SPEO_MODE_FUSED;
        const int u = fused ? p : pu, f = fused ? p : pf;
        a.pending = fused || pending;
        a.fX_prev = fX[f];
        a.U_prev = U[u];
        a.fU_prev = fU[u];
        a.fX_new = fX[1 - f];
        a.U_new = U[1 - u];
        a.fU_new = fU[1 - u];
        if (!all_small) {
            a.tiles = tiles_dev[kTrialRows];
            SPEO_TRY(launch_trials(kModeFusedGen, a, ntiles[kTrialRows], s));
            return eval_wide_rows(a.U_new, a.fU_new, rt_, s);
        }
        break;
    }
    }
    if (mode == kModeGen || mode == kModeSelect) {
        a.tiles = tiles_dev[kTrialRows];
        return launch_trials(mode, a, ntiles[kTrialRows], s);
    }
    return launch_any(rt_, cfg.precision, mode, a, ntiles[rt_], s);
}

// Donors and j_rand of generations [gen_offset, gen_offset + L), L <= donor_gens,
// into donor_buf, where launch() reads generation g's at g % donor_gens.
int Engine::draw_ahead(int gen_offset, int L, hipStream_t s) {
    return epoch_donors(isl_dev, row_island_dev, total_rows, L, cfg.seed, gen_base, (uint32_t)gen_offset,
                        donor_buf, s);
}

// L generations of a plain engine (or of an epoch engine that runs by launches)
// as L fused launches and one selection: L + 1
// launches instead of 3 L (100 rows, D = 10, ten generations and the best:
// 144 us as separate launches, 100 us so).  The parities are chosen so that the
// last trials end in U[0], fU[0] and the last selection writes fX[0]: the
// buffers the three separate launches leave.
int Engine::enqueue_plain(int L, hipStream_t s) {
    pf = 0;
    pu = L & 1;
    pending = false;
    for (int g = 0; g < L; ++g) {
        if (g % donor_gens == 0) {
            const int Ls = std::min(donor_gens, L - g);
            if (g > 0) SPEO_TRY(prof_end(s));
            SPEO_TRY(prof_begin(5, Ls, s));
            SPEO_TRY(draw_ahead(g, Ls, s));
            SPEO_TRY(prof_end(s));
            SPEO_TRY(prof_begin(4, Ls, s));
        }
        SPEO_TRY(launch(kModeFused, g, rt, s));
        pf = 1 - pf;
        pu = 1 - pu;
        pending = true;
    }
    if (L > 0) {
        SPEO_TRY(launch(kModeSelect, 0, rt, s));
        SPEO_TRY(prof_end(s));
    }
    pf = pu = 0;
    pending = false;
    return SPEO_OK;
}

// ------------------------------------------------- sub-islands (plain mode)

int Engine::configure_setup() {
    doff.assign((size_t)I + 1, 0);
    subs_h.assign((size_t)I, 1);
    perm_h.resize((size_t)I);
    info_h.resize((size_t)I);
    base_h.resize((size_t)I);
    for (int i = 0; i < I; ++i) {
        const IslandDesc &d = isl[(size_t)i];
        doff[(size_t)i + 1] = doff[(size_t)i] + d.np / 4;
        subs_h[(size_t)i] = cfg.subisland_size > 0 ? d.np / cfg.subisland_size : 1;
        perm_h[(size_t)i].resize((size_t)d.np);
        for (int r = 0; r < d.np; ++r) perm_h[(size_t)i][(size_t)r] = r;
        info_h[(size_t)i].assign((size_t)(d.np / 4), DEInfo{});
        // DE_CUDA::Initilize: CR 0.9, F 0.5, strategy 4 (DE_CUDA.cc:61-63);
        // here the engine's per-island F, CR and strategy
        base_h[(size_t)i] = DEInfo{d.CR, d.F, cfg.de_strategy ? cfg.de_strategy - 1 : 4, -1};
    }
    SPEO_TRY_HIP(hipMalloc(&perm_dev, sizeof(int) * (size_t)total_rows));
    SPEO_TRY_HIP(hipMalloc(&info_dev, sizeof(DEInfo) * (size_t)std::max(1, doff[(size_t)I])));
    SPEO_TRY_HIP(hipMalloc(&best_sub_dev, sizeof(int) * (size_t)std::max(1, doff[(size_t)I])));
    return regroup(true);
}

// One regroup event of every island (event 0: the initial ConfigureEA),
// then the new partitions and configurations uploaded.
int Engine::regroup(bool initial) {
    const int event = initial ? 0 : ++regroup_events;
    const bool noop = !initial && cfg.regroup_option == SPEO_REGROUP_STATIC_ORDERED;
    if (noop) return SPEO_OK;
    SPEO_TRY_HIP(hipStreamSynchronize(stream));  // the previous upload's host arrays
    for (int i = 0; i < I; ++i) {
        const IslandDesc &d = isl[(size_t)i];
        int subs = subs_h[(size_t)i];
        SPEO_TRY(speo_island_regroup(cfg.seed, i, event, cfg.regroup_option, cfg.configure_EA,
                                     d.np, subs, perm_h[(size_t)i].data(), &base_h[(size_t)i],
                                     info_h[(size_t)i].data(), &subs));
        subs_h[(size_t)i] = subs;
        SPEO_TRY_HIP(hipMemcpy(perm_dev + d.row_off, perm_h[(size_t)i].data(), sizeof(int) * d.np,
                               hipMemcpyHostToDevice));
        SPEO_TRY_HIP(hipMemcpy(info_dev + doff[(size_t)i], info_h[(size_t)i].data(),
                               sizeof(DEInfo) * (size_t)subs, hipMemcpyHostToDevice));
    }
    return SPEO_OK;
}

// The generation of every island through the reference's operator kernel
// (sub-islands, permutation, per sub-island DEInfo, strategies 0-8), one
// launch per island; strategies that use the best member get each
// sub-island's best slot first (global_DE_FindBestIndividualInIsland).
int Engine::generate_configured(int gen_offset, hipStream_t s) {
    const uint32_t gen = (uint32_t)(gens + gen_offset);
    for (int i = 0; i < I; ++i) {
        const IslandDesc &d = isl[(size_t)i];
        const int subs = subs_h[(size_t)i], S = d.np / subs;
        bool need_best = false;
        for (int q = 0; q < subs; ++q) {
            const int st = info_h[(size_t)i][(size_t)q].strategy_ID;
            need_best = need_best || st == 2 || st == 3 || st == 6 || st == 7;
        }
        int *best = best_sub_dev + doff[(size_t)i];
        if (need_best) SPEO_TRY(subisland_best(fX[0] + d.row_off, perm_dev + d.row_off, S, subs, best, s));
        GenArgs a{U[0] + d.elem_off, X + d.elem_off, d.ld, d.np, d.dim, S, perm_dev + d.row_off,
                  info_dev + doff[(size_t)i], need_best ? best : nullptr, cfg.min_bound,
                  cfg.max_bound, cfg.seed, gen, (uint32_t)d.row_off, nullptr, 0, nullptr, nullptr,
                  nullptr};
        SPEO_TRY(de_generate(a, s));
    }
    return SPEO_OK;
}

int Engine::subislands(int island, int *subs_out, int *perm_out, DEInfo *info_out) {
    if (island < 0 || island >= I) return set_error(SPEO_ERR_ARG, "speo_engine_subislands: bad island");
    const int np = isl[(size_t)island].np;
    if (!configured) {
        if (subs_out) *subs_out = 1;
        if (perm_out)
            for (int r = 0; r < np; ++r) perm_out[r] = r;
        if (info_out) info_out[0] = DEInfo{isl[(size_t)island].CR, isl[(size_t)island].F, 4, np};
        return SPEO_OK;
    }
    SPEO_TRY_HIP(hipStreamSynchronize(stream));
    const int subs = subs_h[(size_t)island];
    if (subs_out) *subs_out = subs;
    if (perm_out) std::copy(perm_h[(size_t)island].begin(), perm_h[(size_t)island].end(), perm_out);
    if (info_out)
        for (int q = 0; q < subs; ++q) info_out[q] = info_h[(size_t)island][(size_t)q];
    return SPEO_OK;
}

// Islands whose problem the generic kernel evaluates: one launch per island.
int Engine::eval_generic_islands(const float *src, float *out, hipStream_t s) {
    if (!any_generic) return SPEO_OK;
    for (int i = 0; i < I; ++i) {
        const IslandDesc &d = isl[(size_t)i];
        const ProblemHost &P = problems[(size_t)d.problem]->h;
        if (!P.generic) continue;
        SPEO_TRY(eval_problem_generic(P, src + d.elem_off, d.ld, d.np, out + d.row_off, nullptr,
                                      nullptr, 0, s));
    }
    return SPEO_OK;
}

int Engine::finalize_pending(hipStream_t s) {
    if (cfg.mode != SPEO_MODE_FUSED || !pending) return SPEO_OK;
    SPEO_TRY(launch(kModeSelect, 0, rt, s, 1));
    pending = false;
    return SPEO_OK;
}

int Engine::migrate(hipStream_t s) {
    if (cfg.migration_size <= 0) return SPEO_OK;
    SPEO_TRY(finalize_pending(s));
    const int cur = cfg.mode == SPEO_MODE_FUSED ? p : 0;
    return migrate_ring(X, fX[cur], isl_dev, row_off_dev, dst_dev, best_buf, worst_buf, I, max_np,
                        cfg.migration_size, s);
}

// Whether a plain engine's generations are fused launches (enqueue_plain).
bool Engine::runs_fused() const {
    return cfg.mode == SPEO_MODE_PLAIN && cfg.surrogate_candidates == 0 && !configured && !any_generic;
}

// L generations, then (optionally) migration, then gen_base += L.  The parity
// `p` and `pending` advance on the host as the launches are enqueued.
int Engine::enqueue_chunk(int L, bool do_migrate, hipStream_t s) {
    if (cfg.mode == SPEO_MODE_EPOCH) {
        SPEO_TRY(launch_epoch_chunk(L, s));
    } else if (runs_fused()) {
        SPEO_TRY(enqueue_plain(L, s));
    } else {
        for (int g = 0; g < L; ++g) {
            if (C == 0 && donor_buf && g % donor_gens == 0) SPEO_TRY(draw_ahead(g, std::min(donor_gens, L - g), s));
            if (C > 0) {
                SPEO_TRY(surrogate_generation(g, s));
            } else if (cfg.mode == SPEO_MODE_FUSED) {
                SPEO_TRY(launch(kModeFused, g, rt, s));
                p = 1 - p;
                pending = true;
            } else {
                if (configured)
                    SPEO_TRY(generate_configured(g, s));
                else
                    SPEO_TRY(launch(kModeGen, g, rt, s));
                SPEO_TRY(launch(kModeEval, g, rt, s));
                SPEO_TRY(eval_generic_islands(U[0], fU[0], s));
                SPEO_TRY(launch(kModeSelect, g, rt, s));
            }
        }
    }
    if (do_migrate) SPEO_TRY(migrate(s));
    hipLaunchKernelGGL(k_add_u32, dim3(1), dim3(64), 0, s, gen_base, (uint32_t)L);
    return check_launch("k_add_u32");
}

// Generations are counted from 0; migration follows generation g when
// g % interval == 0 (island_EA.cc:93-99).  Returns the generations up to and
// including the next migration point, or `left` when it lies beyond.
int Engine::next_chunk(int left, bool *mig) const {
    *mig = false;
    if (cfg.interval > 0 && cfg.migration_size > 0) {
        const int64_t g0 = gens;
        const int64_t next = (g0 % cfg.interval == 0) ? g0 : (g0 / cfg.interval + 1) * cfg.interval;
        const int64_t to_mig = next - g0 + 1;
        if (to_mig <= left) {
            *mig = true;
            return (int)to_mig;
        }
    }
    return left;
}

// A migration point of a timed run: the work before it completes, then the
// migration (and, for configured engines, the regroup) runs eagerly and its
// wall time until completion is added to comm_seconds.
int Engine::timed_point(bool mig, bool point) {
    SPEO_TRY_HIP(hipStreamSynchronize(stream));
    const auto t0 = std::chrono::steady_clock::now();
    if (mig) SPEO_TRY(migrate(stream));
    if (point && configured) SPEO_TRY(regroup(false));
    SPEO_TRY_HIP(hipStreamSynchronize(stream));
    comm_seconds += std::chrono::duration<double>(std::chrono::steady_clock::now() - t0).count();
    return SPEO_OK;
}

int Engine::prepare(int generations) {
    if (C > 0 || !cfg.use_graph || graph_failed) return SPEO_OK;
    const int64_t g0 = gens, f0 = fes, m0 = migrations, gl0 = graph_launches;
    const int p0 = p, ep0 = ep_par;
    const bool pend0 = pending;
    const int rc = run(generations, true);
    gens = g0;
    fes = f0;
    migrations = m0;
    graph_launches = gl0;
    p = p0;
    pending = pend0;
    if (ep_par != ep0) swap_epoch_buffers();
    return rc;
}

// A surrogate round: the train_interval generations up to a training point
// (migration after generation mig_pos when >= 0), the generation counter, then
// the training.  The same launches surrogate generations and training enqueue
// one by one, with the generations' counters offset within the round.
int Engine::enqueue_surrogate_round(int TI, int mig_pos, hipStream_t s) {
    for (int k = 0; k < TI; ++k) {
        SPEO_TRY(surrogate_generation(k, s));
        if (k == mig_pos) SPEO_TRY(migrate(s));
    }
    hipLaunchKernelGGL(k_add_u32, dim3(1), dim3(64), 0, s, gen_base, (uint32_t)TI);
    SPEO_TRY(check_launch("k_add_u32"));
    return surrogate_train(s);
}

// The host-side counters a replayed surrogate round advances (a captured
// round advanced them once while it was enqueued).
void Engine::surrogate_round_host(int TI) {
    const int64_t cap = cfg.surrogate_archive;
    for (int k = 0; k < TI; ++k) {
        last_Ce = any_trained ? C : 1;
        // (the one-kernel screening counts its candidates on the device)
        if (any_trained && (retain_cand || Kp > kFusedMaxKp)) surr_pred += (int64_t)Q * last_Ce;
        for (auto &sp : surr) {
            sp->head = (int)(((int64_t)sp->head + sp->rows) % cap);
            sp->appended += sp->rows;
        }
    }
    ++surr_rounds;
}

// Rounds are replayable once every network screens and every archive is full:
// then no launch argument changes from one round to the next.
bool Engine::surrogate_round_replayable() const {
    if (!any_trained || Kp > kFusedMaxKp || cfg.surrogate_archive < std::max(cfg.surrogate_batch, 512))
        return false;
    for (const auto &sp : surr)
        if (sp->rows > 0 && (!sp->trained || sp->appended < cfg.surrogate_archive)) return false;
    return true;
}

int Engine::run(int generations, bool dry) {
    if (C > 0) {
        const int TI = cfg.surrogate_train_interval;
        const bool mig_on = cfg.interval > 0 && cfg.migration_size > 0;
        int left = generations;
        while (left > 0) {
            if (cfg.use_graph && !graph_failed && !dry && gens % TI == 0 && left >= TI &&
                surrogate_round_replayable()) {
                int mig_pos = -1, nmig = 0;
                for (int k = 0; k < TI && mig_on; ++k)
                    if ((gens + k) % cfg.interval == 0) {
                        mig_pos = k;
                        ++nmig;
                    }
                if (nmig <= 1) {
                    const auto key = std::make_tuple(-TI, mig_pos, retain_cand ? 1 : 0);
                    auto it = graphs.find(key);
                    bool captured = false;
                    if (it == graphs.end()) {
                        hipGraph_t g = nullptr;
                        hipGraphExec_t ge = nullptr;
                        SPEO_TRY_HIP(hipStreamBeginCapture(stream, hipStreamCaptureModeThreadLocal));
                        const int rc = enqueue_surrogate_round(TI, mig_pos, stream);
                        hipError_t e = hipStreamEndCapture(stream, &g);
                        if (rc != SPEO_OK || e != hipSuccess ||
                            hipGraphInstantiate(&ge, g, nullptr, nullptr, 0) != hipSuccess) {
                            // the host counters advanced during the attempt: this
                            // engine cannot continue consistently
                            if (g) (void)hipGraphDestroy(g);
                            (void)hipGetLastError();
                            graph_failed = true;
                            return rc != SPEO_OK ? rc
                                                 : set_error(SPEO_ERR_HIP, "surrogate round capture failed");
                        }
                        (void)hipGraphDestroy(g);
                        it = graphs.emplace(key, ge).first;
                        captured = true;
                    }
                    SPEO_TRY_HIP(hipGraphLaunch(it->second, stream));
                    ++graph_launches;
                    if (!captured) surrogate_round_host(TI);
                    gens += TI;
                    fes += (int64_t)TI * total_rows;
                    migrations += nmig;
                    left -= TI;
                    continue;
                }
            }
            const bool mig = mig_on && gens % cfg.interval == 0;
            SPEO_TRY(enqueue_chunk(1, mig, stream));
            ++gens;
            fes += total_rows;
            if (mig) ++migrations;
            if (gens % TI == 0) SPEO_TRY(surrogate_train(stream));
            --left;
        }
        return SPEO_OK;
    }
    if (configured && !dry) {
        // generation by generation: after generation g with g % interval == 0
        // the ring migration and then the regroup of every island
        // (island_EA.cc:94-99; migrate.cc:59)
        for (int g = 0; g < generations; ++g) {
            const bool point = cfg.interval > 0 && gens % cfg.interval == 0;
            const bool mig = point && cfg.migration_size > 0;
            SPEO_TRY(enqueue_chunk(1, mig && !time_comm, stream));
            ++gens;
            fes += total_rows;
            if (mig) ++migrations;
            if (time_comm && point) {
                SPEO_TRY(timed_point(mig, true));
            } else if (point) {
                SPEO_TRY(regroup(false));
            }
        }
        return SPEO_OK;
    }
    int left = generations;
    while (left > 0) {
        bool mig_point = false;
        const int L = next_chunk(left, &mig_point);
        const bool mig = mig_point && !(time_comm && !dry);  // timed: migrate after the chunk
        const bool use_graph = cfg.use_graph && !graph_failed;
        if (use_graph) {
            const auto key = std::make_tuple(L, cfg.mode == SPEO_MODE_FUSED ? p : ep_par,
                                             (mig ? 1 : 0) | (pending ? 2 : 0));
            auto it = graphs.find(key);
            const int p_before = p;
            const bool pend_before = pending;
            const int ep_before = ep_par;
            if (it == graphs.end()) {
                hipGraph_t g = nullptr;
                hipGraphExec_t ge = nullptr;
                SPEO_TRY_HIP(hipStreamBeginCapture(stream, hipStreamCaptureModeThreadLocal));
                const int rc = enqueue_chunk(L, mig, stream);
                hipError_t e = hipStreamEndCapture(stream, &g);
                if (rc != SPEO_OK || e != hipSuccess ||
                    hipGraphInstantiate(&ge, g, nullptr, nullptr, 0) != hipSuccess) {
                    if (g) (void)hipGraphDestroy(g);
                    (void)hipGetLastError();
                    graph_failed = true;  // fall back to eager launches
                    p = p_before;
                    pending = pend_before;
                    if (ep_par != ep_before) swap_epoch_buffers();
                    continue;
                }
                (void)hipGraphDestroy(g);
                it = graphs.emplace(key, ge).first;
                // enqueue_chunk advanced the host-side parity during capture
                p = p_before;
                pending = pend_before;
                if (ep_par != ep_before) swap_epoch_buffers();
            }
            if (!dry) SPEO_TRY_HIP(hipGraphLaunch(it->second, stream));
            ++graph_launches;
            if (cfg.mode == SPEO_MODE_FUSED) {
                if (L % 2) p = 1 - p;
                pending = L > 0 ? true : pending;
                if (mig && cfg.migration_size > 0) pending = false;
            }
            if (cfg.mode == SPEO_MODE_EPOCH && epoch_parts > 1 && !by_launches && L % 2) swap_epoch_buffers();
        } else if (!dry) {
            SPEO_TRY(enqueue_chunk(L, mig, stream));
        }
        if (mig_point && !mig) SPEO_TRY(timed_point(true, false));
        gens += L;
        fes += (int64_t)L * total_rows;
        if (mig_point) ++migrations;
        left -= L;
    }
    return SPEO_OK;
}

int Engine::profile(int generations, double *avg_ms) {
    if (cfg.mode == SPEO_MODE_EPOCH) return profile_epoch(generations, avg_ms);
    const int roles = 6;
    std::vector<hipEvent_t> ev;
    std::vector<int> role;
    auto record = [&](int r) -> int {
        hipEvent_t a, b;
        SPEO_TRY_HIP(hipEventCreate(&a));
        SPEO_TRY_HIP(hipEventCreate(&b));
        ev.push_back(a);
        ev.push_back(b);
        role.push_back(r);
        return SPEO_OK;
    };
    for (int g = 0; g < generations; ++g) {
        if (donor_buf) SPEO_TRY(draw_ahead(0, 1, stream));
        const int64_t gi = gens;
        const int modes[3] = {kModeGen, kModeEval, kModeSelect};
        if (cfg.mode == SPEO_MODE_FUSED) {
            SPEO_TRY(record(3));
            SPEO_TRY_HIP(hipEventRecord(ev[ev.size() - 2], stream));
            SPEO_TRY(launch(kModeFused, 0, rt, stream));
            SPEO_TRY_HIP(hipEventRecord(ev.back(), stream));
            p = 1 - p;
            pending = true;
        } else {
            for (int m = 0; m < 3; ++m) {
                SPEO_TRY(record(m));
                SPEO_TRY_HIP(hipEventRecord(ev[ev.size() - 2], stream));
                if (modes[m] == kModeGen && configured)
                    SPEO_TRY(generate_configured(0, stream));
                else
                    SPEO_TRY(launch(modes[m], 0, rt, stream));
                if (modes[m] == kModeEval) SPEO_TRY(eval_generic_islands(U[0], fU[0], stream));
                SPEO_TRY_HIP(hipEventRecord(ev.back(), stream));
            }
        }
        const bool point = cfg.interval > 0 && gi % cfg.interval == 0;
        const bool mig = point && cfg.migration_size > 0;
        if (mig) SPEO_TRY(migrate(stream));
        hipLaunchKernelGGL(k_add_u32, dim3(1), dim3(64), 0, stream, gen_base, 1u);
        SPEO_TRY(check_launch("k_add_u32"));
        ++gens;
        fes += total_rows;
        if (mig) ++migrations;
        if (point && configured) SPEO_TRY(regroup(false));
    }
    SPEO_TRY_HIP(hipStreamSynchronize(stream));
    double sum[roles] = {0, 0, 0, 0, 0, 0};
    int cnt[roles] = {0, 0, 0, 0, 0, 0};
    for (size_t i = 0; i < role.size(); ++i) {
        float ms = 0.f;
        SPEO_TRY_HIP(hipEventElapsedTime(&ms, ev[2 * i], ev[2 * i + 1]));
        sum[role[i]] += ms;
        cnt[role[i]] += 1;
    }
    for (auto e : ev) (void)hipEventDestroy(e);
    for (int r = 0; r < roles; ++r) avg_ms[r] = cnt[r] ? sum[r] / cnt[r] : 0.0;
    return SPEO_OK;
}

// Epoch mode: epochs on the run schedule, HIP events around every epoch
// launch; role 4 is the launch duration per generation.
int Engine::prof_begin(int role, int gens_covered, hipStream_t s) {
    if (!prof) return SPEO_OK;
    ProfEvent p{role, nullptr, nullptr, gens_covered};
    SPEO_TRY_HIP(hipEventCreate(&p.a));
    SPEO_TRY_HIP(hipEventCreate(&p.b));
    prof->push_back(p);
    SPEO_TRY_HIP(hipEventRecord(p.a, s));
    return SPEO_OK;
}

int Engine::prof_end(hipStream_t s) {
    if (!prof) return SPEO_OK;
    SPEO_TRY_HIP(hipEventRecord(prof->back().b, s));
    return SPEO_OK;
}

int Engine::profile_epoch(int generations, double *avg_ms) {
    for (int r = 0; r < 6; ++r) avg_ms[r] = 0.0;
    std::vector<ProfEvent> events;
    prof = &events;
    int64_t total_gens = 0;
    int left = generations, rc = SPEO_OK;
    while (left > 0 && rc == SPEO_OK) {
        bool mig = false;
        const int L = next_chunk(left, &mig);
        if ((rc = launch_epoch_chunk(L, stream)) != SPEO_OK) break;
        if (mig && (rc = migrate(stream)) != SPEO_OK) break;
        hipLaunchKernelGGL(k_add_u32, dim3(1), dim3(64), 0, stream, gen_base, (uint32_t)L);
        if ((rc = check_launch("k_add_u32")) != SPEO_OK) break;
        total_gens += L;
        gens += L;
        fes += (int64_t)L * total_rows;
        if (mig) ++migrations;
        left -= L;
    }
    prof = nullptr;
    if (rc == SPEO_OK) rc = check_hip(hipStreamSynchronize(stream), "hipStreamSynchronize");
    double sum[6] = {0, 0, 0, 0, 0, 0};
    for (const ProfEvent &p : events) {
        float ms = 0.f;
        if (rc == SPEO_OK) rc = check_hip(hipEventElapsedTime(&ms, p.a, p.b), "hipEventElapsedTime");
        sum[p.role] += ms;
        (void)hipEventDestroy(p.a);
        (void)hipEventDestroy(p.b);
    }
    if (total_gens > 0)
        for (int r = 4; r < 6; ++r) avg_ms[r] = sum[r] / (double)total_gens;
    return rc;
}

// Times the generation kernel with each row tile on scratch copies of the
// state and keeps the fastest.  Results are cached per configuration shape.
int Engine::autotune() {
    static std::mutex mu;
    static std::map<std::vector<int>, int> cache;
    // timed by the kernel that the engine's generations run
    const bool plain = runs_fused();
    const int mode = cfg.mode == SPEO_MODE_FUSED || by_launches || plain ? kModeFused : kModeEval;
    std::vector<int> key{cfg.precision, by_launches ? -1 : plain ? -2 : cfg.mode};
    for (const auto &d : isl) {
        key.push_back(d.np);
        key.push_back(d.dim);
    }
    {
        std::lock_guard<std::mutex> lk(mu);
        auto it = cache.find(key);
        if (it != cache.end()) {
            rt = it->second;
            return SPEO_OK;
        }
    }
    const std::string pkey = tune_key(by_launches ? "rt_launches" : plain ? "rt_plain" : "rt");
    int stored = 0;
    if (tune_lookup(pkey, &stored) && (stored == 16 || stored == 32 || stored == 64)) {
        rt = stored;
        tuned_from_cache |= 1;
        std::lock_guard<std::mutex> lk(mu);
        cache[key] = rt;
        return SPEO_OK;
    }
    float *saveX = X, *savefX[2] = {fX[0], fX[1]}, *saveU[2] = {U[0], U[1]},
          *savefU[2] = {fU[0], fU[1]};
    const size_t E = (size_t)total_elems, R = (size_t)total_rows;
    float *tX = nullptr, *tf[4] = {nullptr, nullptr, nullptr, nullptr}, *tU[2] = {nullptr, nullptr};
    SPEO_TRY_HIP(hipMalloc(&tX, sizeof(float) * E));
    SPEO_TRY_HIP(hipMalloc(&tU[0], sizeof(float) * E));
    SPEO_TRY_HIP(hipMalloc(&tU[1], sizeof(float) * E));
    for (auto &b : tf) SPEO_TRY_HIP(hipMalloc(&b, sizeof(float) * R));
    SPEO_TRY_HIP(hipMemcpyAsync(tX, saveX, sizeof(float) * E, hipMemcpyDeviceToDevice, stream));
    SPEO_TRY_HIP(hipMemsetAsync(tU[0], 0, sizeof(float) * E, stream));
    SPEO_TRY_HIP(hipMemsetAsync(tU[1], 0, sizeof(float) * E, stream));
    for (auto &b : tf) {
        hipLaunchKernelGGL(k_fill, dim3(256), dim3(256), 0, stream, b, total_rows, INFINITY);
        SPEO_TRY(check_launch("k_fill"));
    }
    X = tX;
    fX[0] = tf[0];
    fX[1] = tf[1];
    fU[0] = tf[2];
    fU[1] = tf[3];
    U[0] = tU[0];
    U[1] = tU[1];
    hipEvent_t e0, e1;
    SPEO_TRY_HIP(hipEventCreate(&e0));
    SPEO_TRY_HIP(hipEventCreate(&e1));
    float best_ms = 1e30f;
    int best_rt = 32;
    const int saved_p = p;
    const bool saved_pending = pending;
    pending = true;  // as all generations of a run but its first
    SPEO_TRY(build_tiles(kTrialRows));
    for (int cand : {16, 32, 64}) {
        SPEO_TRY(build_tiles(cand));
        if (donor_buf) SPEO_TRY(draw_ahead(0, std::min(6, donor_gens), stream));
        for (int rep = 0; rep < 2; ++rep) SPEO_TRY(launch(mode, rep, cand, stream));
        SPEO_TRY_HIP(hipEventRecord(e0, stream));
        const int reps = 6;
        for (int rep = 0; rep < reps; ++rep) {
            SPEO_TRY(launch(mode, rep, cand, stream));
            if (mode == kModeFused) p = 1 - p;
        }
        SPEO_TRY_HIP(hipEventRecord(e1, stream));
        SPEO_TRY_HIP(hipEventSynchronize(e1));
        float ms = 0.f;
        SPEO_TRY_HIP(hipEventElapsedTime(&ms, e0, e1));
        if (ms < best_ms) {
            best_ms = ms;
            best_rt = cand;
        }
    }
    p = saved_p;
    pending = saved_pending;
    (void)hipEventDestroy(e0);
    (void)hipEventDestroy(e1);
    X = saveX;
    fX[0] = savefX[0];
    fX[1] = savefX[1];
    U[0] = saveU[0];
    U[1] = saveU[1];
    fU[0] = savefU[0];
    fU[1] = savefU[1];
    (void)hipFree(tX);
    (void)hipFree(tU[0]);
    (void)hipFree(tU[1]);
    for (auto &b : tf) (void)hipFree(b);
    rt = best_rt;
    tune_store(pkey, rt);
    std::lock_guard<std::mutex> lk(mu);
    cache[key] = rt;
    return SPEO_OK;
}

std::string Engine::tune_key(const char *what) const {
    std::vector<std::pair<int, int>> dn;
    for (const auto &d : isl) {
        int b = 1;
        while (b < d.np) b <<= 1;
        dn.emplace_back(d.dim, b);
    }
    std::sort(dn.begin(), dn.end());
    std::ostringstream k;
    k << what << ":m" << cfg.mode << ":p" << cfg.precision << ":n" << I;
    for (size_t i = 0; i < dn.size();) {  // runs of equal (dim, bucket) as dim/bucket*count
        size_t j = i;
        while (j < dn.size() && dn[j] == dn[i]) ++j;
        k << ':' << dn[i].first << '/' << dn[i].second << '*' << (j - i);
        i = j;
    }
    return k.str();
}

// The key of a choice that was timed by whole runs: they have graphs or not, and
// their launches end at the migration points.
std::string Engine::plan_key(const char *what) const {
    return tune_key(what) + ":g" + (cfg.use_graph ? '1' : '0') + ":i" +
           std::to_string(cfg.migration_size > 0 ? cfg.interval : 0);
}

// Seconds a generation of a throwaway engine of this configuration, graphs or
// not as it has them: the median of three runs of whole intervals (16 generations
// where none are shorter), which are all of one launch sequence; the graphs that a
// run needs are captured before its clock starts, and the first, cold one counts
// no more than the others.
int Engine::time_plan(int parts, bool launches, double *seconds) {
    constexpr int kGens = 16;
    speo_engine_config c2 = cfg;
    c2.epoch_parts = parts;
    c2.rows_per_block = cfg.rows_per_block ? cfg.rows_per_block : 32;
    const bool migrates = cfg.interval > 0 && cfg.migration_size > 0;
    if (migrates) c2.interval = std::min(cfg.interval, kGens);
    const int gens_timed = migrates ? kGens / c2.interval * c2.interval : kGens;
    auto child = std::make_unique<Engine>();
    child->tuning_child = true;
    child->by_launches = launches;
    SPEO_TRY(child->create(c2, stream));
    if (migrates) SPEO_TRY(child->run(1));  // up to the first migration point
    double t[3];
    for (double &dt : t) {
        SPEO_TRY(child->prepare(gens_timed));
        SPEO_TRY_HIP(hipStreamSynchronize(stream));
        const auto t0 = std::chrono::steady_clock::now();
        SPEO_TRY(child->run(gens_timed));
        SPEO_TRY_HIP(hipStreamSynchronize(stream));
        dt = std::chrono::duration<double>(std::chrono::steady_clock::now() - t0).count();
    }
    std::sort(t, t + 3);
    *seconds = t[1] / gens_timed;
    return SPEO_OK;
}

// Whether the generations of an epoch engine with an automatic plan run as
// fused launches, which spread an island over as many workgroups as it has row
// tiles: measured against the plan chosen (the same results either way).  An
// epoch kernel's time grows with the rows of its largest island and, beyond two
// islands a compute unit, in rounds; the launches' with all rows.  Us a generation,
// epoch plan against launches of 32 rows: 16 x 512, D = 100: 85 / 14; 100 x 400,
// D = 128: 79 / 38; 1024 x 64, D = 30: 27 / 17; 64 x 128, D = 100: 9.5 / 14.  Up
// to 64 rows and two islands a unit the epoch kernel always was the faster one
// or within 20 %, and nothing is measured.
int Engine::tune_launches() {
    static std::mutex mu;
    static std::map<std::string, int> chosen;  // bounded by the workload shapes a program uses
    int dev = 0, cus = 0;
    SPEO_TRY_HIP(hipGetDevice(&dev));
    SPEO_TRY_HIP(hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev));
    if (max_np <= 64 && I <= 2 * cus) return SPEO_OK;
    std::vector<EpochPlan> plans;
    int lds = 0;
    if (epoch_plan_all(cfg.epoch_parts, &plans, &lds) != SPEO_OK) return SPEO_OK;  // epoch_setup reports it
    const std::string key = plan_key(("launches" + std::to_string(cfg.epoch_parts)).c_str());
    int stored = 0;
    const bool on_file = tune_lookup(key, &stored) && (stored == 0 || stored == 1);
    bool known = on_file;
    if (!known) {
        std::lock_guard<std::mutex> lk(mu);
        auto it = chosen.find(key);
        known = it != chosen.end();
        if (known) stored = it->second;
    }
    if (!known) {
        double plan = 0.0, launches = 0.0;
        if (time_plan(cfg.epoch_parts, false, &plan) != SPEO_OK ||
            time_plan(cfg.epoch_parts, true, &launches) != SPEO_OK) {
            // no room beside this engine, say: it runs as planned, unmeasured
            (void)hipGetLastError();
            return SPEO_OK;
        }
        stored = launches < plan ? 1 : 0;
    }
    if (!on_file) tune_store(key, stored);  // (also a choice measured while another file was in use)
    by_launches = stored != 0;
    std::lock_guard<std::mutex> lk(mu);
    chosen[key] = stored;
    return SPEO_OK;
}

// Workgroups per island for epoch mode: every feasible power of two up to 8
// (islands x parts at most four per compute unit) timed on a throwaway
// engine of this configuration; the fastest is kept and persisted.
int Engine::tune_epoch_parts() {
    const std::string key = plan_key("epoch_parts");
    int stored = 0;
    if (tune_lookup(key, &stored) && (stored == 1 || stored == 2 || stored == 4 || stored == 8)) {
        cfg.epoch_parts = stored;
        tuned_from_cache |= 2;
        return SPEO_OK;
    }
    int dev = 0, cus = 0;
    SPEO_TRY_HIP(hipGetDevice(&dev));
    SPEO_TRY_HIP(hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev));
    std::vector<int> cands;
    for (int parts = 1; parts <= kEpochMaxParts; parts *= 2) {
        std::vector<EpochPlan> plans;
        int lds = 0;
        if ((int64_t)I * parts > 4 * (int64_t)cus) break;
        if (epoch_plan_all(parts, &plans, &lds) == SPEO_OK) cands.push_back(parts);
    }
    if (cands.empty()) return SPEO_OK;  // epoch_setup reports the reason
    int best = cands[0];
    if (cands.size() > 1) {
        double best_s = 1e30;
        for (int parts : cands) {
            double dt = 0.0;
            SPEO_TRY(time_plan(parts, false, &dt));
            if (dt < best_s) {
                best_s = dt;
                best = parts;
            }
        }
    }
    cfg.epoch_parts = best;
    tune_store(key, best);
    return SPEO_OK;
}

int Engine::best(int *row_out, float *f32_out, double *f64_out) {
    SPEO_TRY(finalize_pending(stream));
    const int cur = cfg.mode == SPEO_MODE_FUSED ? p : 0;
    const int chunks = (max_dim + kBestCols - 1) / kBestCols;
    BestArgs a{isl_dev, probs_dev, params_tab_dev, X, fX[cur], best_row_dev, best_out_dev, best_part, chunks};
    int nc = 1;
    for (const auto *q : problems) nc = std::max(nc, q->h.ncomp);
    SPEO_TRY(best_rows(a, I, nc, max_dim, stream));
    for (int i = 0; i < I && any_generic; ++i) {  // generic problems: the FP64 generic kernel
        const IslandDesc &d = isl[(size_t)i];
        const ProblemHost &P = problems[(size_t)d.problem]->h;
        if (P.generic)
            SPEO_TRY(eval_problem_generic(P, X + d.elem_off, d.ld, 1, nullptr, &best_out_dev[i].f64,
                                          best_row_dev + i, d.row_off, stream));
    }
    SPEO_TRY_HIP(hipStreamSynchronize(stream));
    for (int i = 0; i < I; ++i) {
        if (row_out) row_out[i] = best_out[i].row;
        if (f32_out) f32_out[i] = best_out[i].f32;
        if (f64_out) f64_out[i] = best_out[i].f64;
    }
    return SPEO_OK;
}

int Engine::read(float *Xo, float *fo) {
    SPEO_TRY(finalize_pending(stream));
    const int cur = cfg.mode == SPEO_MODE_FUSED ? p : 0;
    return read_rows(X, fX[cur], Xo, fo);
}

int Engine::read_rows(const float *src, const float *fsrc, float *Xo, float *fo) {
    if (Xo) {
        std::vector<float> h((size_t)total_elems);
        SPEO_TRY_HIP(hipMemcpyAsync(h.data(), src, sizeof(float) * h.size(), hipMemcpyDeviceToHost, stream));
        SPEO_TRY_HIP(hipStreamSynchronize(stream));
        for (const auto &d : isl)
            for (int r = 0; r < d.np; ++r)
                for (int j = 0; j < max_dim; ++j)
                    Xo[(size_t)(d.row_off + r) * max_dim + j] =
                        j < d.dim ? h[(size_t)d.elem_off + (size_t)r * d.ld + j] : 0.f;
    }
    if (fo) {
        SPEO_TRY_HIP(hipMemcpyAsync(fo, fsrc, sizeof(float) * total_rows, hipMemcpyDeviceToHost, stream));
        SPEO_TRY_HIP(hipStreamSynchronize(stream));
    }
    return SPEO_OK;
}

int Engine::write(const float *Xi, const float *fi) {
    SPEO_TRY(finalize_pending(stream));
    const int cur = cfg.mode == SPEO_MODE_FUSED ? p : 0;
    if (Xi) {
        std::vector<float> h((size_t)total_elems, 0.f);
        for (const auto &d : isl)
            for (int r = 0; r < d.np; ++r)
                for (int j = 0; j < d.dim; ++j)
                    h[(size_t)d.elem_off + (size_t)r * d.ld + j] = Xi[(size_t)(d.row_off + r) * max_dim + j];
        SPEO_TRY_HIP(hipMemcpyAsync(X, h.data(), sizeof(float) * h.size(), hipMemcpyHostToDevice, stream));
        SPEO_TRY_HIP(hipStreamSynchronize(stream));
    }
    if (fi) {
        SPEO_TRY_HIP(hipMemcpyAsync(fX[cur], fi, sizeof(float) * total_rows, hipMemcpyHostToDevice, stream));
        SPEO_TRY_HIP(hipStreamSynchronize(stream));
    }
    return SPEO_OK;
}

}  // namespace speo

struct speo_engine_s {
    speo::Engine e;
};

using namespace speo;

extern "C" {

int speo_engine_create(const speo_engine_config *cfg, speo_stream_t stream, speo_engine *out) {
    if (!cfg || !out) return set_error(SPEO_ERR_ARG, "speo_engine_create: null argument");
    *out = nullptr;
    auto *h = new (std::nothrow) speo_engine_s;
    if (!h) return set_error(SPEO_ERR_ALLOC, "speo_engine_create: out of host memory");
    const int rc = h->e.create(*cfg, as_stream(stream));
    if (rc != SPEO_OK) {
        const std::string msg = speo_last_error();
        delete h;
        return set_error(rc, msg);
    }
    *out = h;
    return SPEO_OK;
}

int speo_engine_destroy(speo_engine e) {
    delete e;
    return SPEO_OK;
}

int speo_engine_run(speo_engine e, int generations) {
    if (!e || generations < 0) return set_error(SPEO_ERR_ARG, "speo_engine_run: bad arguments");
    return e->e.run(generations);
}

// IslandEA::Execute's budget loop (src/island_EA.cc:86-104) over the engine's
// evaluation count; speo_engine_run splits the generations at the migration
// points as the reference migrates at generation % interval == 0.
int speo_engine_run_fes(speo_engine e, int64_t max_FEs, int *generations_out) {
    if (!e) return set_error(SPEO_ERR_ARG, "speo_engine_run_fes: null engine");
    const int64_t g = speo_generations_for_fes(max_FEs, e->e.fes, e->e.total_rows);
    if (g > 0x7fffffff) return set_error(SPEO_ERR_ARG, "speo_engine_run_fes: budget beyond 2^31 generations");
    if (generations_out) *generations_out = (int)g;
    return e->e.run((int)g);
}

int speo_engine_run_fes_timed(speo_engine e, int64_t max_FEs, int *generations_out,
                              double *seconds_out, double *comm_seconds_out) {
    if (!e) return set_error(SPEO_ERR_ARG, "speo_engine_run_fes_timed: null engine");
    Engine &E = e->e;
    const int64_t g = speo_generations_for_fes(max_FEs, E.fes, E.total_rows);
    if (g > 0x7fffffff) return set_error(SPEO_ERR_ARG, "speo_engine_run_fes_timed: budget beyond 2^31 generations");
    if (generations_out) *generations_out = (int)g;
    SPEO_TRY_HIP(hipStreamSynchronize(E.stream));
    E.time_comm = true;
    E.comm_seconds = 0.0;
    const auto t0 = std::chrono::steady_clock::now();
    int rc = E.run((int)g);
    if (rc == SPEO_OK) rc = check_hip(hipStreamSynchronize(E.stream), "speo_engine_run_fes_timed");
    const double dt = std::chrono::duration<double>(std::chrono::steady_clock::now() - t0).count();
    E.time_comm = false;
    if (seconds_out) *seconds_out = dt;
    if (comm_seconds_out) *comm_seconds_out = E.comm_seconds;
    return rc;
}

int speo_engine_subislands(speo_engine e, int island, int *subisland_num_out, int *perm_out,
                           DEInfo *info_out) {
    if (!e) return set_error(SPEO_ERR_ARG, "speo_engine_subislands: null engine");
    return e->e.subislands(island, subisland_num_out, perm_out, info_out);
}

int speo_engine_prepare(speo_engine e, int generations) {
    if (!e || generations < 0) return set_error(SPEO_ERR_ARG, "speo_engine_prepare: bad arguments");
    return e->e.prepare(generations);
}

int speo_engine_sync(speo_engine e) {
    if (!e) return set_error(SPEO_ERR_ARG, "speo_engine_sync: null engine");
    return check_hip(hipStreamSynchronize(e->e.stream), "speo_engine_sync");
}

int speo_engine_best(speo_engine e, int *row_out, float *f32_out, double *f64_out) {
    if (!e) return set_error(SPEO_ERR_ARG, "speo_engine_best: null engine");
    return e->e.best(row_out, f32_out, f64_out);
}

int speo_engine_read(speo_engine e, float *X_out, float *f_out) {
    if (!e) return set_error(SPEO_ERR_ARG, "speo_engine_read: null engine");
    return e->e.read(X_out, f_out);
}

int speo_engine_read_trials(speo_engine e, float *U_out, float *fU_out) {
    if (!e) return set_error(SPEO_ERR_ARG, "speo_engine_read_trials: null engine");
    const int cur = e->e.cfg.mode == SPEO_MODE_FUSED ? e->e.p : 0;
    return e->e.read_rows(e->e.U[cur], e->e.fU[cur], U_out, fU_out);
}

int speo_engine_write(speo_engine e, const float *X_in, const float *f_in) {
    if (!e) return set_error(SPEO_ERR_ARG, "speo_engine_write: null engine");
    return e->e.write(X_in, f_in);
}

int speo_engine_get_stats(speo_engine e, speo_engine_stats *out) {
    if (!e || !out) return set_error(SPEO_ERR_ARG, "speo_engine_get_stats: null argument");
    out->generations = e->e.gens;
    out->evaluations = e->e.fes;
    out->migrations = e->e.migrations;
    out->graph_launches = e->e.graph_launches;
    out->rows_per_block = e->e.rt;
    out->surrogate_predictions = e->e.surr_pred;
    if (e->e.scored_dev) {
        // the one-kernel screening's count lives on the device
        const size_t P = (size_t)e->e.cfg.num_problems;
        std::vector<long long> scored(P, 0);
        SPEO_TRY_HIP(hipStreamSynchronize(e->e.stream));
        SPEO_TRY_HIP(hipMemcpy(scored.data(), e->e.scored_dev, sizeof(long long) * P, hipMemcpyDeviceToHost));
        for (long long v : scored) out->surrogate_predictions += v;
    }
    out->surrogate_rounds = e->e.surr_rounds;
    out->epoch_parts = e->e.cfg.mode == SPEO_MODE_EPOCH ? e->e.epoch_parts : 0;
    return SPEO_OK;
}

int speo_engine_surrogate_stats(speo_engine e, float *rho_out, int *active_out, float *loss_out) {
    if (!e) return set_error(SPEO_ERR_ARG, "speo_engine_surrogate_stats: null engine");
    Engine &E = e->e;
    const int P = E.cfg.num_problems;
    std::vector<float> rho((size_t)P, -1.f), loss((size_t)P, 0.f);
    if (E.C > 0) {
        SPEO_TRY_HIP(hipStreamSynchronize(E.stream));
        SPEO_TRY_HIP(hipMemcpy(rho.data(), E.rho_dev, sizeof(float) * P, hipMemcpyDeviceToHost));
        for (int p = 0; p < P; ++p)
            if (E.surr[(size_t)p]->rows > 0 && E.surr[(size_t)p]->trained)
                SPEO_TRY_HIP(hipMemcpy(&loss[(size_t)p], E.surr[(size_t)p]->net.stats, sizeof(float),
                                       hipMemcpyDeviceToHost));
    }
    for (int p = 0; p < P; ++p) {
        if (rho_out) rho_out[p] = rho[(size_t)p];
        if (active_out)
            active_out[p] = (E.C > 0 && E.surr[(size_t)p]->trained && rho[(size_t)p] >= E.cfg.surrogate_rho_min) ? 1 : 0;
        if (loss_out) loss_out[p] = loss[(size_t)p];
    }
    return SPEO_OK;
}

int speo_engine_surrogate_dump(speo_engine e, int problem, int *cands_out, float *cand_out,
                               float *pred_out, float *archive_X, float *archive_y, int *head_out,
                               int64_t *appended_out) {
    if (!e || e->e.C <= 0 || problem < 0 || problem >= e->e.cfg.num_problems)
        return set_error(SPEO_ERR_ARG, "speo_engine_surrogate_dump: no surrogate or bad problem");
    Engine &E = e->e;
    const auto &sp = *E.surr[(size_t)problem];
    const size_t Kp = (size_t)E.Kp, Ce = (size_t)E.last_Ce, cap = (size_t)E.cfg.surrogate_archive;
    SPEO_TRY_HIP(hipStreamSynchronize(E.stream));
    if (cands_out) *cands_out = E.last_Ce;
    if (cand_out)
        SPEO_TRY_HIP(hipMemcpy(cand_out, E.cand + (size_t)sp.qoff * Ce * Kp,
                               sizeof(float) * (size_t)sp.rows * Ce * Kp, hipMemcpyDeviceToHost));
    if (pred_out)
        SPEO_TRY_HIP(hipMemcpy(pred_out, E.pred + (size_t)sp.qoff * Ce, sizeof(float) * (size_t)sp.rows * Ce,
                               hipMemcpyDeviceToHost));
    if (archive_X)
        SPEO_TRY_HIP(hipMemcpy(archive_X, E.AX + (size_t)problem * cap * Kp, sizeof(float) * cap * Kp,
                               hipMemcpyDeviceToHost));
    if (archive_y)
        SPEO_TRY_HIP(hipMemcpy(archive_y, E.Ay + (size_t)problem * cap, sizeof(float) * cap,
                               hipMemcpyDeviceToHost));
    if (head_out) *head_out = sp.head;
    if (appended_out) *appended_out = sp.appended;
    E.retain_cand = true;  // later generations keep their candidates for the next dump
    return SPEO_OK;
}

int speo_engine_surrogate_set_labels(speo_engine e, int problem, const float *archive_y) {
    if (!e || e->e.C <= 0 || problem < 0 || problem >= e->e.cfg.num_problems || !archive_y)
        return set_error(SPEO_ERR_ARG, "speo_engine_surrogate_set_labels: no surrogate or bad arguments");
    Engine &E = e->e;
    const size_t cap = (size_t)E.cfg.surrogate_archive;
    SPEO_TRY_HIP(hipStreamSynchronize(E.stream));
    SPEO_TRY_HIP(hipMemcpy(E.Ay + (size_t)problem * cap, archive_y, sizeof(float) * cap,
                           hipMemcpyHostToDevice));
    return SPEO_OK;
}

int speo_engine_profile(speo_engine e, int generations, double *avg_ms_out) {
    if (!e || generations < 1 || !avg_ms_out)
        return set_error(SPEO_ERR_ARG, "speo_engine_profile: bad arguments");
    return e->e.profile(generations, avg_ms_out);
}

int speo_engine_total_rows(speo_engine e) { return e ? e->e.total_rows : 0; }
int speo_engine_max_dim(speo_engine e) { return e ? e->e.max_dim : 0; }

int speo_engine_buffers(speo_engine e, float **X, float **fX, int64_t *elem_off, int *row_off,
                        int *ld) {
    if (!e) return set_error(SPEO_ERR_ARG, "speo_engine_buffers: null engine");
    if (X) *X = e->e.X;
    if (fX) *fX = e->e.fX[e->e.cfg.mode == SPEO_MODE_FUSED ? e->e.p : 0];
    for (int i = 0; i < e->e.I; ++i) {
        if (elem_off) elem_off[i] = e->e.isl[(size_t)i].elem_off;
        if (row_off) row_off[i] = e->e.isl[(size_t)i].row_off;
        if (ld) ld[i] = e->e.isl[(size_t)i].ld;
    }
    return SPEO_OK;
}

}  // extern "C"

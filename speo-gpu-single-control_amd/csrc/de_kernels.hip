// de_kernels.hip -- DE operator kernels and the drop-in DE entry points.
//
// Operator math follows the reference GPU kernels exactly (bit for bit, given
// the same uniforms):
//   donor draw with redraw quirks        kernel_DE_CUDA.cu:183-216
//   j_rand without "== dim" guard        kernel_DE_CUDA.cu:218-222
//   crossover test j == j_rand || u < CR kernel_DE_CUDA.cu:229-241
//   strategies 0-8                       kernel_DE_CUDA.cu:243-282
//   reflective bound                     kernel_DE_CUDA.cu:160-170
//   strict "<" selection                 kernel_DE_CUDA.cu:305-327
//   uniform init                         kernel_EA_CUDA.cu:91-118
// F*(a-b) terms are fused into the running sum with fmaf (nvcc's contraction
// of the reference expression); nothing else may contract.
#pragma clang fp contract(off)

#include "de.h"

namespace speo {

// ------------------------------------------------------------------ init

__global__ void k_init_population(float *X, int ld, int n, int dim, float lo, float hi,
                                  uint64_t seed, uint32_t row_base) {
    const int groups = ld >> 2;
    const int64_t total = (int64_t)n * groups;
    const float span = hi - lo;
    for (int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; t < total;
         t += (int64_t)gridDim.x * blockDim.x) {
        const int row = (int)(t / groups), g = (int)(t % groups);
        const U4 w = philox_block(seed, (uint32_t)g, row_base + (uint32_t)row, 0u, kPurposeInit);
        const int j0 = g * 4;
        float4 v;
        v.x = j0 + 0 < dim ? fmaf(u01(w.x), span, lo) : 0.f;
        v.y = j0 + 1 < dim ? fmaf(u01(w.y), span, lo) : 0.f;
        v.z = j0 + 2 < dim ? fmaf(u01(w.z), span, lo) : 0.f;
        v.w = j0 + 3 < dim ? fmaf(u01(w.w), span, lo) : 0.f;
        *reinterpret_cast<float4 *>(X + (size_t)row * ld + j0) = v;
    }
}

int init_population(float *X, int ld, int n, int dim, float lo, float hi, uint64_t seed,
                    uint32_t row_base, hipStream_t s) {
    if (n <= 0) return SPEO_OK;
    const int64_t total = (int64_t)n * (ld >> 2);
    const int blocks = (int)std::min<int64_t>((total + 255) / 256, 4096);
    hipLaunchKernelGGL(k_init_population, dim3(blocks), dim3(256), 0, s, X, ld, n, dim, lo, hi,
                       seed, row_base);
    return check_launch("k_init_population");
}

// -------------------------------------------------------------- generate

// Four consecutive coordinates of a row; those past the dimension are 0.
struct Four {
    float v[4];
};

// The mutant's coordinates (row(i): those of population row i).
template <typename Row>
__device__ __forceinline__ Four mutant(int st, float F, int sel, int r0, int r1, int r2, int r3, int r4, int best,
                                       Row row) {
    auto add = [F](Four x, const Four &a, const Four &b) {
#pragma unroll
        for (int q = 0; q < 4; ++q) x.v[q] = fmaf(F, a.v[q] - b.v[q], x.v[q]);
        return x;
    };
    switch (st) {
    case 0: return add(row(sel), row(r0), row(r1));
    case 1: return add(add(row(sel), row(r0), row(r1)), row(r2), row(r3));
    case 2: {
        const Four s = row(sel);
        return add(add(s, row(best), s), row(r0), row(r1));
    }
    case 3: {
        const Four s = row(sel), b = row(r1);
        return add(add(add(s, row(best), s), row(r0), b), b, row(r2));
    }
    case 4: return add(row(r0), row(r1), row(r2));
    case 5: return add(add(row(r0), row(r1), row(r2)), row(r3), row(r4));
    case 6: return add(row(best), row(r0), row(r1));
    case 7: return add(add(row(best), row(r0), row(r1)), row(r2), row(r3));
    case 8: {
        const Four s = row(sel);
        return add(add(s, row(r0), s), row(r1), row(r2));
    }
    default: return row(sel);
    }
}
__device__ __forceinline__ bool uses_best(int st) { return st == 2 || st == 3 || st == 6 || st == 7; }

// LPR lanes per row, four coordinates each.  The call is bound by latency at
// the drop-in sizes (donor draws, indices, rows, crossover draws, one after
// another), so up to kWaveRows rows take a wave each: its draws diverge over no
// other row and its rows' addresses are scalars.  Beyond, 16 lanes a row repeat
// the draws least (D = 100, rand/1, a wave / 16 lanes a row: 1,024 rows 5.0 / 6.1
// us, 2,048 6.9 / 6.2, 4,096 11.5 / 8.7).
// a.fit: the sub-islands' best members are found here too, by blocks past the
// rows' for the caller and, where the strategy reads it, by the rows' own blocks
// (S a multiple of a block's rows): 4 to 5 us less than a launch of its own.  The
// rows' searches are row blocks x S reads; up to kBestReads of them such a strategy
// costs within 2 us of the two launches up to 16,384 rows (best/1, here / apart:
// 8,192 as 1 island 20.5 / 20.9 us, 16,384 as 4 22.5 / 21.2) and the others gain;
// at twice that (65,536 as 32: 55.6 / 32.6) it is slower than ever.
// 1,024 rows, D = 100: best 5.1 us and generate 10.7 us as two launches of 16
// lanes a row and scalar loads, 5.0 us now.
constexpr int kWaveRows = 1024;
constexpr int64_t kBestReads = 1 << 22;

template <bool INJ, int LPR>
__global__ __launch_bounds__(256) void k_de_generate(GenArgs a) {
    constexpr int RB = 256 / LPR;
    __shared__ float sf[4];
    __shared__ int si[4], sbest;
    const int tid = threadIdx.x, l = tid & (LPR - 1);
    const int sub = LPR == 64 ? __builtin_amdgcn_readfirstlane(tid >> 6) : tid / LPR;
    const int rowblocks = (a.n + RB - 1) / RB;
    int found = -1;
    if (a.fit) {
        const bool extra = (int)blockIdx.x >= rowblocks;
        const int isl = extra ? (int)blockIdx.x - rowblocks : (int)blockIdx.x * RB / a.S;
        if (extra || uses_best(a.de_info[isl].strategy_ID)) {
            const int b = block_argmin(a.fit, a.perm, isl * a.S, a.S, sf, si);
            if (tid == 0) {
                sbest = b;
                if (extra) a.best_out[isl] = b;
            }
            if (extra) return;
            __syncthreads();
            found = sbest;
        }
    }
    const int i = blockIdx.x * RB + sub;
    if (i >= a.n) return;
    const uint32_t row = a.row_base + (uint32_t)i;

    DonorStream ds(a.seed, row, a.gen);
    const float *inj = nullptr;
    if (INJ && a.inj_r) inj = a.inj_r + (size_t)i * a.n_inj;
    int r[kMaxR];
    int jr;
    draw_donors(ds, inj, INJ ? a.n_inj : 0, a.S, a.dim, r, jr);

    const int isl = i / a.S;
    const int sel = a.perm ? a.perm[i] : i;
    auto member = [&](int k) { return a.perm ? a.perm[k + isl * a.S] : k + isl * a.S; };
    const int r0 = member(r[0]), r1 = member(r[1]), r2 = member(r[2]), r3 = member(r[3]), r4 = member(r[4]);
    if (l == 0) {
        if (a.r_out) {
            int *out = a.r_out + (size_t)i * kMaxR;
            out[0] = r0;
            out[1] = r1;
            out[2] = r2;
            out[3] = r3;
            out[4] = r4;
        }
        if (a.jrand_out) a.jrand_out[i] = jr;
    }
    const DEInfo info = a.de_info[isl];
    const int b = a.fit ? found : a.best ? a.best[isl] : sel;
    const int ngroups = (a.dim + 3) >> 2;
    // 16-byte loads where the rows allow them (a group's last columns may be padding)
    const bool vec = (a.ld & 3) == 0 && ((reinterpret_cast<uintptr_t>(a.X) | reinterpret_cast<uintptr_t>(a.U)) & 15) == 0;
    for (int g = l; g < ngroups; g += LPR) {
        auto at = [&](int i_) {
            const float *p = a.X + (size_t)i_ * a.ld + 4 * g;
            Four x;
            if (vec) {
                const float4 v = *reinterpret_cast<const float4 *>(p);
                x = Four{{v.x, v.y, v.z, v.w}};
            } else {
#pragma unroll
                for (int q = 0; q < 4; ++q) x.v[q] = 4 * g + q < a.dim ? p[q] : 0.f;
            }
            return x;
        };
        const Four own = at(sel);
        const Four mut = mutant(info.strategy_ID, info.F, sel, r0, r1, r2, r3, r4, b, at);
        const U4 w = philox_block(a.seed, (uint32_t)g, row, a.gen, kPurposeCross);
        Four out;
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const int j = g * 4 + q;
            float u = u01(word(w, q));
            if (INJ && a.inj_cr && j < a.dim) u = a.inj_cr[(size_t)i * a.dim + j];
            const float v = (j == jr) || (u < info.CR) ? mut.v[q] : own.v[q];
            out.v[q] = j < a.dim ? check_bound(v, a.lo, a.hi) : 0.f;
        }
        float *p = a.U + (size_t)sel * a.ld + 4 * g;
        if (vec && 4 * g + 4 <= a.dim) {
            *reinterpret_cast<float4 *>(p) = float4{out.v[0], out.v[1], out.v[2], out.v[3]};
        } else {
#pragma unroll
            for (int q = 0; q < 4; ++q)
                if (4 * g + q < a.dim) p[q] = out.v[q];
        }
    }
}

template <bool INJ, int LPR>
static int launch_generate(GenArgs a, hipStream_t s) {
    constexpr int RB = 256 / LPR;
    int blocks = (a.n + RB - 1) / RB;
    if (a.fit) {
        if (a.S % RB == 0 && (int64_t)blocks * a.S <= kBestReads) {
            blocks += a.n / a.S;
        } else {
            SPEO_TRY(subisland_best(a.fit, a.perm, a.S, a.n / a.S, a.best_out, s));
            a.best = a.best_out;
            a.fit = nullptr;
        }
    }
    hipLaunchKernelGGL((k_de_generate<INJ, LPR>), dim3(blocks), dim3(256), 0, s, a);
    return check_launch("k_de_generate");
}

int de_generate(const GenArgs &a, hipStream_t s) {
    if (a.n <= 0) return SPEO_OK;
    const bool inj = a.inj_r || a.inj_cr;
    // (sub-islands that only the smaller blocks divide keep them to 4,096 rows: 1,024 a
    // sub-island 8.4 us, 10.5 with the search apart)
    const bool wave = a.n <= kWaveRows || (a.fit && a.n <= 4 * kWaveRows && a.S % 16 && a.S % 4 == 0);
    if (wave) return inj ? launch_generate<true, 64>(a, s) : launch_generate<false, 64>(a, s);
    return inj ? launch_generate<true, 16>(a, s) : launch_generate<false, 16>(a, s);
}

// ---------------------------------------------------------------- select

// 32 lanes per row, 16-byte copies where the rows allow them.
__global__ __launch_bounds__(256) void k_de_select(float *X, float *fX, const float *U, float *fU, int ld, int n,
                                                   int dim, uint8_t *accept_out, int clear_trials) {
    const int tid = threadIdx.x;
    const int i = blockIdx.x * 8 + (tid >> 5);
    const int l = tid & 31;
    if (i >= n) return;
    const float fu = fU[i], fx = fX[i];
    const bool acc = fu < fx;
    if (acc) {
        float *x = X + (size_t)i * ld;
        const float *u = U + (size_t)i * ld;
        const bool vec = (ld & 3) == 0 && ((reinterpret_cast<uintptr_t>(X) | reinterpret_cast<uintptr_t>(U)) & 15) == 0;
        const int ng = vec ? dim >> 2 : 0;
        for (int g = l; g < ng; g += 32)
            reinterpret_cast<float4 *>(x)[g] = reinterpret_cast<const float4 *>(u)[g];
        for (int j = 4 * ng + l; j < dim; j += 32) x[j] = u[j];
    }
    if (l == 0) {
        if (acc) fX[i] = fu;
        if (accept_out) accept_out[i] = acc ? 1 : 0;
        if (clear_trials) fU[i] = INFINITY;
    }
}

int de_select(float *X, float *fX, const float *U, float *fU, int ld, int n, int dim,
              uint8_t *accept_out, int clear_trials, hipStream_t s) {
    if (n <= 0) return SPEO_OK;
    hipLaunchKernelGGL(k_de_select, dim3((n + 7) / 8), dim3(256), 0, s, X, fX, U, fU, ld, n,
                       dim, accept_out, clear_trials);
    return check_launch("k_de_select");
}

// ---------------------------------------------------------------- argmin

__global__ void k_segment_argmin(const float *f, const int *off, int *best_out) {
    __shared__ float sf[4];
    __shared__ int si[4];
    const int s = blockIdx.x;
    const int b = block_argmin(f, nullptr, off[s], off[s + 1] - off[s], sf, si);
    if (threadIdx.x == 0) best_out[s] = b;
}

__global__ void k_subisland_best(const float *f, const int *perm, int S, int *best_out) {
    __shared__ float sf[4];
    __shared__ int si[4];
    const int b = block_argmin(f, perm, blockIdx.x * S, S, sf, si);
    if (threadIdx.x == 0) best_out[blockIdx.x] = b;
}

int subisland_best(const float *f, const int *perm, int S, int subs, int *best_out, hipStream_t s) {
    if (subs <= 0) return SPEO_OK;
    hipLaunchKernelGGL(k_subisland_best, dim3(subs), dim3(256), 0, s, f, perm, S, best_out);
    return check_launch("k_subisland_best");
}

int segment_argmin(const float *f, const int *off, int nseg, int *best_out, hipStream_t s) {
    if (nseg <= 0) return SPEO_OK;
    hipLaunchKernelGGL(k_segment_argmin, dim3(nseg), dim3(256), 0, s, f, off, best_out);
    return check_launch("k_segment_argmin");
}

// ------------------------------------------------------------- migration

// The rank of each row of an island in the order (f ascending, row ascending,
// NaN last); the first k rows are its best, the last k its worst.  Block b of
// an island's `parts` ranks rows 64 b .. 64 b + 63 with four lanes a row, each against
// every fourth row of the island, whose keys pass through LDS kRankLds at a
// time.  np compares a row, so an island's work is np^2: spread over np / 64
// blocks and four lanes it takes 14 us for 8 islands of 2,048 rows
// (595 us with a block an island) and 8 us for 256 of 50 to 512 (40 us).
constexpr int kRankLds = 4096, kRankRows = 64;

// A value's place in the order as an unsigned integer (-0 as 0).
__device__ __forceinline__ uint32_t rank_key(float f) {
    if (f != f) return 0xffffffffu;
    const uint32_t b = __float_as_uint(f == 0.f ? 0.f : f);
    return (b >> 31) ? ~b : (b | 0x80000000u);
}

__global__ __launch_bounds__(256) void k_rank_islands(const float *f, const int *row_off, int parts, int k,
                                                      int *best_out, int *worst_out) {
    __shared__ uint32_t keys[kRankLds];
    const int isl = blockIdx.x / parts, b = blockIdx.x % parts;
    const int r0 = row_off[isl], np = row_off[isl + 1] - r0;
    if (b * kRankRows >= np) return;
    const int r = b * kRankRows + (threadIdx.x >> 2), part = threadIdx.x & 3;
    const uint32_t mine = r < np ? rank_key(f[r0 + r]) : 0u;
    const uint64_t me = ((uint64_t)mine << 32) | (uint32_t)r;
    int rank = 0;
    for (int q0 = 0; q0 < np; q0 += kRankLds) {
        const int m = min(kRankLds, np - q0);
        __syncthreads();
        for (int q = threadIdx.x; q < m; q += 256) keys[q] = rank_key(f[r0 + q0 + q]);
        __syncthreads();
#pragma unroll 8
        for (int q = part; q < m; q += 4)
            rank += (((uint64_t)keys[q] << 32) | (uint32_t)(q0 + q)) < me ? 1 : 0;
    }
    rank += __shfl_xor(rank, 1, 64);
    rank += __shfl_xor(rank, 2, 64);
    if (part == 0 && r < np) {
        if (rank < k) best_out[isl * k + rank] = r0 + r;
        if (rank >= np - k) worst_out[isl * k + (np - 1 - rank)] = r0 + r;
    }
}

// Block per (island, migrant): island isl's t-th best row replaces the t-th
// worst row of island dst[isl].
__global__ void k_migrate_apply(float *X, float *fX, const IslandDesc *isl_desc, const int *dst,
                                const int *best, const int *worst, int k) {
    const int isl = blockIdx.x / k, t = blockIdx.x % k;
    const int d = dst[isl];
    if (d < 0) return;
    const IslandDesc S = isl_desc[isl], T = isl_desc[d];
    const int sr = best[isl * k + t] - S.row_off, tr = worst[d * k + t] - T.row_off;
    const float *src = X + S.elem_off + (size_t)sr * S.ld;
    float *out = X + T.elem_off + (size_t)tr * T.ld;
    for (int j = threadIdx.x; j < S.dim; j += blockDim.x) out[j] = src[j];
    if (threadIdx.x == 0) fX[T.row_off + tr] = fX[S.row_off + sr];
}

int migrate_ring(float *X, float *fX, const IslandDesc *isl_desc_dev, const int *row_off_dev,
                 const int *dst_dev, int *best_buf, int *worst_buf, int I, int max_np, int k,
                 hipStream_t s) {
    if (I <= 0 || k <= 0) return SPEO_OK;
    const int parts = (max_np + kRankRows - 1) / kRankRows;
    hipLaunchKernelGGL(k_rank_islands, dim3((unsigned)I * parts), dim3(256), 0, s, fX, row_off_dev, parts, k,
                       best_buf, worst_buf);
    SPEO_TRY(check_launch("k_rank_islands"));
    hipLaunchKernelGGL(k_migrate_apply, dim3(I * k), dim3(128), 0, s, X, fX, isl_desc_dev, dst_dev,
                       best_buf, worst_buf, k);
    return check_launch("k_migrate_apply");
}

}  // namespace speo

// ======================================================================
//  C ABI
// ======================================================================
using namespace speo;

extern "C" {

int speo_init_population(float *X, int ld, int n, int dim, float lo, float hi, uint64_t seed,
                         uint32_t row_base, speo_stream_t stream) {
    if (!X || n < 0 || dim < 1 || ld < dim || (ld & 3) || (reinterpret_cast<uintptr_t>(X) & 15))
        return set_error(SPEO_ERR_ARG, "speo_init_population: need ld >= dim, ld % 4 == 0 and "
                                       "a 16-byte aligned X");
    return init_population(X, ld, n, dim, lo, hi, seed, row_base, as_stream(stream));
}

int speo_de_generate(float *U, const float *X, int ld, int n, int dim, int subisland_num,
                     const int *perm, const DEInfo *de_info, const int *best, float lo, float hi,
                     SPEO_RandState rng, const float *inj_r, int n_inj, const float *inj_cr,
                     int *r_out, int *jrand_out, speo_stream_t stream) {
    if (!U || !X || !de_info || n < 0 || dim < 1 || ld < dim || subisland_num < 1 ||
        n % subisland_num || (n > 0 && n / subisland_num < 4) || n_inj < 0 ||
        (inj_r && n_inj == 0))
        return set_error(SPEO_ERR_ARG, "speo_de_generate: need ld >= dim and equal sub-islands "
                                       "of at least 4 rows");
    GenArgs a{U, X, ld, n, dim, n > 0 ? n / subisland_num : 1, perm, de_info, best, lo, hi,
              rng.seed, rng.generation, rng.row_base, inj_r, n_inj, inj_cr, r_out, jrand_out};
    return de_generate(a, as_stream(stream));
}

int speo_de_select(float *X, float *fX, const float *U, const float *fU, int ld, int n, int dim,
                   uint8_t *accept_out, speo_stream_t stream) {
    if (!X || !fX || !U || !fU || n < 0 || ld < dim)
        return set_error(SPEO_ERR_ARG, "speo_de_select: bad arguments");
    return de_select(X, fX, U, const_cast<float *>(fU), ld, n, dim, accept_out, 0,
                     as_stream(stream));
}

int speo_segment_argmin(const float *f, const int *off, int nseg, int *best_out,
                        speo_stream_t stream) {
    if (!f || !off || !best_out || nseg < 0)
        return set_error(SPEO_ERR_ARG, "speo_segment_argmin: bad arguments");
    return segment_argmin(f, off, nseg, best_out, as_stream(stream));
}

// ---- drop-in layer ----------------------------------------------------

int API_Initilize(GPU_Population d_population, SPEO_RandState *rand_state,
                  GPU_IslandInfo info, ProblemInfo pi) {
    if (!rand_state || !d_population.elements || info.island_size < 0 || pi.dim < 1)
        return set_error(SPEO_ERR_ARG, "API_Initilize: bad arguments");
    // global_SetupRandomState(d_rand_states, problem_info.seed), kernel_EA_CUDA.cu:128
    rand_state->seed = (uint64_t)(uint32_t)pi.seed;
    rand_state->generation = 0;
    rand_state->row_base = 0;
    const int ld = next_pow2_dim(pi.dim);
    return init_population(d_population.elements, ld, info.island_size, pi.dim, pi.min_bound,
                           pi.max_bound, rand_state->seed, rand_state->row_base, nullptr);
}

int API_DE_GenerateNewPopulation(GPU_Population d_candidate, GPU_Population d_population,
                                 int *d_best_individual_ID, GPU_IslandInfo info,
                                 DEInfo *d_DE_info, SPEO_RandState *rand_state,
                                 ProblemInfo pi) {
    const int n = info.island_size, subs = info.subisland_num;
    if (!rand_state || !d_DE_info || !d_candidate.elements || !d_population.elements ||
        !d_population.fitness_value || n <= 0 || subs < 1 || n % subs || n / subs < 4 ||
        pi.dim < 1)
        return set_error(SPEO_ERR_ARG, "API_DE_GenerateNewPopulation: need equal sub-islands "
                                       "of at least 4 individuals");
    const int S = n / subs;
    // global_DE_FindBestIndividualInIsland (kernel_DE_CUDA.cu:120-158), with
    // each sub-island's own offset into permutated_index.
    GenArgs a{d_candidate.elements, d_population.elements, next_pow2_dim(pi.dim), n, pi.dim, S,
              info.permutated_index, d_DE_info, nullptr, pi.min_bound,
              pi.max_bound, rand_state->seed, rand_state->generation, rand_state->row_base,
              nullptr, 0, nullptr, nullptr, nullptr};
    if (d_best_individual_ID) {
        a.fit = d_population.fitness_value;
        a.best_out = d_best_individual_ID;
    }
    SPEO_TRY(de_generate(a, nullptr));
    rand_state->generation++;
    return SPEO_OK;
}

int API_DE_SelectSurvival(GPU_Population d_population, GPU_Population d_candidate,
                          GPU_IslandInfo info, ProblemInfo pi) {
    if (!d_population.elements || !d_population.fitness_value || !d_candidate.elements ||
        !d_candidate.fitness_value || info.island_size < 0 || pi.dim < 1)
        return set_error(SPEO_ERR_ARG, "API_DE_SelectSurvival: bad arguments");
    return de_select(d_population.elements, d_population.fitness_value, d_candidate.elements,
                     d_candidate.fitness_value, next_pow2_dim(pi.dim), info.island_size, pi.dim,
                     nullptr, 0, nullptr);
}

}  // extern "C"

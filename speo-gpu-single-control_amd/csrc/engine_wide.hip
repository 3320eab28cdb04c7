// engine_wide.hip -- evaluation of the engine's islands wider than 128 columns:
// every row's objective as the generation kernel's K-chunked form computes it
// (gemm_chunk over the 128-column chunks in order, the lane's sums carried from
// chunk to chunk, then the 16 lanes and the column classes), on the pipelined
// tile kernel of wide_core.h.
//
// What bounds it: the tile kernel's matrix work and its stages' LDS reads
// (BF16x3, 8 islands x 2048 rows x 1000, three components: 335 us, 45 % of the
// matrix pipe), then the row traffic of the trials (55 us) and the distances'
// serial sums (26 us).  Evaluated inside the generation kernel, one block per
// 64 rows with its components one after another and one lane per row for the
// distances, a generation took 8.5 ms; 0.42 ms now.
//
// Reference counterpart: API_evaluateFitness on an island's population
// (kernel_CEC2014_CUDA.cu:147-181, 1672-1797) and the composition chain
// CalW / CombineFitness (:1416-1671).
#pragma clang fp contract(off)

#include <algorithm>
#include <mutex>

#include "engine.h"
#include "eval.h"
#include "wide_core.h"

namespace speo {

namespace {

// 64 rows x 128 columns per block of four waves, the wave's share of a chunk
// its column class.  Three blocks fit a compute unit (two stage buffers each):
// 8 islands of 2048 rows and three components are 768 blocks, three per unit.
template <int PREC, int NSPLIT> using RowsTile = WideTile<PREC, 4 / NSPLIT, NSPLIT, 1, NSPLIT, 2>;

template <int OBJ, int RTW, int TPW, int NSPLIT>
__device__ __forceinline__ void chain_terms(const floatx4 (&acc)[RTW][TPW], const float *colw, int n0, int dim,
                                            int lr, float unscale, float (&s1)[RTW][4], float (&s2)[RTW][4]) {
#pragma unroll
    for (int t = 0; t < TPW; ++t) {
        const int col = n0 + t * NSPLIT * 16 + lr;
        if (col < dim) {
            const float w = OBJ == SPEO_OBJ_ELLIPTIC ? gld(colw + col) : 1.0f;
#pragma unroll
            for (int i = 0; i < RTW; ++i)
#pragma unroll
                for (int q = 0; q < 4; ++q) add_terms(OBJ, acc[i][t][q] * unscale, w, s1[i][q], s2[i][q]);
        }
    }
}

// The value of one component for the item's rows, from its row sums.
__device__ __forceinline__ void put_value(const WideRowsArgs &p, const WideItem &it, const FusedProblem *P, int r,
                                          float g) {
    if (P->ncomp == 1)
        p.f[it.row + r] = fmaf(P->lambda[0], g, P->bias[0]);
    else
        p.gval[(size_t)it.comp * p.rows + it.row + r] = g;
}

template <int PREC, int NSPLIT>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(PREC == SPEO_PREC_BF16X6 ? 2 : 3))) void
k_rows_wide(WideRowsArgs p) {
    using W = RowsTile<PREC, NSPLIT>;
    static_assert(W::RB == kWideRows && W::NT == 256, "tile");
    extern __shared__ __align__(16) char lds[];
    const WideItem it = p.items[blockIdx.x];
    const FusedProblem *P = p.probs + it.problem;
    const CompDev &c = P->comp[it.comp];
    const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
    const int lr = lane & 15, lk = lane >> 4;
    const int wn = wave % NSPLIT, rg = wave / NSPLIT, dim = it.dim;
    const float *rows = p.src + it.elem;
    float *shs = reinterpret_cast<float *>(lds + W::LDS);
    for (int k = tid; k < round_up(dim, 32); k += W::NT) shs[k] = k < dim ? gld(c.shift + k) : 0.f;
    __syncthreads();
    const float unscale = W::H ? kF16Unscale : 1.0f;
    const int objective = c.objective;
    const float *colw = c.colw;
    float s1[W::RTW][4], s2[W::RTW][4];
#pragma unroll
    for (int i = 0; i < W::RTW; ++i)
#pragma unroll
        for (int q = 0; q < 4; ++q) s1[i][q] = s2[i][q] = 0.f;
    const WideOperands o{rows, it.ld, it.nrows, dim, c.wide, (int)(2 * wide_frag_elems(dim)),
                         c.rate == 1.0f ? 1 : 0, c.rate};
    wide_gemm<PREC, W>(o, 0, (dim + kNC - 1) / kNC, lds, shs,
                       [&](int chunk, const floatx4 (&acc)[W::RTW][W::TPW]) __attribute__((always_inline)) {
                           const int n0 = chunk * kNC + wn * 16;
                           switch (objective) {  // the objective dispatch of with_objective
#define SPEO_TERMS(O) chain_terms<O, W::RTW, W::TPW, NSPLIT>(acc, colw, n0, dim, lr, unscale, s1, s2); break
                           case SPEO_OBJ_ELLIPTIC: SPEO_TERMS(SPEO_OBJ_ELLIPTIC);
                           case SPEO_OBJ_RASTRIGIN: SPEO_TERMS(SPEO_OBJ_RASTRIGIN);
                           case SPEO_OBJ_ACKLEY: SPEO_TERMS(SPEO_OBJ_ACKLEY);
                           case SPEO_OBJ_SCHWEFEL: SPEO_TERMS(SPEO_OBJ_SCHWEFEL);
                           default: SPEO_TERMS(SPEO_OBJ_HAPPYCAT);
#undef SPEO_TERMS
                           }
                       });
    __syncthreads();  // the stage buffers become the row-sum area
    float *red = reinterpret_cast<float *>(lds);  // [class][row][2]
#pragma unroll
    for (int i = 0; i < W::RTW; ++i)
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const float a1 = sum16(s1[i][q]), a2 = sum16(s2[i][q]);
            if (lr == 0) {
                const int r = rg * W::WR + i * 16 + lk * 4 + q;
                red[(wn * kWideRows + r) * 2 + 0] = a1;
                red[(wn * kWideRows + r) * 2 + 1] = a2;
            }
        }
    __syncthreads();
    float *g = red + NSPLIT * kWideRows * 2;
    if (tid < it.nrows) {
        float a = 0.f, b = 0.f;
        for (int w = 0; w < NSPLIT; ++w) {
            a += red[(w * kWideRows + tid) * 2 + 0];
            b += red[(w * kWideRows + tid) * 2 + 1];
        }
        g[tid] = finish_objective_ext(objective, a, b, dim);
    }
    if (c.heavy.j >= 0) {
        // the heavy column's FP64 term, one wave per row
        __syncthreads();
        for (int r = wave; r < it.nrows; r += W::NW) {
            const double h = heavy_term(c.heavy, rows + (size_t)r * it.ld, dim, lane);
            if (lane == 0) g[r] = with_heavy(g[r], (float)h);
        }
        __syncthreads();
    }
    if (tid < it.nrows) put_value(p, it, P, tid, g[tid]);
}

// The same from gemm_chunk itself, for components the tile kernel does not
// take (fragments beyond 2 GiB, a shift that does not fit LDS; engines created
// with the tile kernels switched off).  RT = 64 / NSPLIT.
template <int PREC, int NSPLIT>
__global__ __launch_bounds__(256) void k_rows_chunk(WideRowsArgs p) {
    constexpr int RT = 64 / NSPLIT;
    extern __shared__ __align__(16) char lds[];
    const WideItem it = p.items[blockIdx.x];
    const FusedProblem *P = p.probs + it.problem;
    const CompDev c = P->comp[it.comp];
    const int tid = threadIdx.x, dim = it.dim;
    for (int r0 = 0; r0 < it.nrows; r0 += RT) {
        const int nrows = min(RT, it.nrows - r0);
        const RowSource src{p.src + it.elem + (size_t)r0 * it.ld, it.ld, nrows};
        float *red = reinterpret_cast<float *>(lds);
        float *o1 = red + 8 * RT, *o2 = o1 + RT, *g = o2 + RT;
        float s1[4] = {0.f, 0.f, 0.f, 0.f}, s2[4] = {0.f, 0.f, 0.f, 0.f};
        for (int n0 = 0; n0 < dim; n0 += kNC) gemm_chunk<RT, PREC>(c, src, dim, n0, lds, s1, s2);
        reduce_rows<RT>(s1, s2, red, o1, o2);
        if (tid < nrows) g[tid] = finish_objective_ext(c.objective, o1[tid], o2[tid], dim);
        if (c.heavy.j >= 0) {
            __syncthreads();
            const int wave = tid >> 6, lane = tid & 63;
            for (int r = wave; r < nrows; r += 4) {
                const double h = heavy_term(c.heavy, src.rows + (size_t)r * src.ld, dim, lane);
                if (lane == 0) g[r] = with_heavy(g[r], (float)h);
            }
            __syncthreads();
        }
        if (tid < nrows) put_value(p, it, P, r0 + tid, g[tid]);
        __syncthreads();
    }
}

// cf_cal weights (CEC2014.cc:1481-1519) in the log domain and the weighted sum
// of a composition's component values, for an item's 64 rows (components at
// distance 0 share the weight equally, as cf_cal's w = 1e99 each).  The squared
// distances are the generation kernel's: one fused multiply-add chain over the
// coordinates in order, here one lane per (row, component) over 64-column
// pieces of the rows and shifts staged in LDS (a lane per row reading its row
// and every shift from memory took milliseconds at D = 1000).
// The next two pieces are in flight while this one is summed: with two barriers a
// piece and its loads between them 16,384 rows of D = 1000 and three components
// took 52 us, 26 us so.
constexpr int kCombLd = 68;  // row stride (floats) in LDS: 16-byte reads of 16 rows in different banks
constexpr int kCombGroups = kWideRows * 16 / 128;  // 16-byte groups of a piece per thread, two components or more
__global__ __launch_bounds__(64 * kMaxComp) void k_rows_combine(WideRowsArgs p) {
    __shared__ __align__(16) float xs[2][kWideRows * kCombLd], os[2][kMaxComp * 64];
    __shared__ float lws[kMaxComp][kWideRows], ds[kMaxComp][kWideRows];
    const WideItem it = p.items[blockIdx.x];
    const FusedProblem *P = p.probs + it.problem;
    const int nc = P->ncomp, dim = it.dim;
    if (it.comp != 0 || nc == 1) return;
    const int tid = threadIdx.x, c = tid >> 6, r = tid & 63, nt = blockDim.x;
    const bool mine = c < nc && r < it.nrows;
    const float *rows = p.src + it.elem;
    struct Piece {
        floatx4 x[kCombGroups];
        float o;
    };
    const float *shift = P->comp[min(c, nc - 1)].shift;
    // (addresses are clamped, not loads skipped: nothing waits on a merge)
    auto load = [&](Piece &q, int k0) {
        if (k0 >= dim) return;
        const int kc = min(64, dim - k0);
#pragma unroll
        for (int i = 0; i < kCombGroups; ++i)
            if (i * nt < kWideRows * 16) {
                const int e = tid + i * nt, rr = min(e >> 4, it.nrows - 1), k = (e & 15) * 4;
                q.x[i] = gld(reinterpret_cast<const floatx4 *>(rows + (size_t)rr * it.ld + k0 + (k < kc ? k : 0)));
            }
        q.o = shift[k0 + min(r, kc - 1)];
    };
    auto store = [&](const Piece &q, int b, int k0) {
        if (k0 >= dim) return;
#pragma unroll
        for (int i = 0; i < kCombGroups; ++i)
            if (i * nt < kWideRows * 16) {
                const int e = tid + i * nt, rr = e >> 4, k = (e & 15) * 4;
                if (rr < kWideRows) *reinterpret_cast<floatx4 *>(xs[b] + rr * kCombLd + k) = q.x[i];
            }
        os[b][c * 64 + r] = q.o;
    };
    float d = 0.f;
    auto sum = [&](int b, int k0) {
        const int kc = min(64, dim - k0);
        if (!mine || kc <= 0) return;
        const float *xr = xs[b] + r * kCombLd, *o = os[b] + c * 64;
        if (kc == 64) {
#pragma unroll
            for (int k = 0; k < 64; k += 4) {
                const float4 xv = *reinterpret_cast<const float4 *>(xr + k);
                const float4 ov = *reinterpret_cast<const float4 *>(o + k);
                const float v0 = xv.x - ov.x, v1 = xv.y - ov.y, v2 = xv.z - ov.z, v3 = xv.w - ov.w;
                d = fmaf(v0, v0, d);
                d = fmaf(v1, v1, d);
                d = fmaf(v2, v2, d);
                d = fmaf(v3, v3, d);
            }
        } else {
            for (int k = 0; k < kc; ++k) {
                const float v = xr[k] - o[k];
                d = fmaf(v, v, d);
            }
        }
    };
    // each buffer is written after the barrier behind its last reads
    Piece qa, qb;
    load(qa, 0);
    load(qb, 64);
    store(qa, 0, 0);
    __syncthreads();
    for (int k0 = 0; k0 < dim; k0 += 128) {
        load(qa, k0 + 128);
        sum(0, k0);
        store(qb, 1, k0 + 64);
        __syncthreads();
        load(qb, k0 + 192);
        sum(1, k0 + 64);
        store(qa, 0, k0 + 128);
        __syncthreads();
    }
    if (mine) {
        const float s = P->sigma[c];
        ds[c][r] = d;
        lws[c][r] = -0.5f * logf(d) - d / (2.0f * (float)dim * s * s);
    }
    __syncthreads();
    if (c == 0 && r < it.nrows) {
        float lwmax = -INFINITY;
        bool any_zero = false;
        for (int k = 0; k < nc; ++k) {
            any_zero = any_zero || ds[k][r] == 0.f;
            lwmax = fmaxf(lwmax, lws[k][r]);
        }
        float wsum = 0.f, acc = 0.f;
        for (int k = 0; k < nc; ++k) {
            const float w = any_zero ? (ds[k][r] == 0.f ? 1.f : 0.f) : expf(lws[k][r] - lwmax);
            wsum += w;
            acc = fmaf(w, fmaf(P->lambda[k], p.gval[(size_t)k * p.rows + it.row + r], P->bias[k]), acc);
        }
        p.f[it.row + r] = acc / wsum;
    }
}

template <int PREC, int NSPLIT>
int launch_rows(const WideRowsArgs &a, int nitems, int max_dim, bool chunk, hipStream_t s) {
    using W = RowsTile<PREC, NSPLIT>;
    static std::once_flag once;
    std::call_once(once, [] {
        (void)hipFuncSetAttribute(reinterpret_cast<const void *>(&k_rows_wide<PREC, NSPLIT>),
                                  hipFuncAttributeMaxDynamicSharedMemorySize, kWideLdsMax);
        (void)hipFuncSetAttribute(reinterpret_cast<const void *>(&k_rows_chunk<PREC, NSPLIT>),
                                  hipFuncAttributeMaxDynamicSharedMemorySize, kWideLdsMax);
    });
    if (chunk) {
        constexpr int RT = 64 / NSPLIT;
        hipLaunchKernelGGL((k_rows_chunk<PREC, NSPLIT>), dim3(nitems), dim3(256),
                           std::max(gemm_lds_bytes<RT, PREC>(), 11 * RT * 4), s, a);
        return check_launch("k_rows_chunk");
    }
    hipLaunchKernelGGL((k_rows_wide<PREC, NSPLIT>), dim3(nitems), dim3(256), W::LDS + 4 * round_up(max_dim, 32),
                       s, a);
    return check_launch("k_rows_wide");
}

template <int PREC>
int launch_split(const WideRowsArgs &a, int nitems, int max_dim, int nsplit, bool chunk, hipStream_t s) {
    switch (nsplit) {
    case 1: return launch_rows<PREC, 1>(a, nitems, max_dim, chunk, s);
    case 2: return launch_rows<PREC, 2>(a, nitems, max_dim, chunk, s);
    default: return launch_rows<PREC, 4>(a, nitems, max_dim, chunk, s);
    }
}

int launch_any(const WideRowsArgs &a, int nitems, int max_dim, int precision, int nsplit, bool chunk,
               hipStream_t s) {
    if (nitems <= 0) return SPEO_OK;
    switch (precision) {
    case SPEO_PREC_FP32: return launch_split<SPEO_PREC_FP32>(a, nitems, max_dim, nsplit, chunk, s);
    case SPEO_PREC_BF16: return launch_split<SPEO_PREC_BF16>(a, nitems, max_dim, nsplit, chunk, s);
    case SPEO_PREC_FP16: return launch_split<SPEO_PREC_FP16>(a, nitems, max_dim, nsplit, chunk, s);
    case SPEO_PREC_BF16X3: return launch_split<SPEO_PREC_BF16X3>(a, nitems, max_dim, nsplit, chunk, s);
    case SPEO_PREC_FP16X3: return launch_split<SPEO_PREC_FP16X3>(a, nitems, max_dim, nsplit, chunk, s);
    case SPEO_PREC_BF16X6: return launch_split<SPEO_PREC_BF16X6>(a, nitems, max_dim, nsplit, chunk, s);
    default: return set_error(SPEO_ERR_ARG, "unknown precision");
    }
}

}  // namespace

bool rows_wide_applies(const CompDev &c, int dim, int precision) {
    const int parts = precision == SPEO_PREC_FP32 ? 2
                      : precision == SPEO_PREC_BF16 || precision == SPEO_PREC_FP16 ? 1
                      : precision == SPEO_PREC_BF16X6 ? 3 : 2;
    const int lds = 2 * (kWideRows * 128 + 8 * parts * 1024);
    return wide_eval_enabled() && c.wide && lds + 4 * (int64_t)round_up(dim, 32) <= kWideLdsMax;
}

int rows_wide(const WideRowsArgs &a, int nitems, int max_dim, int precision, int nsplit, hipStream_t s) {
    return launch_any(a, nitems, max_dim, precision, nsplit, false, s);
}
int rows_chunk(const WideRowsArgs &a, int nitems, int precision, int nsplit, hipStream_t s) {
    return launch_any(a, nitems, 0, precision, nsplit, true, s);
}
int rows_combine(const WideRowsArgs &a, int nitems, int ncomp, hipStream_t s) {
    if (nitems <= 0) return SPEO_OK;
    hipLaunchKernelGGL(k_rows_combine, dim3(nitems), dim3(64 * ncomp), 0, s, a);
    return check_launch("k_rows_combine");
}

}  // namespace speo

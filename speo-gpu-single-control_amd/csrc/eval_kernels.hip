// eval_kernels.hip -- fused shift + rotation-GEMM + objective kernels, the FP64
// re-verification kernel and the composition combine.
//
// Replaces the reference's per-objective launch chains (API_evaluateFitness,
// kernel_CEC2014_CUDA.cu:1672-1797: ShiftAndRotation -> global_fN, plus
// CalW/CombineFitness for compositions) by one kernel per N chunk of Z.
#include <algorithm>
#include <atomic>
#include <map>
#include <mutex>
#include <tuple>
#include <unordered_map>

#include "cec_generic.h"
#include "eval.h"

namespace speo {

// ------------------------------------------------------------------ kernels

template <int RT, int PREC> constexpr int eval_small_lds_bytes() {
    return RT * kTS * 4 + small_scratch_bytes<RT>(Prec<PREC>::parts) + 10 * RT * 4;
}

// How a kernel evaluates its rows: by K chunks (gemm_chunk), the rotation in a
// problem's layouts for up to 128 columns, or in c.B32's rows alone (the same
// columns, FP32).  A kernel holds one of them: with the small path's code beside
// it the chunked form was 1 to 2 % slower (FP32, one component: a row of D = 1000
// 45.3 us, 44.6 alone; 1,000 rows of D = 500 25.5 / 25.2).
enum EvalForm { kEvalChunk, kEvalSmall, kEvalRaw };
template <int RT, int PREC, EvalForm FORM>
__device__ __forceinline__ void eval_rows(const EvalLaunch &p, const CompDev &c, int chunk, float *f_out) {
    extern __shared__ __align__(16) char lds[];
    const int row0 = blockIdx.x * RT;
    const int nrows = min(RT, p.n - row0);
    float *o1, *o2;
    if constexpr (FORM != kEvalChunk) {
        constexpr bool RAW = FORM == kEvalRaw;
        float *rows = reinterpret_cast<float *>(lds);
        char *scratch = lds + RT * kTS * 4;
        float *red = reinterpret_cast<float *>(scratch + small_scratch_bytes<RT>(Prec<PREC>::parts));
        o1 = red + 8 * RT;
        o2 = o1 + RT;
        const int kp4 = (p.dim + 3) & ~3, cls = column_class();
        SmallB B;
        constexpr bool F32 = Prec<PREC>::parts == 0;
        if constexpr (RAW) B.load_rows(c, p.dim, cls);
        else if constexpr (F32) B.load(c, p.dim, cls);
        if ((p.ld & 3) == 0 && (reinterpret_cast<uintptr_t>(p.X) & 15) == 0) {
            // 16-byte loads, all of the tile issued before the first is
            // stored; columns >= dim set to 0 (the row's padding may hold
            // anything)
            constexpr int G = RT * (kSmallD / 4) / 256;  // groups per thread at most
            const int ng = kp4 >> 2;
            floatx4 x[G];
#pragma unroll
            for (int i = 0; i < G; ++i) {
                const int e = threadIdx.x + i * 256, r = e / ng, g = e - r * ng;
                const bool ok = e < RT * ng && r < nrows;
                x[i] = gld(reinterpret_cast<const floatx4 *>(p.X + (ok ? (size_t)(row0 + r) * p.ld + 4 * g : 0)));
            }
#pragma unroll
            for (int i = 0; i < G; ++i) {
                const int e = threadIdx.x + i * 256, r = e / ng, g = e - r * ng;
                if (e >= RT * ng) break;
                floatx4 v = x[i];
#pragma unroll
                for (int q = 0; q < 4; ++q)
                    if (r >= nrows || 4 * g + q >= p.dim) v[q] = 0.f;
                *reinterpret_cast<floatx4 *>(rows + r * kTS + 4 * g) = v;
            }
        } else {
            // a wave per row, every fourth row; all loads of the tile issued
            // before the first is stored
            const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
            float x[RT / 4][2];
#pragma unroll
            for (int i = 0; i < RT / 4; ++i)
#pragma unroll
                for (int h = 0; h < 2; ++h) {
                    const int r = min(wave + 4 * i, nrows - 1), k = min(lane + 64 * h, p.dim - 1);
                    x[i][h] = gld(p.X + (size_t)(row0 + r) * p.ld + k);
                }
#pragma unroll
            for (int i = 0; i < RT / 4; ++i)
#pragma unroll
                for (int h = 0; h < 2; ++h) {
                    const int r = wave + 4 * i, k = lane + 64 * h;
                    if (k < kp4) rows[r * kTS + k] = r < nrows && k < p.dim ? x[i][h] : 0.f;
                }
        }
        if constexpr (F32) B.stage(scratch);
        __syncthreads();
        float s1[RT / 16][4], s2[RT / 16][4];
        if constexpr (F32) gemm_small_f32<RT>(c, B, rows, p.dim, cls, scratch, s1, s2);
        else gemm_small<RT, PREC>(c, rows, p.dim, cls, scratch, s1, s2);
        reduce_rows_small<RT>(s1, s2, cls, red, o1, o2);
    } else {
        RowSource src{p.X + (size_t)row0 * p.ld, p.ld, nrows};
        float s1[4] = {0.f, 0.f, 0.f, 0.f}, s2[4] = {0.f, 0.f, 0.f, 0.f};
        gemm_chunk<RT, PREC>(c, src, p.dim, chunk * kNC, lds, s1, s2);
        float *red = reinterpret_cast<float *>(lds);
        o1 = red + 4 * RT * 2;
        o2 = o1 + RT;
        reduce_rows<RT>(s1, s2, red, o1, o2);
    }
    if (c.heavy.j >= 0 && chunk == 0) {
        // the heavy column's FP64 term, one wave per row, into the row sums
        // (the row staging area is free after the reductions' barriers)
        const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
        heavy_rows(c.heavy, p.dim, wave, 4, nrows, lane,
                   [&](int r) { return p.X + (size_t)(row0 + r) * p.ld; },
                   [&](int r, double h) { if (lane == 0) o1[r] = with_heavy(o1[r], (float)h); });
        __syncthreads();
    }
    const int t = threadIdx.x;
    if (t < RT && row0 + t < p.n) {
        const int row = row0 + t;
        if (p.nchunks == 1) {
            const float g = finish_objective_ext(c.objective, o1[t], o2[t], p.dim);
            f_out[row] = p.raw ? g : fmaf(p.lambda, g, p.bias);
        } else {
            p.part[((size_t)chunk * 2 + 0) * p.n + row] = o1[t];
            p.part[((size_t)chunk * 2 + 1) * p.n + row] = o2[t];
        }
    }
}

template <int RT, int PREC, EvalForm FORM>
__global__ __launch_bounds__(256) void k_eval(EvalLaunch p) {
    eval_rows<RT, PREC, FORM>(p, p.comp, blockIdx.y, p.f_out);
}

// The components of a composition of up to 128 columns in one launch: block row
// blockIdx.y is component y, its values at f_out + y n.
struct EvalComps {
    EvalLaunch p;
    CompDev comp[kMaxComp];
};
template <int RT, int PREC>
__global__ __launch_bounds__(256) void k_eval_comps(EvalComps a) {
    eval_rows<RT, PREC, kEvalSmall>(a.p, a.comp[blockIdx.y], 0, a.p.f_out + (size_t)blockIdx.y * a.p.n);
}

// The chunks' sums of component blockIdx.y (in chunk order) and its value.
struct FinalizeObjectives {
    int obj[kMaxComp];
};
__global__ void k_eval_finalize(const float *part, int nchunks, int n, int dim, FinalizeObjectives objectives,
                                float lambda, float bias, int raw, float *f_out) {
    const int row = blockIdx.x * blockDim.x + threadIdx.x, k = blockIdx.y;
    if (row >= n) return;
    part += (size_t)k * nchunks * 2 * n;
    float a = 0.f, b = 0.f;
    for (int c = 0; c < nchunks; ++c) {
        a += part[((size_t)c * 2 + 0) * n + row];
        b += part[((size_t)c * 2 + 1) * n + row];
    }
    const float g = finish_objective_ext(objectives.obj[k], a, b, dim);
    f_out[(size_t)k * n + row] = raw ? g : fmaf(lambda, g, bias);
}

// Composition (cf_cal, CEC2014.cc:1481-1519) in FP32: one wave per row.
// Weights in the log domain, lw_c = -log(d_c)/2 - d_c / (2 D sigma_c^2),
// normalised by their maximum, so no weight underflows before the ratio is
// formed; components with d_c == 0 share all the weight equally (cf_cal gives
// each of them w = 1e99, beside which every other weight vanishes).
// One wave per row: the row's squared distance to each component's shift
// (per-lane partial sums, then a butterfly over the 64 lanes), the cf_cal
// weights in the log domain and the weighted sum.  When the row stride, X and
// every shift allow 16-byte loads and dim % 4 == 0, lane l takes coordinates
// 4 (l + 64 i) .. + 3; otherwise coordinates l + 64 i.  Up to 1024 coordinates
// the row is read once into registers for all components (4,000 rows of D = 515
// and three components in BF16: 46.2 us with the row read again for each, 41.8
// so; compiled for at most four waves a SIMD unit it was slower than either).
__global__ void k_comp_combine(const CompParams *comps, int ncomp, int dim, const float *X,
                               int ld, int n, const float *g, float *f_out) {
    constexpr int kGroups = 4;  // float4 groups per lane held in registers
    const int wave = (blockIdx.x * blockDim.x + threadIdx.x) >> 6;
    const int lane = threadIdx.x & 63;
    if (wave >= n) return;
    const float *x = X + (size_t)wave * ld;
    const int ng = dim >> 2;
    bool vec = (dim & 3) == 0 && (ld & 3) == 0 && (reinterpret_cast<uintptr_t>(X) & 15) == 0 &&
               ng <= 64 * kGroups;
    for (int c = 0; c < ncomp; ++c) vec = vec && (reinterpret_cast<uintptr_t>(comps[c].shift32) & 15) == 0;
    float4 xr[kGroups];
    if (vec) {
#pragma unroll
        for (int i = 0; i < kGroups; ++i) {
            const int q = lane + 64 * i;
            xr[i] = q < ng ? *reinterpret_cast<const float4 *>(x + 4 * q) : float4{0.f, 0.f, 0.f, 0.f};
        }
    }
    constexpr int kSingles = 16;  // coordinates per lane held where 16-byte loads cannot be used
    const bool held = !vec && dim <= 64 * kSingles;
    float xs[kSingles];
    if (held) {
#pragma unroll
        for (int i = 0; i < kSingles; ++i)
            if (64 * i < dim) xs[i] = gld(x + min(lane + 64 * i, dim - 1));
    }
    float lw[kMaxComp];
    bool zero[kMaxComp];
    bool any_zero = false;
    float lwmax = -INFINITY;
    for (int c = 0; c < ncomp; ++c) {
        const float *o = comps[c].shift32;
        float d = 0.f;
        if (held) {
            float os[kSingles];
#pragma unroll
            for (int i = 0; i < kSingles; ++i)
                if (64 * i < dim) os[i] = gld(o + min(lane + 64 * i, dim - 1));
#pragma unroll
            for (int i = 0; i < kSingles; ++i)
                if (lane + 64 * i < dim) {
                    const float v = xs[i] - os[i];
                    d = fmaf(v, v, d);
                }
        } else if (vec) {
#pragma unroll
            for (int i = 0; i < kGroups; ++i) {
                const int q = lane + 64 * i;
                if (q < ng) {
                    const float4 ov = *reinterpret_cast<const float4 *>(o + 4 * q);
                    const float v0 = xr[i].x - ov.x, v1 = xr[i].y - ov.y, v2 = xr[i].z - ov.z,
                                v3 = xr[i].w - ov.w;
                    d = fmaf(v0, v0, d);
                    d = fmaf(v1, v1, d);
                    d = fmaf(v2, v2, d);
                    d = fmaf(v3, v3, d);
                }
            }
        } else {
            for (int j = lane; j < dim; j += 64) {
                const float v = x[j] - o[j];
                d = fmaf(v, v, d);
            }
        }
        for (int off = 32; off > 0; off >>= 1) d += __shfl_xor(d, off, 64);
        zero[c] = d == 0.f;
        any_zero = any_zero || zero[c];
        const float s = (float)comps[c].sigma;
        lw[c] = -0.5f * logf(d) - d / (2.0f * (float)dim * s * s);
        lwmax = fmaxf(lwmax, lw[c]);
    }
    if (lane == 0) {
        float wsum = 0.f, acc = 0.f;
        for (int c = 0; c < ncomp; ++c) {
            const float w = any_zero ? (zero[c] ? 1.f : 0.f) : expf(lw[c] - lwmax);
            const float fit = fmaf((float)comps[c].lambda, g[(size_t)c * n + wave], (float)comps[c].bias);
            wsum += w;
            acc = fmaf(w, fit, acc);
        }
        f_out[wave] = acc / wsum;
    }
}

// k_comp_combine's 16-byte path for many rows: the shifts staged in LDS once
// per block, kCombRows rows per wave with the next row's loads (X and the
// component values g) in flight while the current row is combined.  Lane c
// (c < ncomp) forms component c's weight and value, and lane 0 sums them in
// component order: the same arithmetic as k_comp_combine, result for result.
constexpr int kCombRows = 4;
__global__ __launch_bounds__(256) void k_comp_combine_rows(const CompParams *comps, int ncomp, int dim,
                                                           const float *X, int ld, int n,
                                                           const float *g, float *f_out) {
    constexpr int kGroups = 4;
    extern __shared__ __align__(16) float osh[];  // [ncomp][dim]
    __shared__ float sig[kMaxComp], lam[kMaxComp], bia[kMaxComp];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int ng = dim >> 2;
    for (int c = 0; c < ncomp; ++c)
        for (int q = tid; q < ng; q += 256)
            reinterpret_cast<float4 *>(osh + (size_t)c * dim)[q] =
                reinterpret_cast<const float4 *>(comps[c].shift32)[q];
    if (tid < ncomp) {
        sig[tid] = (float)comps[tid].sigma;
        lam[tid] = (float)comps[tid].lambda;
        bia[tid] = (float)comps[tid].bias;
    }
    const int row0 = (blockIdx.x * 4 + wave) * kCombRows;
    auto load = [&](int r, float4 (&xr)[kGroups], float &gv) {
#pragma unroll
        for (int i = 0; i < kGroups; ++i) {
            const int q = lane + 64 * i;
            xr[i] = r < n && q < ng ? *reinterpret_cast<const float4 *>(X + (size_t)r * ld + 4 * q)
                                    : float4{0.f, 0.f, 0.f, 0.f};
        }
        gv = r < n && lane < ncomp ? g[(size_t)lane * n + r] : 0.f;
    };
    float4 cur[kGroups], nxt[kGroups];
    float gcur, gnxt;
    load(row0, cur, gcur);
    __syncthreads();
    for (int k = 0; k < kCombRows; ++k) {
        const int r = row0 + k;
        if (r >= n) break;  // wave-uniform
        load(r + 1, nxt, gnxt);
        float my_lw = -INFINITY, lwmax = -INFINITY;
        bool my_zero = false, any_zero = false;
        for (int c = 0; c < ncomp; ++c) {
            const float *o = osh + (size_t)c * dim;
            float d = 0.f;
#pragma unroll
            for (int i = 0; i < kGroups; ++i) {
                const int q = lane + 64 * i;
                if (q < ng) {
                    const float4 ov = *reinterpret_cast<const float4 *>(o + 4 * q);
                    const float v0 = cur[i].x - ov.x, v1 = cur[i].y - ov.y, v2 = cur[i].z - ov.z,
                                v3 = cur[i].w - ov.w;
                    d = fmaf(v0, v0, d);
                    d = fmaf(v1, v1, d);
                    d = fmaf(v2, v2, d);
                    d = fmaf(v3, v3, d);
                }
            }
            for (int off = 32; off > 0; off >>= 1) d += __shfl_xor(d, off, 64);
            const float s = sig[c];
            const float lw = -0.5f * logf(d) - d / (2.0f * (float)dim * s * s);
            any_zero = any_zero || d == 0.f;
            lwmax = fmaxf(lwmax, lw);
            if (lane == c) {
                my_lw = lw;
                my_zero = d == 0.f;
            }
        }
        float w = 0.f, fit = 0.f;
        if (lane < ncomp) {
            w = any_zero ? (my_zero ? 1.f : 0.f) : expf(my_lw - lwmax);
            fit = fmaf(lam[lane], gcur, bia[lane]);
        }
        float wsum = 0.f, acc = 0.f;
        for (int c = 0; c < ncomp; ++c) {
            const float wc = __shfl(w, c, 64), fc = __shfl(fit, c, 64);
            wsum += wc;
            acc = fmaf(wc, fc, acc);
        }
        if (lane == 0) f_out[r] = acc / wsum;
#pragma unroll
        for (int i = 0; i < kGroups; ++i) cur[i] = nxt[i];
        gcur = gnxt;
    }
}

// ------------------------------------------------------------------ launch

// k_eval_wide for the wide evaluations that k_eval<64> would run.
static std::atomic<int> g_wide_eval{1};
static std::atomic<long long> g_wide_launches{0};
bool wide_eval_enabled() { return g_wide_eval.load(std::memory_order_relaxed) != 0; }

template <int RT, int PREC, EvalForm FORM>
static int launch_form(const EvalLaunch &p, int n, int nchunks, hipStream_t s) {
    static std::once_flag once;
    constexpr int lds = FORM == kEvalChunk ? gemm_lds_bytes<RT, PREC>() : eval_small_lds_bytes<RT, PREC>();
    std::call_once(once, [] {
        (void)hipFuncSetAttribute(reinterpret_cast<const void *>(&k_eval<RT, PREC, FORM>),
                                  hipFuncAttributeMaxDynamicSharedMemorySize, lds);
    });
    dim3 grid((n + RT - 1) / RT, nchunks);
    hipLaunchKernelGGL((k_eval<RT, PREC, FORM>), grid, dim3(256), lds, s, p);
    return check_launch("k_eval");
}

// (up to 128 columns: tiles of 16 and 32 rows, default_rows_per_block)
template <int RT, int PREC>
static int launch_rt_prec(const EvalLaunch &p, int n, int nchunks, hipStream_t s) {
    if constexpr (RT < 64)
        if (p.small) return launch_form<RT, PREC, kEvalSmall>(p, n, nchunks, s);
    return launch_form<RT, PREC, kEvalChunk>(p, n, nchunks, s);
}

template <int RT, int PREC>
static int launch_comps(const EvalComps &a, int ncomp, hipStream_t s) {
    static std::once_flag once;
    constexpr int lds = eval_small_lds_bytes<RT, PREC>();
    std::call_once(once, [] {
        (void)hipFuncSetAttribute(reinterpret_cast<const void *>(&k_eval_comps<RT, PREC>),
                                  hipFuncAttributeMaxDynamicSharedMemorySize, lds);
    });
    hipLaunchKernelGGL((k_eval_comps<RT, PREC>), dim3((a.p.n + RT - 1) / RT, ncomp), dim3(256), lds, s, a);
    return check_launch("k_eval_comps");
}

template <int RT>
static int launch_comps_rt(const EvalComps &a, int ncomp, int precision, hipStream_t s) {
    switch (precision) {
    case SPEO_PREC_FP32: return launch_comps<RT, SPEO_PREC_FP32>(a, ncomp, s);
    case SPEO_PREC_BF16: return launch_comps<RT, SPEO_PREC_BF16>(a, ncomp, s);
    case SPEO_PREC_FP16: return launch_comps<RT, SPEO_PREC_FP16>(a, ncomp, s);
    case SPEO_PREC_BF16X3: return launch_comps<RT, SPEO_PREC_BF16X3>(a, ncomp, s);
    case SPEO_PREC_FP16X3: return launch_comps<RT, SPEO_PREC_FP16X3>(a, ncomp, s);
    case SPEO_PREC_BF16X6: return launch_comps<RT, SPEO_PREC_BF16X6>(a, ncomp, s);
    default: return set_error(SPEO_ERR_ARG, "unknown precision mode");
    }
}

template <int RT>
static int launch_rt(const EvalLaunch &p, int precision, int n, int nchunks, hipStream_t s) {
    switch (precision) {
    case SPEO_PREC_FP32: return launch_rt_prec<RT, SPEO_PREC_FP32>(p, n, nchunks, s);
    case SPEO_PREC_BF16: return launch_rt_prec<RT, SPEO_PREC_BF16>(p, n, nchunks, s);
    case SPEO_PREC_FP16: return launch_rt_prec<RT, SPEO_PREC_FP16>(p, n, nchunks, s);
    case SPEO_PREC_BF16X3: return launch_rt_prec<RT, SPEO_PREC_BF16X3>(p, n, nchunks, s);
    case SPEO_PREC_FP16X3: return launch_rt_prec<RT, SPEO_PREC_FP16X3>(p, n, nchunks, s);
    case SPEO_PREC_BF16X6: return launch_rt_prec<RT, SPEO_PREC_BF16X6>(p, n, nchunks, s);
    default: return set_error(SPEO_ERR_ARG, "unknown precision mode");
    }
}

static bool use_wide(const CompDev &comp, const float *X, int ld, int n, int dim, int precision,
                     int rows_per_block) {
    return rows_per_block == 64 && wide_eval_enabled() &&
           eval_wide_applies(comp, X, ld, n, dim, precision);
}

int eval_component(const CompDev &comp, const float *X, int ld, int n, int dim, float *f_out,
                   float *part, float lambda, float bias, int raw, int precision,
                   int rows_per_block, hipStream_t s) {
    if (n <= 0) return SPEO_OK;
    const int nchunks = (dim + kNC - 1) / kNC;
    if (nchunks > 1 && part == nullptr) return set_error(SPEO_ERR_ARG, "eval: missing partial buffer");
    const int small = (dim <= kSmallD && comp.B32s != nullptr) ? 1 : 0;
    if (small && rows_per_block == 64)
        return set_error(SPEO_ERR_ARG, "up to 128 columns: 16 or 32 rows per block");
    EvalLaunch p{comp, X, ld, n, dim, f_out, part, nchunks, lambda, bias, raw, small};
    int rc;
    if (use_wide(comp, X, ld, n, dim, precision, rows_per_block)) {
        // the same bits as k_eval<64, precision>, on wider tiles
        rc = eval_wide(&comp, 1, X, ld, n, dim, part, precision, s);
        g_wide_launches.fetch_add(1, std::memory_order_relaxed);
    } else if (rows_per_block == 16 && precision == SPEO_PREC_FP32 && dim <= kSmallD && !small) {
        // the row-major matrix straight into registers; the 16-row tile's sums
        // are those of the staged path (four column classes in either)
        rc = launch_form<16, SPEO_PREC_FP32, kEvalRaw>(p, n, nchunks, s);
    } else switch (rows_per_block) {
    case 16: rc = launch_rt<16>(p, precision, n, nchunks, s); break;
    case 32: rc = launch_rt<32>(p, precision, n, nchunks, s); break;
    case 64: rc = launch_rt<64>(p, precision, n, nchunks, s); break;
    default: return set_error(SPEO_ERR_ARG, "rows_per_block must be 16, 32 or 64");
    }
    if (rc != SPEO_OK || nchunks == 1) return rc;
    hipLaunchKernelGGL(k_eval_finalize, dim3((n + 255) / 256), dim3(256), 0, s, part, nchunks, n, dim,
                       FinalizeObjectives{{comp.objective}}, lambda, bias, raw, f_out);
    return check_launch("k_eval_finalize");
}

// All components of a composition of up to 128 columns in one launch: three
// components of 100 rows, D = 30 were four dependent launches (19.7 us), two now
// (10.3 us).  Same bits: each component's blocks are k_eval's.
static int eval_components_small(const CompDev *comp, int ncomp, const float *X, int ld, int n, int dim,
                                 float *gbuf, int precision, int rows_per_block, hipStream_t s) {
    EvalComps a{};
    a.p = EvalLaunch{comp[0], X, ld, n, dim, gbuf, nullptr, 1, 1.f, 0.f, 1, 1};
    for (int c = 0; c < ncomp; ++c) a.comp[c] = comp[c];
    switch (rows_per_block) {
    case 16: return launch_comps_rt<16>(a, ncomp, precision, s);
    case 32: return launch_comps_rt<32>(a, ncomp, precision, s);
    default: return set_error(SPEO_ERR_ARG, "eval_components_small: 16 or 32 rows per block");
    }
}

// All components of a wide composition in one launch (no drain and refill of
// the chip between them), their chunk sums finalized in another.
static int eval_components_wide(const CompDev *comp, int ncomp, const float *X, int ld, int n, int dim,
                                float *gbuf, float *part, int precision, hipStream_t s) {
    SPEO_TRY(eval_wide(comp, ncomp, X, ld, n, dim, part, precision, s));
    g_wide_launches.fetch_add(ncomp, std::memory_order_relaxed);
    FinalizeObjectives o{};
    for (int c = 0; c < ncomp; ++c) o.obj[c] = comp[c].objective;
    hipLaunchKernelGGL(k_eval_finalize, dim3((n + 255) / 256, ncomp), dim3(256), 0, s, part,
                       (dim + kNC - 1) / kNC, n, dim, o, 1.f, 0.f, 1, gbuf);
    return check_launch("k_eval_finalize");
}

int eval_problem_generic(const ProblemHost &P, const float *X, int ld, int n, float *f32,
                         double *f64, const int *rows, int row_base, hipStream_t s) {
    GenLaunch g{};
    g.P = P.gen;
    g.dim = P.dim;
    g.ncomp = P.ncomp;
    g.X = X;
    g.ld = ld;
    g.n = n;
    g.rows = rows;
    g.row_base = row_base;
    g.f32 = f32;
    g.f64 = f64;
    return eval_generic(g, s);
}

size_t eval_scratch_floats(int ncomp, int dim, int n) {
    const int nchunks = (dim + kNC - 1) / kNC;
    size_t part = nchunks > 1 ? (size_t)nchunks * 2 * n : 0;
    size_t comp = ncomp > 1 ? (size_t)ncomp * n : 0;
    return part + comp;
}

size_t eval_scratch_batched(int ncomp, int dim, int n) {
    const int nchunks = (dim + kNC - 1) / kNC;
    if (ncomp == 1 || nchunks == 1) return eval_scratch_floats(ncomp, dim, n);
    return (size_t)ncomp * n * (2 * nchunks + 1);
}

// Rows copied to a stride of a multiple of four floats, the padding zero: a wave
// a row, consecutive lanes consecutive floats.
__global__ __launch_bounds__(256) void k_pack_rows(const float *X, int ld, int n, int dim, int ldp, float *out) {
    const int r = blockIdx.x * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63;
    if (r >= n) return;
    const float *x = X + (size_t)r * ld;
    float *o = out + (size_t)r * ldp;
#pragma unroll 4
    for (int j = lane; j < ldp; j += 64) o[j] = j < dim ? x[j] : 0.f;
}

size_t eval_pack_floats(const ProblemHost &P, const float *X, int ld, int n) {
    if (P.generic || P.dim <= kSmallD || n <= 0) return 0;
    if ((ld & 3) == 0 && (reinterpret_cast<uintptr_t>(X) & 15) == 0) return 0;
    const size_t floats = (size_t)n * round_up(P.dim, 4);
    return floats <= (size_t(1) << 28) ? floats : 0;
}

int eval_problem(const ProblemHost &P, const float *X, int ld, int n, float *f_out, float *scratch,
                 size_t scratch_floats, float *packed, int precision, int rows_per_block, hipStream_t s) {
    if (n <= 0) return SPEO_OK;
    if (P.generic) return eval_problem_generic(P, X, ld, n, f_out, nullptr, nullptr, 0, s);
    const int nchunks = (P.dim + kNC - 1) / kNC;
    // Rows that 16-byte accesses cannot take (an odd stride, as torch's rows of
    // an odd dimension have) are copied once where there is room: staged element by
    // element they kept the tile kernels out altogether (16,172 rows of D = 991 in
    // BF16: 702 us, 73 us with the copy; 64 rows of D = 131 19 and 10 us; same
    // bits).  The combination below reads the caller's rows, as its sums' order
    // depends on the alignment.
    const float *Xc = X;
    const int ldc = ld;
    if (packed) {
        const int ldp = round_up(P.dim, 4);
        hipLaunchKernelGGL(k_pack_rows, dim3((n + 3) / 4), dim3(256), 0, s, X, ld, n, P.dim, ldp, packed);
        SPEO_TRY(check_launch("k_pack_rows"));
        X = packed;
        ld = ldp;
    }
    float *part = nchunks > 1 ? scratch : nullptr;
    float *gbuf = scratch + (nchunks > 1 ? (size_t)nchunks * 2 * n : 0);
    // an unrotated component's z = (x - o) rate is exact in FP32; a 16-bit
    // identity GEMM would round it to the operand precision
    auto prec_of = [&](int c) { return P.comp[c].unrotated ? (int)SPEO_PREC_FP32 : precision; };
    if (P.ncomp == 1) {
        const CompHost &c = P.comp[0];
        return eval_component(P.view(0, prec_of(0)), X, ld, n, P.dim, f_out, part,
                              (float)c.lambda, (float)c.bias, 0, prec_of(0), rows_per_block, s);
    }
    CompDev view[kMaxComp];
    bool batched = nchunks > 1 && scratch_floats >= eval_scratch_batched(P.ncomp, P.dim, n);
    bool small = nchunks == 1;
    for (int c = 0; c < P.ncomp; ++c) {
        view[c] = P.view(c, prec_of(c));
        small = small && prec_of(c) == prec_of(0) && view[c].B32s != nullptr;
        batched = batched && prec_of(c) == prec_of(0) &&
                  use_wide(view[c], X, ld, n, P.dim, prec_of(c), rows_per_block);
    }
    if (batched) {
        gbuf = scratch + (size_t)P.ncomp * nchunks * 2 * n;
        SPEO_TRY(eval_components_wide(view, P.ncomp, X, ld, n, P.dim, gbuf, scratch, prec_of(0), s));
    }
    if (small)
        SPEO_TRY(eval_components_small(view, P.ncomp, X, ld, n, P.dim, gbuf, prec_of(0), rows_per_block, s));
    for (int c = 0; c < P.ncomp && !batched && !small; ++c)
        SPEO_TRY(eval_component(view[c], X, ld, n, P.dim, gbuf + (size_t)c * n, part,
                                1.f, 0.f, 1, prec_of(c), rows_per_block, s));
    bool rows = (P.dim & 3) == 0 && P.dim <= 1024 && (ldc & 3) == 0 &&
                (reinterpret_cast<uintptr_t>(Xc) & 15) == 0 && n >= 4096;
    for (int c = 0; c < P.ncomp; ++c) rows = rows && (reinterpret_cast<uintptr_t>(P.comp[c].shift32) & 15) == 0;
    if (rows) {
        hipLaunchKernelGGL(k_comp_combine_rows, dim3((n + 4 * kCombRows - 1) / (4 * kCombRows)), dim3(256),
                           sizeof(float) * (size_t)P.ncomp * P.dim, s, P.params_dev, P.ncomp, P.dim, Xc, ldc,
                           n, gbuf, f_out);
        return check_launch("k_comp_combine_rows");
    }
    const int waves_per_block = 4;
    hipLaunchKernelGGL(k_comp_combine, dim3((n + waves_per_block - 1) / waves_per_block),
                       dim3(64 * waves_per_block), 0, s, P.params_dev, P.ncomp, P.dim, Xc, ldc, n,
                       gbuf, f_out);
    return check_launch("k_comp_combine");
}

int eval_problem_f64(const ProblemHost &P, const float *X, int ld, int n, double *f_out,
                     hipStream_t s) {
    if (n <= 0) return SPEO_OK;
    if (P.gen) return eval_problem_generic(P, X, ld, n, nullptr, f_out, nullptr, 0, s);
    return eval_rows_f64(P.params_dev, P.ncomp, P.dim, X, ld, n, f_out, s);
}

int default_rows_per_block(int n, int dim, int precision, bool kept) {
    // Up to 128 columns from a problem's layouts the tile changes no result: 32
    // rows once they give a block a compute unit (Rastrigin, us at 16 / 32 / 64
    // rows: 4,096 x 100 FP32 5.3 / 6.5 / 9.8, 65,536 x 100 BF16 19.5 / 15.6 /
    // 17.3, 65,536 x 128 FP32 29.7 / 29.7 / 31.0).
    if (kept && dim <= kSmallD) return (n + 31) / 32 >= 256 ? 32 : 16;
    // Enough blocks to cover the 256 CUs; larger tiles share B staging.
    const int nchunks = (dim + kNC - 1) / kNC;
    // 16-bit evaluations wider than one chunk: 64-row arithmetic from 1024
    // rows on, which k_eval_wide runs on its own wider tiles
    if (precision != SPEO_PREC_FP32 && nchunks > 1 && n >= 1024) return 64;
    if ((long)((n + 63) / 64) * nchunks >= 512) return 64;
    if ((long)((n + 31) / 32) * nchunks >= 256) return 32;
    return 16;
}

// ------------------------------------------------- drop-in API_evaluateFitness

namespace {
struct DimTables {
    float *colw[3] = {nullptr, nullptr, nullptr};  // elliptic, bent cigar, discus weights
    float *identity = nullptr;
    int heavy_j[3] = {-1, -1, -1};  // their heavy columns
    double heavy_w[3] = {0.0, 0.0, 0.0};
};
std::mutex g_tables_mu;
std::unordered_map<int, DimTables> g_tables;

int dim_tables(int dim, DimTables &out) {
    std::lock_guard<std::mutex> lk(g_tables_mu);
    auto it = g_tables.find(dim);
    if (it != g_tables.end()) {
        out = it->second;
        return SPEO_OK;
    }
    DimTables t;
    std::vector<float> w((size_t)dim), I((size_t)dim * dim, 0.f);
    for (int j = 0; j < dim; ++j) I[(size_t)j * dim + j] = 1.f;
    const int kinds[3] = {SPEO_OBJ_ELLIPTIC, SPEO_OBJ_BENT_CIGAR, SPEO_OBJ_DISCUS};
    for (int k = 0; k < 3; ++k) {
        column_weights(kinds[k], dim, w.data());
        t.heavy_j[k] = heavy_column(kinds[k], dim, &t.heavy_w[k]);
        SPEO_TRY_HIP(hipMalloc(&t.colw[k], sizeof(float) * dim));
        SPEO_TRY_HIP(hipMemcpy(t.colw[k], w.data(), sizeof(float) * dim, hipMemcpyHostToDevice));
    }
    SPEO_TRY_HIP(hipMalloc(&t.identity, sizeof(float) * dim * dim));
    SPEO_TRY_HIP(hipMemcpy(t.identity, I.data(), sizeof(float) * dim * dim, hipMemcpyHostToDevice));
    g_tables[dim] = t;
    out = t;
    return SPEO_OK;
}
}  // namespace

// The reference's CEC2014_CUDA (CEC2014_CUDA.cc:68-128, 160-289) hands every
// call its device buffers: d_shift_data [ncomp][next_pow2(dim)],
// d_rotated_data [ncomp][next_pow2(dim)][dim] (B = M^T, row-padded),
// d_shuffle_data [ncomp][next_pow2(dim)] (1-based), d_sigma [ncomp] and the
// scratch rows d_rotated_elements [pop_size][next_pow2(dim)].
//
// The device description of function `fid` at `dim` (objectives, segments,
// rates and composition parameters; the arrays come with each call), built at
// the first call that needs it on a device and kept, as the dimension's tables
// are: at most 30 of 2 KB per dimension.
static int dropin_problem(int fid, int dim, const GenProblem **out, int *ncomp) {
    static std::mutex mu;
    static std::map<std::tuple<int, int, int>, std::pair<GenProblem *, int>> table;
    int dev = 0;
    SPEO_TRY_HIP(hipGetDevice(&dev));
    std::lock_guard<std::mutex> lk(mu);
    auto &e = table[std::make_tuple(dev, fid, dim)];
    if (!e.first) {
        int nc = 0;
        CecComp cc[kMaxComp];
        if (!cec_function(fid, &nc, cc)) return set_error(SPEO_ERR_UNSUPPORTED, "unknown function");
        GenProblem g{};
        g.dim = dim;
        g.ncomp = nc;
        for (int c = 0; c < nc; ++c) {
            GenComp &G = g.comp[c];
            if (cc[c].objective >= SPEO_OBJ_HYBRID_1) {
                hybrid_segments(cc[c].objective, dim, G);
            } else {
                G.nseg = 1;
                G.seg[0] = gen_seg(cc[c].objective, dim, 1.0);
            }
            G.rate = cc[c].rate;
            G.rotate = cc[c].rotate;
            G.lambda = cc[c].lambda;
            G.bias = cc[c].bias;
            G.sigma = cc[c].sigma;
        }
        SPEO_TRY(check_gen_problem(g, true));
        GenProblem *d = nullptr;
        SPEO_TRY_HIP(hipMalloc(reinterpret_cast<void **>(&d), sizeof(g)));
        SPEO_TRY_HIP(hipMemcpy(d, &g, sizeof(g), hipMemcpyHostToDevice));
        e = {d, nc};
    }
    *out = e.first;
    *ncomp = e.second;
    return SPEO_OK;
}

static int dropin_generic(real *f, real *X, real *shift, real *B, int *shuffle, real *sigma,
                          int n, int dim, real bias, int fid) {
    int nc = 0;
    CecComp cc[kMaxComp];
    if (!cec_function(fid, &nc, cc)) return set_error(SPEO_ERR_UNSUPPORTED, "unknown function");
    if (dim > kGenMaxDim)
        return set_error(SPEO_ERR_UNSUPPORTED, "generic evaluation: dim must be in [1, 1024]");
    bool hybrid = false;
    for (int c = 0; c < nc; ++c) {
        hybrid = hybrid || cc[c].objective >= SPEO_OBJ_HYBRID_1;
        if (cc[c].rotate && !B) return set_error(SPEO_ERR_ARG, "missing rotation matrix");
    }
    if (hybrid && !shuffle) return set_error(SPEO_ERR_ARG, "missing shuffle data");
    GenLaunch g{};
    SPEO_TRY(dropin_problem(fid, dim, &g.P, &g.ncomp));
    g.dim = dim;
    g.X = X;
    g.ld = next_pow2_dim(dim);
    g.n = n;
    g.f32 = f;
    // F1-F16 ignore the call's bias; the hybrid and composition chains add it
    // in CombineFitness (kernel_CEC2014_CUDA.cu:205, 1227, 1447).
    g.out_bias = fid >= 17 ? bias : 0.0;
    g.o32 = shift;
    g.B32 = B;
    g.sigma32 = sigma;
    g.perm = hybrid ? shuffle : nullptr;
    g.stride = g.ld;
    return eval_generic(g, nullptr);
}

}  // namespace speo

using namespace speo;

extern "C" int speo_wide_eval(int enable, long long *launches) {
    if (launches) *launches = g_wide_launches.load();
    return enable < 0 ? g_wide_eval.load() : g_wide_eval.exchange(enable ? 1 : 0);
}

extern "C" void API_evaluateFitness(real *d_fitness_value, real *, real *d_rotated_elements,
                                    real *d_original_elements, real *d_shift_data,
                                    real *d_rotated_data, int *d_shuffle_data, real *,
                                    real *, real *d_sigma, int pop_size, int problem_dim,
                                    real bias, int function_ID) {
    if (pop_size <= 0 || problem_dim < 2 || !d_fitness_value || !d_original_elements ||
        !d_shift_data) {
        defer_error(SPEO_ERR_ARG, "API_evaluateFitness: invalid arguments");
        return;
    }
    if (function_ID < 1 || function_ID > 30) {
        defer_error(SPEO_ERR_UNSUPPORTED, "API_evaluateFitness: function_ID " +
                                              std::to_string(function_ID) + " is not in 1..30");
        return;
    }
    CompDev c{};
    bool rotate = true;
    int weights = 0;  // DimTables::colw entry of the weighted-sphere objectives
    switch (function_ID) {
    case 1: c.objective = SPEO_OBJ_ELLIPTIC; c.rate = 1.0f; break;       // F1, kernel_CEC2014_CUDA.cu:1105
    // F2 bent cigar and F3 discus (:1111, :1117; global_f2 / global_f3 at
    // :287-352): the weighted sphere with their own column weights.
    case 2: c.objective = SPEO_OBJ_ELLIPTIC; c.rate = 1.0f; weights = 1; break;
    case 3: c.objective = SPEO_OBJ_ELLIPTIC; c.rate = 1.0f; weights = 2; break;
    case 5: c.objective = SPEO_OBJ_ACKLEY; c.rate = 1.0f; break;         // F5, :1130
    case 8: c.objective = SPEO_OBJ_RASTRIGIN; c.rate = 0.0512f; rotate = false; break;  // F8, :1150
    case 9: c.objective = SPEO_OBJ_RASTRIGIN; c.rate = 0.0512f; break;   // F9, :1156
    case 10: c.objective = SPEO_OBJ_SCHWEFEL; c.rate = 10.0f; rotate = false; break;  // F10, :1162
    case 11: c.objective = SPEO_OBJ_SCHWEFEL; c.rate = 10.0f; break;     // F11, :1168
    case 13: c.objective = SPEO_OBJ_HAPPYCAT; c.rate = 0.05f; break;     // F13, :1180
    case 14: c.objective = SPEO_OBJ_HGBAT; c.rate = 0.05f; break;        // F14, :1186
    default: {
        // F4, F6, F7, F12, F15, F16, the hybrids F17-F22 and the compositions
        // F23-F30 (:1123-1671): the FP64 generic kernel.
        const int rc = dropin_generic(d_fitness_value, d_original_elements, d_shift_data,
                                      d_rotated_data, d_shuffle_data, d_sigma, pop_size,
                                      problem_dim, bias, function_ID);
        if (rc != SPEO_OK) defer_error(rc, std::string("API_evaluateFitness: ") + speo_last_error());
        return;
    }
    }
    if (rotate && !d_rotated_data) {
        defer_error(SPEO_ERR_ARG, "API_evaluateFitness: missing rotation matrix");
        return;
    }
    DimTables t;
    if (dim_tables(problem_dim, t) != SPEO_OK) {
        defer_error(SPEO_ERR_HIP, "API_evaluateFitness: table allocation failed");
        return;
    }
    c.shift = d_shift_data;
    c.B32 = rotate ? d_rotated_data : t.identity;
    c.ldb32 = problem_dim;  // reference layout [next_pow2(dim)][dim] (CEC2014_CUDA.cc:255)
    c.colw = t.colw[weights];
    c.heavy.j = -1;
    if (c.objective == SPEO_OBJ_ELLIPTIC) {
        c.heavy.j = t.heavy_j[weights];
        c.heavy.w = t.heavy_w[weights];
        c.heavy.m32 = c.B32 + (c.heavy.j >= 0 ? c.heavy.j : 0);  // column j of B = row j of M
        c.heavy.ld = problem_dim;
        c.heavy.o32 = d_shift_data;
        c.heavy.rate = 1.0;
    }
    const int ld = next_pow2_dim(problem_dim);
    // Above 128 columns the per-chunk row sums go to the caller's rotated-row
    // buffer (pop_size * next_pow2(dim) floats, at least 2 * chunks * pop_size).
    float *part = nullptr;
    if (problem_dim > kNC) {
        if (!d_rotated_elements) {
            defer_error(SPEO_ERR_ARG, "API_evaluateFitness: dim > 128 needs d_rotated_elements");
            return;
        }
        part = d_rotated_elements;
    }
    const int rc = eval_component(c, d_original_elements, ld, pop_size, problem_dim,
                                  d_fitness_value, part, 1.f, 0.f, 0, SPEO_PREC_FP32,
                                  default_rows_per_block(pop_size, problem_dim, SPEO_PREC_FP32, false),
                                  nullptr);
    if (rc != SPEO_OK) defer_error(rc, speo_last_error());
}

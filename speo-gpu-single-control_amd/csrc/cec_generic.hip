// cec_generic.hip -- FP64 evaluation of the CEC2014 objectives that the fused
// FP32 epilogues do not take (see cec_generic.h).
//
// Reference counterparts: the basic kernels global_f4, f6, f7, f10, f13, f14
// (kernel_CEC2014_CUDA.cu:355-387, 443-556, 649-701, 809-976), the hybrid
// chains HybirdFunc1-6 (:1204-1415: ShiftAndRotation, Shuffle, one kernel per
// segment, CombineFitness) and the compositions CompFunc1-8 (:1416-1671:
// ShiftAndRotation per component, CalW, CombineFitness).  The arithmetic
// follows the reference's FP64 CPU forms (CEC2014.cc:481-1519), which define
// the values; here one launch does all of it for a tile of 16 rows.
#include <algorithm>
#include <cmath>
#include <mutex>

#include "cec_generic.h"
#include "eval_f64.h"

namespace speo {

typedef double doublex4 __attribute__((ext_vector_type(4)));
typedef double doublex2 __attribute__((ext_vector_type(2)));

namespace {

__device__ __forceinline__ double wave_prod(double v) {
    for (int off = 32; off > 0; off >>= 1) v *= __shfl_xor(v, off, 64);
    return v;
}

// Coordinate i of a segment: rate * z[j], j = start + i, through the shuffle
// (1-based, as the reference's global_Shuffle reads it, kernel_CEC2014_CUDA.cu:144).
struct Seg {
    const double *z;
    const int *perm;
    int start, len;
    double rate, par;
    __device__ __forceinline__ double y(int i) const {
        int j = start + i;
        if (perm) j = gld(perm + j) - 1;
        return rate * z[j];
    }
};

__device__ __forceinline__ double grie_of_rosen(double a, double b) {
    const double t1 = a * a - b, t2 = a - 1.0;
    const double t = 100.0 * t1 * t1 + t2 * t2;
    return (t * t) / 4000.0 - cos64(t) + 1.0;
}

__device__ __forceinline__ double scaffer6(double r2) {
    double t1 = sin64(sqrt(r2));
    t1 = t1 * t1;
    const double t2 = 1.0 + 0.001 * r2;
    return 0.5 + (t1 - 0.5) / (t2 * t2);
}

// The objective of one segment (FP64, CEC2014.cc forms), every lane of the
// wave taking coordinates lane, lane + 64, ...; the wave's value is
// returned on every lane.
__device__ __forceinline__ double seg_value(int obj, const Seg &s, int lane) {
    const int n = s.len;
    double a = 0.0, b = 0.0;
    switch (obj) {
    case SPEO_OBJ_ROSENBROCK:  // :552-568, fixed shift 1
        for (int i = lane; i < n - 1; i += 64) {
            const double y0 = s.y(i) + 1.0, y1 = s.y(i + 1) + 1.0;
            const double t1 = y0 * y0 - y1, t2 = y0 - 1.0;
            a += 100.0 * t1 * t1 + t2 * t2;
        }
        return wave_sum64(a);
    case SPEO_OBJ_WEIERSTRASS: {  // :615-644, a = 0.5, b = 3, k_max = 20
        // a^k and b^k as running products: 2^-k and 3^k (< 2^53) are exact in
        // FP64, so these are the values pow(a, k), pow(b, k) return
        for (int i = lane; i < n; i += 64) {
            const double y = s.y(i);
            double t = 0.0, ak = 1.0, bk = 1.0;
#pragma unroll 3
            for (int k = 0; k <= 20; ++k, ak *= 0.5, bk *= 3.0) t += ak * cos64(2.0 * kPi64 * bk * (y + 0.5));
            a += t;
        }
        // the constant at y = 0: sum_k 2^-k cos(3^k pi) = -(2 - 2^-20)
        return wave_sum64(a) + n * (2.0 - 0x1p-20);
    }
    case SPEO_OBJ_GRIEWANK: {  // :646-666
        double p = 1.0;
        for (int i = lane; i < n; i += 64) {
            const double y = s.y(i);
            a += y * y;
            p *= cos64(y / sqrt(1.0 + i));
        }
        return 1.0 + wave_sum64(a) / 4000.0 - wave_prod(p);
    }
    case SPEO_OBJ_KATSUURA: {  // :739-765
        // |v - floor(v + 1/2)| and |v - rint(v)| differ at halves only, where
        // both are 1/2; 2^j and its inverse as running products are exact.
        // A lane's factors are multiplied before their common power
        // par = 10 / n^1.2 is taken (at most 16 of them, each <= 1 + n / 2: no
        // overflow).
        double p = 1.0;
        for (int i = lane; i < n; i += 64) {
            const double y = s.y(i);
            double t = 0.0, sc = 2.0, inv = 0.5;
#pragma unroll 4
            for (int j = 1; j <= 32; ++j, sc *= 2.0, inv *= 0.5) {
                const double v = sc * y;
                t = fma(fabs(v - rint(v)), inv, t);
            }
            p *= 1.0 + (i + 1) * t;
        }
        const double c = 10.0 / n / n;
        return wave_prod(exp(s.par * log(p))) * c - c;
    }
    case SPEO_OBJ_GRIE_ROSEN:  // :842-868, fixed shift 1, wrap-around pair
        for (int i = lane; i < n; i += 64)
            a += grie_of_rosen(s.y(i) + 1.0, s.y(i + 1 < n ? i + 1 : 0) + 1.0);
        return wave_sum64(a);
    case SPEO_OBJ_ESCAFFER6:  // :870-905, wrap-around pair; one coordinate alone
        if (n == 1) {
            const double y = s.y(0);
            return scaffer6(y * y);
        }
        for (int i = lane; i < n; i += 64) {
            const double y0 = s.y(i), y1 = s.y(i + 1 < n ? i + 1 : 0);
            a += scaffer6(y0 * y0 + y1 * y1);
        }
        return wave_sum64(a);
    default:  // the objectives of two coordinate sums (1..8)
        if (obj < SPEO_OBJ_ELLIPTIC || obj > SPEO_OBJ_SCHWEFEL) return __builtin_nan("");
        for (int i = lane; i < n; i += 64) add_terms64(obj, i, n, s.y(i), a, b);
        return finish_objective64(obj, wave_sum64(a), wave_sum64(b), n);
    }
}

}  // namespace

// LDS: 16 rows of round_up(dim, 8) + 2 doubles, the shifted rows and then z in
// the same place, and each row's component values.  (The stride is 4 banks past
// a multiple of 16, so the 16 rows of a 16-byte operand read start in different
// banks.)
static int generic_ld(int dim) { return round_up(dim, 8) + 2; }
static size_t generic_lds_bytes(int dim) { return sizeof(double) * (size_t)kGenRows * (generic_ld(dim) + 2 * kMaxComp); }

// A block takes up to 16 rows (generic_block_rows), a wave each, through every
// component: wave r shifts row r into LDS (and sums its squared distance), the
// waves share the 16-column tiles of z (a wave each, up to sixteen waves; NQ per
// wave, dim <= 256 NQ) on v_mfma_f64_16x16x4f64 with the accumulators in
// registers, z replaces the rows in LDS, and wave r evaluates row r.  K runs in steps of 8 as two MFMA steps whose lanes take
// k = 8 s + 2 lk and + 1, so that a lane's part of M is one 16-byte load; four
// of them are in flight before the first is used.
//
// What bounds it: at D = 100 the objective phase (FP64 vector work, one row
// per wave) and the latency of the phases, at D >= 250 the FP64 matrix pipe (64
// cycles per step of 4).  Measured, FP64 values of 2048 rows x 250, three
// components: 770 us with a block per row (M read again for every row), 39 us
// here; a five-component CEC2014 composition on 4096 rows x 100: 164 us with
// four waves per block (four rows per wave one after another, 8-byte strided
// loads of M, library cosines), 41 us here.  Up to 256 columns two blocks fit a
// compute unit (64 registers); spilled registers cost more than the occupancy
// gives (15 us per component and block at 128 registers with 40 spilled).
template <int NQ, bool ARRAYS>
__global__ __launch_bounds__(kGenThreads) __attribute__((amdgpu_waves_per_eu(NQ == 1 && !ARRAYS ? 8 : 4))) void k_eval_generic(GenLaunch p) {
    extern __shared__ __align__(16) char lds_raw[];
    const int dim = p.dim, nc = p.ncomp;
    const int ld = round_up(dim, 8) + 2;
    double *As = reinterpret_cast<double *>(lds_raw);
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int nw = blockDim.x >> 6, lr = lane & 15, lk = lane >> 4;
    const int row = blockIdx.x * p.block_rows + wave;  // this wave's row
    const bool mine = wave < p.block_rows && row < p.n;
    const float *x = p.X;
    if (mine) x += (size_t)(p.rows ? p.rows[row] - p.row_base : row) * p.ld;
    double *z = As + wave * ld;
    const int T = (dim + 15) >> 4;

    double *part = As + kGenRows * ld + wave * 2 * kMaxComp;  // per component: fit, squared distance
    for (int ci = 0; ci < nc; ++ci) {
        const GenComp &C = p.P->comp[ci];
        const float *o32 = p.o32 + (size_t)ci * p.stride, *B32 = p.B32 + (size_t)ci * p.stride * dim;
        const int *perm = ARRAYS ? (p.perm ? p.perm + (size_t)ci * p.stride : nullptr) : C.perm;
        const double rate = C.rate;
        double d = 0.0;
        if (mine) {
            for (int k = lane; k < round_up(dim, 8); k += 64) {
                double v = 0.0;
                if (k < dim) v = (double)gld(x + k) - (ARRAYS ? (double)gld(o32 + k) : gld(C.o64 + k));
                z[k] = v * rate;
                d = fma(v, v, d);
            }
        }
        if (C.rotate) {
            __syncthreads();
            doublex4 acc[NQ];
#pragma unroll
            for (int q = 0; q < NQ; ++q) {
                acc[q] = doublex4{0.0, 0.0, 0.0, 0.0};
                __builtin_amdgcn_sched_barrier(0);
                const int t = wave + nw * q;
                if (t >= T) continue;
                const double *a = As + lr * ld + 2 * lk;
                const int steps = ARRAYS ? dim >> 3 : (dim + 7) >> 3;
                const int col = min(16 * t + lr, dim - 1);  // (columns past the last are not stored)
                const double *m = C.M64f + ((size_t)t * ((dim + 7) >> 3) * 64 + lane) * 2;
                const float *bc = B32 + col;
                auto load = [&](int s) __attribute__((always_inline)) {
                    if constexpr (ARRAYS) {
                        const float *q0 = bc + (size_t)(8 * s + 2 * lk) * dim;
                        return doublex2{(double)gld(q0), (double)gld(q0 + dim)};
                    } else {
                        return gld(reinterpret_cast<const doublex2 *>(m + (size_t)s * 128));
                    }
                };
                auto step = [&](int s, doublex2 b) __attribute__((always_inline)) {
                    const doublex2 av = *reinterpret_cast<const doublex2 *>(a + 8 * s);
                    acc[q] = __builtin_amdgcn_mfma_f64_16x16x4f64(av.x, b.x, acc[q], 0, 0, 0);
                    acc[q] = __builtin_amdgcn_mfma_f64_16x16x4f64(av.y, b.y, acc[q], 0, 0, 0);
                };
                constexpr int NB = 4;
                int s = 0;
                for (; s + NB <= steps; s += NB) {
                    doublex2 b[NB];
#pragma unroll
                    for (int u = 0; u < NB; ++u) b[u] = load(s + u);
#pragma unroll
                    for (int u = 0; u < NB; ++u) step(s + u, b[u]);
                }
                for (; s < steps; ++s) step(s, load(s));
                if (ARRAYS && (dim & 7)) {  // the caller's M^T ends inside the step (the rows in LDS are zero there)
                    const int k = 8 * s + 2 * lk;
                    doublex2 b = {0.0, 0.0};
                    if (k < dim) b.x = (double)gld(bc + (size_t)k * dim);
                    if (k + 1 < dim) b.y = (double)gld(bc + (size_t)(k + 1) * dim);
                    step(s, b);
                }
            }
            __syncthreads();
            // accumulator element i of lane l of v_mfma_f64_16x16x4f64: row
            // l / 16 + 4 i, column l % 16
#pragma unroll
            for (int q = 0; q < NQ; ++q) {
                const int col = 16 * (wave + nw * q) + lr;
                if (col < dim)
#pragma unroll
                    for (int i = 0; i < 4; ++i) As[(lk + 4 * i) * ld + col] = acc[q][i];
            }
            __syncthreads();
        }
        if (!mine) continue;
        // (from here to the next component's shift a wave touches its own row only)
        double g = 0.0;
        int start = 0;
        for (int s = 0; s < C.nseg; ++s) {
            const Seg sv{z, perm, start, C.seg[s].len, C.seg[s].rate, C.seg[s].par};
            g += seg_value(C.seg[s].obj, sv, lane);
            start += C.seg[s].len;
        }
        d = wave_sum64(d);
        if (lane == 0) {
            part[2 * ci] = C.lambda * g + C.bias;
            part[2 * ci + 1] = d;
        }
    }
    if (!mine) return;
    double f;
    if (nc == 1) {
        f = part[0];
    } else {
        const int c = min(lane, nc - 1);
        f = combine64(nc, dim, part[2 * c], part[2 * c + 1],
                      p.sigma32 ? (double)p.sigma32[c] : p.P->comp[c].sigma, lane);
    }
    f += p.out_bias;
    if (lane == 0) {
        if (p.f32) p.f32[row] = (float)f;
        if (p.f64) p.f64[row] = f;
    }
}

__global__ void k_gen_fragments(const double *M64, int dim, double *out) {
    const int t = blockIdx.x, S = (dim + 7) >> 3;
    for (int e = threadIdx.x; e < S * 128; e += blockDim.x) {
        const int s = e >> 7, l = (e >> 1) & 63;
        const int col = 16 * t + (l & 15), k = 8 * s + 2 * (l >> 4) + (e & 1);
        out[(size_t)t * S * 128 + e] = col < dim && k < dim ? M64[(size_t)col * dim + k] : 0.0;
    }
}

int gen_fragments(const double *M64, int dim, double *out, hipStream_t s) {
    hipLaunchKernelGGL(k_gen_fragments, dim3((dim + 15) / 16), dim3(256), 0, s, M64, dim, out);
    return check_launch("k_gen_fragments");
}

template <int NQ, bool ARRAYS>
static int launch_generic(const GenLaunch &p, hipStream_t s) {
    static_assert(NQ == 1 || 256 * NQ == kGenMaxDim, "column tiles of a wave");
    static std::once_flag once;
    std::call_once(once, [] {
        (void)hipFuncSetAttribute(reinterpret_cast<const void *>(&k_eval_generic<NQ, ARRAYS>),
                                  hipFuncAttributeMaxDynamicSharedMemorySize,
                                  (int)generic_lds_bytes(256 * NQ));
    });
    const dim3 grid((p.n + p.block_rows - 1) / p.block_rows);
    // a wave per row and, up to sixteen, per column tile
    const int waves = std::min(kGenRows, std::max(p.block_rows, (p.dim + 15) / 16));
    hipLaunchKernelGGL((k_eval_generic<NQ, ARRAYS>), grid, dim3(64 * waves), generic_lds_bytes(p.dim), s, p);
    return check_launch("k_eval_generic");
}

int check_gen_problem(const GenProblem &g, bool arrays) {
    if (g.dim < 1 || g.dim > kGenMaxDim || g.ncomp < 1 || g.ncomp > kMaxComp)
        return set_error(SPEO_ERR_UNSUPPORTED, "generic evaluation: dim must be in [1, 1024]");
    for (int c = 0; c < g.ncomp; ++c) {
        const GenComp &C = g.comp[c];
        int total = 0;
        for (int q = 0; q < C.nseg; ++q) total += C.seg[q].len;
        if (C.nseg < 1 || C.nseg > kGenMaxSeg || total != g.dim)
            return set_error(SPEO_ERR_ARG, "generic evaluation: segments do not cover the dimension");
        if (!arrays && !C.o64) return set_error(SPEO_ERR_ARG, "generic evaluation: missing shift");
        if (!arrays && C.rotate && !C.M64f)
            return set_error(SPEO_ERR_ARG, "generic evaluation: missing rotation");
    }
    return SPEO_OK;
}

// Rows a block: as few as give no more than a block a compute unit.  A row's
// objective is its wave's FP64 work, and sixteen rows on one unit while others had
// none took longer than a block per row had (us, a block of four waves per row /
// sixteen rows a block / now: 300 rows of D = 2, three components 9.7 / 13.3 / 8.9,
// five 14.3 / 19.9 / 13.2; 2,048 of D = 250, three 689 / 42.0 / 38.8).  No result
// depends on it.
static int generic_block_rows(int n) {
    constexpr int kUnits = 256;
    int rows = 1;
    while (rows < kGenRows && (n + rows - 1) / rows > kUnits) rows *= 2;
    return rows;
}

int eval_generic(const GenLaunch &launch, hipStream_t s) {
    GenLaunch p = launch;
    if (p.n <= 0) return SPEO_OK;
    if (!p.P || p.dim < 1 || p.dim > kGenMaxDim || p.ncomp < 1 || p.ncomp > kMaxComp)
        return set_error(SPEO_ERR_UNSUPPORTED, "generic evaluation: dim must be in [1, 1024]");
    p.block_rows = generic_block_rows(p.n);
    if (p.o32) return p.dim <= 256 ? launch_generic<1, true>(p, s) : launch_generic<4, true>(p, s);
    return p.dim <= 256 ? launch_generic<1, false>(p, s) : launch_generic<4, false>(p, s);
}

// ------------------------------------------------------- function tables

GenSeg gen_seg(int objective, int len, double rate) {
    return GenSeg{objective, len, rate, objective == SPEO_OBJ_KATSUURA ? 10.0 / std::pow((double)len, 1.2) : 0.0};
}

bool generic_objective(int objective) {
    return objective > SPEO_OBJ_SCHWEFEL;
}

bool hybrid_segments(int objective, int dim, GenComp &c) {
    struct Def {
        int nseg;
        double p[kGenMaxSeg];
        int obj[kGenMaxSeg];
        double rate[kGenMaxSeg];
    };
    // hf01-hf06, CEC2014.cc:954-1207 (the GPU chains HybirdFunc1-6,
    // kernel_CEC2014_CUDA.cu:1204-1415, use the same objectives and rates)
    static const Def defs[6] = {
        {3, {0.3, 0.3, 0.4}, {SPEO_OBJ_SCHWEFEL, SPEO_OBJ_RASTRIGIN, SPEO_OBJ_ELLIPTIC},
         {1000.0 / 100.0, 5.12 / 100.0, 1.0}},
        {3, {0.3, 0.3, 0.4}, {SPEO_OBJ_BENT_CIGAR, SPEO_OBJ_HGBAT, SPEO_OBJ_RASTRIGIN},
         {1.0, 5.0 / 100.0, 5.12 / 100.0}},
        {4, {0.2, 0.2, 0.3, 0.3},
         {SPEO_OBJ_GRIEWANK, SPEO_OBJ_WEIERSTRASS, SPEO_OBJ_ROSENBROCK, SPEO_OBJ_ESCAFFER6},
         {600.0 / 100.0, 0.5 / 100.0, 2.048 / 100.0, 1.0}},
        {4, {0.2, 0.2, 0.3, 0.3},
         {SPEO_OBJ_HGBAT, SPEO_OBJ_DISCUS, SPEO_OBJ_GRIE_ROSEN, SPEO_OBJ_RASTRIGIN},
         {5.0 / 100.0, 1.0, 5.0 / 100.0, 5.12 / 100.0}},
        {5, {0.1, 0.2, 0.2, 0.2, 0.3},
         {SPEO_OBJ_ESCAFFER6, SPEO_OBJ_HGBAT, SPEO_OBJ_ROSENBROCK, SPEO_OBJ_SCHWEFEL, SPEO_OBJ_ELLIPTIC},
         {1.0, 5.0 / 100.0, 2.048 / 100.0, 1000.0 / 100.0, 1.0}},
        {5, {0.1, 0.2, 0.2, 0.2, 0.2},
         {SPEO_OBJ_KATSUURA, SPEO_OBJ_HAPPYCAT, SPEO_OBJ_GRIE_ROSEN, SPEO_OBJ_SCHWEFEL, SPEO_OBJ_ACKLEY},
         {5.0 / 100.0, 5.0 / 100.0, 5.0 / 100.0, 1000.0 / 100.0, 1.0}},
    };
    const int h = objective - SPEO_OBJ_HYBRID_1;
    if (h < 0 || h >= 6) return false;
    const Def &d = defs[h];
    c.nseg = d.nseg;
    int used = 0;
    for (int s = 0; s < d.nseg; ++s) {
        // ceil(p D) in FP64, CEC2014.cc:961-967; the last segment takes the rest
        const int len = s + 1 < d.nseg ? (int)std::ceil(d.p[s] * dim) : dim - used;
        c.seg[s] = gen_seg(d.obj[s], len, d.rate[s]);
        used += len;
    }
    return true;
}

bool cec_function(int func_id, int *ncomp, CecComp comp[kMaxComp]) {
    // F1-F16 (CEC2014.cc:17-79; kernel_CEC2014_CUDA.cu:1105-1203)
    static const CecComp basic[16] = {
        {SPEO_OBJ_ELLIPTIC, 1.0, 1, 1, 0, 10},           {SPEO_OBJ_BENT_CIGAR, 1.0, 1, 1, 0, 10},
        {SPEO_OBJ_DISCUS, 1.0, 1, 1, 0, 10},             {SPEO_OBJ_ROSENBROCK, 2.048 / 100.0, 1, 1, 0, 10},
        {SPEO_OBJ_ACKLEY, 1.0, 1, 1, 0, 10},             {SPEO_OBJ_WEIERSTRASS, 0.5 / 100.0, 1, 1, 0, 10},
        {SPEO_OBJ_GRIEWANK, 6.0, 1, 1, 0, 10},           {SPEO_OBJ_RASTRIGIN, 5.12 / 100.0, 0, 1, 0, 10},
        {SPEO_OBJ_RASTRIGIN, 5.12 / 100.0, 1, 1, 0, 10}, {SPEO_OBJ_SCHWEFEL, 10.0, 0, 1, 0, 10},
        {SPEO_OBJ_SCHWEFEL, 10.0, 1, 1, 0, 10},          {SPEO_OBJ_KATSUURA, 5.0 / 100.0, 1, 1, 0, 10},
        {SPEO_OBJ_HAPPYCAT, 5.0 / 100.0, 1, 1, 0, 10},   {SPEO_OBJ_HGBAT, 5.0 / 100.0, 1, 1, 0, 10},
        {SPEO_OBJ_GRIE_ROSEN, 5.0 / 100.0, 1, 1, 0, 10}, {SPEO_OBJ_ESCAFFER6, 1.0, 1, 1, 0, 10}};
    if (func_id >= 1 && func_id <= 16) {
        *ncomp = 1;
        comp[0] = basic[func_id - 1];
        return true;
    }
    if (func_id >= 17 && func_id <= 22) {  // hf01-hf06 (CEC2014.cc:80-97)
        *ncomp = 1;
        comp[0] = CecComp{SPEO_OBJ_HYBRID_1 + (func_id - 17), 1.0, 1, 1, 0, 10};
        return true;
    }
    // Compositions cf01-cf08 (CEC2014.cc:1209-1371; CompFunc1-8,
    // kernel_CEC2014_CUDA.cu:1416-1671): lambda is the scaling
    // 10000 * fit / 1e+4 etc. applied before cf_cal adds the bias.
    const double b5[5] = {0, 100, 200, 300, 400};
    auto set = [&](int n, const CecComp *src) {
        *ncomp = n;
        for (int c = 0; c < n; ++c) comp[c] = src[c];
        return true;
    };
    switch (func_id) {
    case 23: {
        const CecComp c[5] = {{SPEO_OBJ_ROSENBROCK, 2.048 / 100.0, 1, 10000 / 1e+4, b5[0], 10},
                              {SPEO_OBJ_ELLIPTIC, 1.0, 1, 10000 / 1e+10, b5[1], 20},
                              {SPEO_OBJ_BENT_CIGAR, 1.0, 1, 10000 / 1e+30, b5[2], 30},
                              {SPEO_OBJ_DISCUS, 1.0, 1, 10000 / 1e+10, b5[3], 40},
                              {SPEO_OBJ_ELLIPTIC, 1.0, 0, 10000 / 1e+10, b5[4], 50}};
        return set(5, c);
    }
    case 24: {
        const CecComp c[3] = {{SPEO_OBJ_SCHWEFEL, 10.0, 0, 1, 0, 20},
                              {SPEO_OBJ_RASTRIGIN, 5.12 / 100.0, 1, 1, 100, 20},
                              {SPEO_OBJ_HGBAT, 5.0 / 100.0, 1, 1, 200, 20}};
        return set(3, c);
    }
    case 25: {
        const CecComp c[3] = {{SPEO_OBJ_SCHWEFEL, 10.0, 1, 1000 / 4e+3, 0, 10},
                              {SPEO_OBJ_RASTRIGIN, 5.12 / 100.0, 1, 1000 / 1e+3, 100, 30},
                              {SPEO_OBJ_ELLIPTIC, 1.0, 1, 1000 / 1e+10, 200, 50}};
        return set(3, c);
    }
    case 26: {
        const CecComp c[5] = {{SPEO_OBJ_SCHWEFEL, 10.0, 1, 1000 / 4e+3, b5[0], 10},
                              {SPEO_OBJ_HAPPYCAT, 5.0 / 100.0, 1, 1000 / 1e+3, b5[1], 10},
                              {SPEO_OBJ_ELLIPTIC, 1.0, 1, 1000 / 1e+10, b5[2], 10},
                              {SPEO_OBJ_WEIERSTRASS, 0.5 / 100.0, 1, 1000 / 400.0, b5[3], 10},
                              {SPEO_OBJ_GRIEWANK, 6.0, 1, 1000 / 100.0, b5[4], 10}};
        return set(5, c);
    }
    case 27: {
        const CecComp c[5] = {{SPEO_OBJ_HGBAT, 5.0 / 100.0, 1, 10000 / 1000.0, b5[0], 10},
                              {SPEO_OBJ_RASTRIGIN, 5.12 / 100.0, 1, 10000 / 1e+3, b5[1], 10},
                              {SPEO_OBJ_SCHWEFEL, 10.0, 1, 10000 / 4e+3, b5[2], 10},
                              {SPEO_OBJ_WEIERSTRASS, 0.5 / 100.0, 1, 10000 / 400.0, b5[3], 20},
                              {SPEO_OBJ_ELLIPTIC, 1.0, 1, 10000 / 1e+10, b5[4], 20}};
        return set(5, c);
    }
    case 28: {
        const CecComp c[5] = {{SPEO_OBJ_GRIE_ROSEN, 5.0 / 100.0, 1, 10000 / 4e+3, b5[0], 10},
                              {SPEO_OBJ_HAPPYCAT, 5.0 / 100.0, 1, 10000 / 1e+3, b5[1], 20},
                              {SPEO_OBJ_SCHWEFEL, 10.0, 1, 10000 / 4e+3, b5[2], 30},
                              {SPEO_OBJ_ESCAFFER6, 1.0, 1, 10000 / 2e+7, b5[3], 40},
                              {SPEO_OBJ_ELLIPTIC, 1.0, 1, 10000 / 1e+10, b5[4], 50}};
        return set(5, c);
    }
    case 29:
    case 30: {
        const int h0 = func_id == 29 ? SPEO_OBJ_HYBRID_1 : SPEO_OBJ_HYBRID_4;
        const CecComp c[3] = {{h0, 1.0, 1, 1, 0, 10}, {h0 + 1, 1.0, 1, 1, 100, 30},
                              {h0 + 2, 1.0, 1, 1, 200, 50}};
        return set(3, c);
    }
    default:
        return false;
    }
}

}  // namespace speo

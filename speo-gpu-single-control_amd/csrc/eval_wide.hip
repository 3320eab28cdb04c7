// eval_wide.hip -- row batches of wide problems (dim > 128) on the pipelined
// tile kernel (wide_core.h), with the arithmetic of k_eval's 64-row form
// (gemm_chunk<64, PREC>): per row and 128-column chunk of Z the partial sums
// k_eval<64, PREC> writes, bit for bit.
//
// A block owns RB rows x 256 columns (two chunks): wave w owns rows
// [WR (w % 4), +WR) of chunk w / 4.  The block order is XCD-aware: the column
// pairs of one row block run on the same XCD (workgroup b on XCD b mod 8), so the
// block's rows are fetched from HBM once into that XCD's L2 and shared.  A
// composition's components run side by side (grid y).
//
// Measured, three components of 16,384 rows x 1000: FP32 1132 -> 839 us (k_eval's
// 64-row tiles, 52 % of the matrix pipe, before; the pipe is 80 % busy now), BF16
// 185 -> 136 us (copies of half cache lines, one launch and one finalize per
// component before).  What bounds it: FP32 the matrix pipe; one 16-bit part the
// LDS reads, conversions and MFMA steps of a stage, which two blocks per compute
// unit overlap in part, and the terms after the last stage.
#include <mutex>

#include "eval.h"
#include "wide_core.h"

namespace speo {

namespace {

// 32 rows per wave.  One 16-bit part: two stage buffers and 128 registers, so
// that two blocks share a compute unit and one block's terms and waits overlap
// the other's MFMA steps (one block of 64 rows per wave and three buffers: 41.5
// us per component of 16,384 rows x 1000, two blocks: 39.3 us).  FP32 and the
// split precisions: their MFMA steps take longer than a stage's loads, and three
// buffers (FP32 295 us either way; BF16x3 102 against 242 us, which spills).
template <int PREC>
using EvalTile = WideTile<PREC, 4, 2, 2, 1, Prec<PREC>::parts == 1 ? 2 : 0>;

// The fields of one component.
struct WideComp {
    const void *wide;
    const float *shift, *colw;
    int objective;
    float rate;
    HeavyCol heavy;
};
struct WideArgs {
    const float *X;
    int ld, n, dim, nchunks, part_bytes;
    float *part;  // [component][nchunks][2][n]
    WideComp comp[kMaxComp];
};

// Per lane, the terms of the wave's eight column tiles in order into the row
// sums of its RTW row tiles (gemm_chunk's epilogue with the objective fixed;
// a function rather than a lambda, so that the accumulators stay in
// registers).
template <int OBJ, int RTW>
__device__ __forceinline__ void wide_terms(const floatx4 (&acc)[RTW][8], const float *colw, int n0,
                                           int dim, int lr, float unscale, float (&s1)[RTW][4],
                                           float (&s2)[RTW][4]) {
#pragma unroll
    for (int t = 0; t < 8; ++t) {
        const int col = n0 + t * 16 + lr;
        if (col < dim) {
            const float w = OBJ == SPEO_OBJ_ELLIPTIC ? colw[col] : 1.0f;
#pragma unroll
            for (int i = 0; i < RTW; ++i)
#pragma unroll
                for (int q = 0; q < 4; ++q) add_terms(OBJ, acc[i][t][q] * unscale, w, s1[i][q], s2[i][q]);
        }
    }
}

template <int PREC>
__global__ __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(Prec<PREC>::parts == 1 ? 4 : 1))) void k_eval_wide(WideArgs p) {
    using W = EvalTile<PREC>;
    extern __shared__ __align__(16) char lds[];
    const int nrb = (p.n + W::RB - 1) / W::RB, ncp = (p.nchunks + 1) / 2;
    const int b = blockIdx.x, xcd = b & 7, j = b >> 3;
    const int cp = j % ncp, rb = (j / ncp) * 8 + xcd;
    if (rb >= nrb) return;  // whole block, before any barrier
    const int row0 = rb * W::RB;
    const WideComp &c = p.comp[blockIdx.y];
    float *part = p.part + (size_t)blockIdx.y * p.nchunks * 2 * p.n;
    const int dim = p.dim;
    const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
    const int lr = lane & 15, lk = lane >> 4;
    const int rg = wave % W::RG, cg = wave / W::RG;

    // The shift, zero-padded to a multiple of 32, stays in LDS after the
    // stage buffers.
    float *shs = reinterpret_cast<float *>(lds + W::LDS);
    for (int k = tid; k < round_up(dim, 32); k += W::NT) shs[k] = k < dim ? c.shift[k] : 0.f;
    __syncthreads();

    // Terms of this wave's columns, in gemm_chunk's order: per lane, the
    // chunk's column tiles in order, then the 16-lane butterfly.
    const float unscale = W::H ? kF16Unscale : 1.0f;
    float s1[W::RTW][4], s2[W::RTW][4];
#pragma unroll
    for (int i = 0; i < W::RTW; ++i)
#pragma unroll
        for (int q = 0; q < 4; ++q) s1[i][q] = s2[i][q] = 0.f;
    const WideOperands o{p.X + (size_t)row0 * p.ld, p.ld, min(W::RB, p.n - row0), dim, c.wide, p.part_bytes,
                         c.rate == 1.0f ? 1 : 0, c.rate};
    wide_gemm<PREC, W>(o, 2 * cp, 1, lds, shs, [&](int chunk, const floatx4 (&acc)[W::RTW][8])
                                                   __attribute__((always_inline)) {
        const int n0 = chunk * kNC;
        switch (c.objective) {  // the objective dispatch of with_objective
        case SPEO_OBJ_ELLIPTIC: wide_terms<SPEO_OBJ_ELLIPTIC>(acc, c.colw, n0, dim, lr, unscale, s1, s2); break;
        case SPEO_OBJ_RASTRIGIN: wide_terms<SPEO_OBJ_RASTRIGIN>(acc, c.colw, n0, dim, lr, unscale, s1, s2); break;
        case SPEO_OBJ_ACKLEY: wide_terms<SPEO_OBJ_ACKLEY>(acc, c.colw, n0, dim, lr, unscale, s1, s2); break;
        case SPEO_OBJ_SCHWEFEL: wide_terms<SPEO_OBJ_SCHWEFEL>(acc, c.colw, n0, dim, lr, unscale, s1, s2); break;
        default: wide_terms<SPEO_OBJ_HAPPYCAT>(acc, c.colw, n0, dim, lr, unscale, s1, s2); break;
        }
    });
    __syncthreads();  // the stage buffers become the row-sum area

    float *red = reinterpret_cast<float *>(lds);  // [2 chunks][RB rows][2]
#pragma unroll
    for (int i = 0; i < W::RTW; ++i)
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const float a1 = sum16(s1[i][q]), a2 = sum16(s2[i][q]);
            if (lr == 0) {
                const int r = rg * W::WR + i * 16 + lk * 4 + q;
                // 0 + s: k_eval's one-term reduction across waves
                red[(cg * W::RB + r) * 2 + 0] = 0.f + a1;
                red[(cg * W::RB + r) * 2 + 1] = 0.f + a2;
            }
        }
    __syncthreads();
    if (c.heavy.j >= 0 && cp == 0) {
        // the heavy column's FP64 term into chunk 0's sums, one wave per row
        for (int r = wave; r < W::RB && row0 + r < p.n; r += W::NW) {
            const double hv = heavy_term(c.heavy, p.X + (size_t)(row0 + r) * p.ld, dim, lane);
            if (lane == 0) red[r * 2] = with_heavy(red[r * 2], (float)hv);
        }
        __syncthreads();
    }
    for (int idx = tid; idx < 2 * W::RB; idx += W::NT) {
        const int g = idx / W::RB, r = idx % W::RB, chunk = 2 * cp + g, row = row0 + r;
        if (chunk < p.nchunks && row < p.n) {
            part[((size_t)chunk * 2 + 0) * p.n + row] = red[idx * 2 + 0];
            part[((size_t)chunk * 2 + 1) * p.n + row] = red[idx * 2 + 1];
        }
    }
}

template <int PREC> int launch_wide(const WideArgs &a, int ncomp, hipStream_t s) {
    using W = EvalTile<PREC>;
    static_assert(2 * W::RB * 2 * 4 <= W::LDS, "row sums must fit in the staging area");
    static std::once_flag once;
    std::call_once(once, [] {
        (void)hipFuncSetAttribute(reinterpret_cast<const void *>(&k_eval_wide<PREC>),
                                  hipFuncAttributeMaxDynamicSharedMemorySize, kWideLdsMax);
    });
    const int nrb = (a.n + W::RB - 1) / W::RB, ncp = (a.nchunks + 1) / 2;
    const int blocks = round_up(nrb, 8) * ncp;
    hipLaunchKernelGGL(k_eval_wide<PREC>, dim3(blocks, ncomp), dim3(W::NT), W::LDS + 4 * round_up(a.dim, 32),
                       s, a);
    return check_launch("k_eval_wide");
}

// One thread per eight values of one (column tile, stage, lane): the two FP32
// pieces' elements and the 16-bit parts of the lane's column.
__global__ void k_wide_fragments(const float *B32, int ldb32, const uint16_t *m0, const uint16_t *m1,
                                 const uint16_t *m2, const uint16_t *m3, const uint16_t *m4,
                                 const uint16_t *m5, int ldm16, int dim, float *f32, uint16_t *f0,
                                 uint16_t *f1, uint16_t *f2, uint16_t *f3, uint16_t *f4, uint16_t *f5) {
    const int nst = (dim + 31) >> 5, ct = blockIdx.x;
    const uint16_t *m[6] = {m0, m1, m2, m3, m4, m5};
    uint16_t *f[6] = {f0, f1, f2, f3, f4, f5};
    for (int e = threadIdx.x; e < nst * 64; e += blockDim.x) {
        const int s = e >> 6, l = e & 63, lr = l & 15, lk = l >> 4, col = 16 * ct + lr;
        const size_t at = (size_t)ct * nst + s;
        for (int u = 0; u < 8 && f32; ++u) {
            const int k = 32 * s + 16 * (u >> 2) + 4 * (u & 3) + lk;
            f32[((at * 2 + (u >> 2)) * 64 + l) * 4 + (u & 3)] =
                col < dim && k < dim ? B32[(size_t)k * ldb32 + col] : 0.f;
        }
#pragma unroll
        for (int p = 0; p < 6; ++p)
            for (int u = 0; u < 8 && f[p]; ++u) {
                const int k = 32 * s + 8 * lk + u;
                f[p][(at * 64 + l) * 8 + u] = col < dim && k < dim ? m[p][(size_t)col * ldm16 + k] : (uint16_t)0;
            }
    }
}

}  // namespace

int wide_fragments(const float *B32, int ldb32, const uint16_t *const M16[6], int ldm16, int dim, float *f32,
                   uint16_t *const f16[6], hipStream_t s) {
    hipLaunchKernelGGL(k_wide_fragments, dim3(round_up((dim + 15) / 16, 16)), dim3(256), 0, s, B32, ldb32,
                       M16[0], M16[1], M16[2], M16[3], M16[4], M16[5], ldm16, dim, f32, f16[0], f16[1], f16[2],
                       f16[3], f16[4], f16[5]);
    return check_launch("k_wide_fragments");
}

bool eval_wide_applies(const CompDev &c, const float *X, int ld, int n, int dim, int precision) {
    int lds = 0;
    switch (precision) {
    case SPEO_PREC_FP32: {
        // from 160 blocks on: a round of up to 256 blocks takes 145 us at D =
        // 1000 whatever its number, as long as 64-row tiles take for 5,800 rows
        // (412 us for 16,384)
        using W = EvalTile<SPEO_PREC_FP32>;
        if ((int64_t)((n + W::RB - 1) / W::RB) * ((dim + 2 * kNC - 1) / (2 * kNC)) < 160) return false;
        lds = W::LDS;
        break;
    }
    case SPEO_PREC_BF16: case SPEO_PREC_FP16: lds = EvalTile<SPEO_PREC_BF16>::LDS; break;
    case SPEO_PREC_BF16X3: case SPEO_PREC_FP16X3: lds = EvalTile<SPEO_PREC_BF16X3>::LDS; break;
    case SPEO_PREC_BF16X6: lds = EvalTile<SPEO_PREC_BF16X6>::LDS; break;
    default: return false;
    }
    static_assert(EvalTile<SPEO_PREC_FP32>::RB == EvalTile<SPEO_PREC_BF16>::RB &&
                  EvalTile<SPEO_PREC_FP32>::RB == EvalTile<SPEO_PREC_BF16X6>::RB, "one bound on the stride");
    return c.wide && dim > kNC && (ld & 3) == 0 && (reinterpret_cast<uintptr_t>(X) & 15) == 0 &&
           wide_stride_fits(EvalTile<SPEO_PREC_FP32>::RB, ld) &&
           lds + 4 * round_up(dim, 32) <= kWideLdsMax;
}

int eval_wide(const CompDev *c, int ncomp, const float *X, int ld, int n, int dim, float *part,
              int precision, hipStream_t s) {
    WideArgs a{X, ld, n, dim, (dim + kNC - 1) / kNC, (int)(2 * wide_frag_elems(dim)), part, {}};
    for (int k = 0; k < ncomp; ++k)
        a.comp[k] = WideComp{c[k].wide, c[k].shift, c[k].colw, c[k].objective, c[k].rate, c[k].heavy};
    switch (precision) {
    case SPEO_PREC_FP32: return launch_wide<SPEO_PREC_FP32>(a, ncomp, s);
    case SPEO_PREC_BF16: return launch_wide<SPEO_PREC_BF16>(a, ncomp, s);
    case SPEO_PREC_FP16: return launch_wide<SPEO_PREC_FP16>(a, ncomp, s);
    case SPEO_PREC_BF16X3: return launch_wide<SPEO_PREC_BF16X3>(a, ncomp, s);
    case SPEO_PREC_FP16X3: return launch_wide<SPEO_PREC_FP16X3>(a, ncomp, s);
    case SPEO_PREC_BF16X6: return launch_wide<SPEO_PREC_BF16X6>(a, ncomp, s);
    default: return set_error(SPEO_ERR_ARG, "eval_wide: unknown precision");
    }
}

}  // namespace speo

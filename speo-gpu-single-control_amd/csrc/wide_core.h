// wide_core.h -- the rotation GEMM of wide problems (rows x 1000 columns) as
// a pipelined tile kernel, shared by the evaluation of row batches
// (eval_wide.hip) and of the engine's islands (engine_wide.hip).
//
// The arithmetic is gemm_chunk's: for every element of Z the same MFMA chain
// over K (v_mfma_f32_16x16x4_f32 in steps of 4, or 16x16x32 with the operand
// parts formed and multiplied in the same order), per row the terms summed lane
// by lane over column tiles in order and then across the 16 lanes by sum16, so
// the sums are gemm_chunk's bit for bit.  What differs is the data path:
//  * a block owns RG x RTW x 16 rows; a wave owns RTW 16-row tiles x
//    TPW 16-column tiles of accumulators;
//  * K in stages of 32 over NBUF LDS buffers, requested NBUF - 1 stages ahead
//    by buffer loads straight into LDS (no registers on the way; the lane's
//    offset is fixed, the stage moves a scalar, rows past the last read as 0);
//  * the rows arrive as FP32, 8 rows x 128 bytes (whole cache lines) per wave
//    load, with the 16-byte groups of row r stored at group ^ (r / 2) % 8, so
//    that the 16 rows of a fragment read fall into different banks;
//  * M is kept in fragment order (wide_fragments): one fragment of a stage is
//    1 KB contiguous in memory and in LDS, read by one conflict-free 16-byte
//    read per lane.
#pragma once

#include <type_traits>

#include "problem.h"

namespace speo {

typedef float floatx8 __attribute__((ext_vector_type(8)));

// PREC: SPEO_PREC_*; a block's waves are RG row groups x CG column chunks x
// NSPLIT column classes (tiles wn, wn + NSPLIT, ... of a chunk); NBUF stage
// buffers (0: three where they fit).
template <int PREC, int RG_, int RTW_, int CG_, int NSPLIT_, int NBUF_ = 0> struct WideTile {
    static constexpr int P = Prec<PREC>::parts;
    static constexpr bool H = Prec<PREC>::half, F32 = P == 0;
    static constexpr int NW = RG_ * CG_ * NSPLIT_, NT = 64 * NW;
    static_assert(NW % 2 == 0, "the waves' row pieces alternate their swizzle");
    static constexpr int RG = RG_, RTW = RTW_, CG = CG_, NSPLIT = NSPLIT_, TPW = 8 / NSPLIT;
    static constexpr int WR = RTW * 16, RB = RG * WR;  // rows per wave, per block
    static constexpr int PIECES = F32 ? 2 : P;         // 1 KB pieces per column tile and stage
    static constexpr int A_BYTES = RB * 128, B_BYTES = 8 * CG * PIECES * 1024, STAGE = A_BYTES + B_BYTES;
    static constexpr int NBUF = NBUF_ ? NBUF_ : 3 * STAGE <= 144 * 1024 ? 3 : 2;
    static constexpr int LDS = NBUF * STAGE;
    static constexpr int NA = RB / 8 / NW, NB = 8 * CG * PIECES / NW, NLD = NA + NB;  // loads per wave and stage
    static_assert(RB % (8 * NW) == 0 && 8 * CG % NW == 0, "loads tile the waves");
};

// s_waitcnt vmcnt(N), the other counters left alone (gfx9 encoding: vmcnt
// in bits 3:0 and 15:14, expcnt 6:4, lgkmcnt 11:8).
template <int N> __device__ __forceinline__ void wait_vm() {
    static_assert(N >= 0 && N < 64, "vmcnt range");
    __builtin_amdgcn_s_waitcnt((N & 15) | (7 << 4) | (15 << 8) | (((N >> 4) & 3) << 14));
}

// A workgroup barrier that neither waits for outstanding memory operations
// (the LDS copies of later stages stay in flight) nor lets the compiler move
// memory accesses across it.
__device__ __forceinline__ void stage_barrier() {
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
}

typedef __attribute__((address_space(3))) void *lds_ptr;

constexpr int kWideLdsMax = 160 * 1024;  // LDS of one CU

// Addresses of a block's rows, in bytes from its first row.  Row piece f holds
// rows 8 f .. 8 f + 7; lane l of the wave that copies it starts at its row 8 f +
// l / 8 with the 16-byte group that the swizzle stores there ((8 f + l / 8) / 2
// mod 8 = 4 (f mod 2) + l / 16), and K stage s adds 128 s.
__host__ __device__ inline int wide_row_offset(int f, int lane, int ld) {
    const int group = (lane & 7) ^ ((4 * (f & 1) + (lane >> 4)) & 7);
    return ((8 * f + (lane >> 3)) * ld + 4 * group) * 4;
}
// What of them may be read: the caller's rows end with the last row's last
// column (rows of a wider matrix's column slice have nothing behind it), and the
// last stage asks for the columns up to a multiple of 32.  The buffer's range
// check, which counts the stage's scalar offset, returns 0 for the rest.
__host__ __device__ inline int wide_row_bytes(int nrows, int ld, int dim) {
    return ((nrows - 1) * ld + round_up(dim, 4)) * 4;
}
// Row strides whose offsets over a block's rows stay within 31 bits.
__host__ __device__ inline bool wide_stride_fits(int rows_per_block, int ld) {
    return (int64_t)rows_per_block * ld * 4 <= 0x7fffffff;
}

// A block's rows and operand.
struct WideOperands {
    const float *rows;   // first row of the block
    int ld, nrows, dim;  // row stride (a multiple of 4 floats, rows 16-byte aligned); rows that exist
    const void *frag;    // the component's M in fragment order (CompDev::wide)
    int part_bytes;      // bytes between its 16-bit parts
    int rate_is_one;
    float rate;
};

// The GEMM of one wave: the accumulators of stage s's operands added, stage by
// stage, over the chunks chunk0, chunk0 + 1, ... (nchunks of them); after each
// chunk done(chunk, acc) consumes the accumulators, which restart at zero.
// Called by all waves of the block; lds holds W::LDS bytes, shs the shift,
// zero-padded to a multiple of 32.  chunk0 is the first chunk of the block's
// columns; wave group cg works on chunk0 + cg (CG > 1: nchunks = 1).
template <int PREC, typename W, typename Done>
__device__ __forceinline__ void wide_gemm(const WideOperands &o, int chunk0, int nchunks, char *lds,
                                          const float *shs, Done done) {
    constexpr int P = W::P;
    constexpr bool H = W::H, F32 = W::F32;
    typedef typename std::conditional<H, halfx8, bf16x8>::type vec8;
    const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
    const int lr = lane & 15, lk = lane >> 4;
    const int wn = wave % W::NSPLIT, rg = (wave / W::NSPLIT) % W::RG, cg = wave / (W::NSPLIT * W::RG);
    const int dim = o.dim, nst = (dim + 31) >> 5;
    const float sa = H ? kF16ScaleA : 1.0f;

    const __amdgpu_buffer_rsrc_t xr = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<float *>(o.rows), (short)0, wide_row_bytes(o.nrows, o.ld, dim), kBufferWord3);
    const __amdgpu_buffer_rsrc_t mr = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<void *>(o.frag), (short)0, (int)0xffffffff, kBufferWord3);
    // row pieces f = wave + NW j (NW is even: one swizzle for all of a wave's)
    const int avoff = wide_row_offset(wave, lane, o.ld);
    const int arow8 = 8 * W::NW * o.ld * 4;  // bytes between the wave's row pieces

    auto issue = [&](int chunk, int s, int buf) __attribute__((always_inline)) {
        char *st = lds + buf * W::STAGE;
#pragma unroll
        for (int j = 0; j < W::NA; ++j)
            __builtin_amdgcn_raw_ptr_buffer_load_lds(xr, (lds_ptr)(st + (wave + W::NW * j) * 1024), 16, avoff,
                                                     j * arow8 + s * 128, 0, 0);
#pragma unroll
        for (int j = 0; j < W::NB; ++j) {
            // piece f = wave + NW j of [column tile][piece]
            const int f = wave + W::NW * j, ct = f / W::PIECES, pc = f % W::PIECES;
            __builtin_amdgcn_raw_ptr_buffer_load_lds(
                mr, (lds_ptr)(st + W::A_BYTES + f * 1024), 16, lane * 16,
                F32 ? (((chunk * 8 + ct) * nst + s) * 2 + pc) * 1024
                    : pc * o.part_bytes + ((chunk * 8 + ct) * nst + s) * 1024,
                0, 0);
        }
    };

    floatx4 acc[W::RTW][W::TPW];
    auto clear = [&]() __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < W::RTW; ++i)
#pragma unroll
            for (int t = 0; t < W::TPW; ++t) acc[i][t] = floatx4{0.f, 0.f, 0.f, 0.f};
    };
    clear();

    const float rate = o.rate;
    const int x8 = (lr >> 1) & 7;
    const int aoff0 = (rg * W::WR + lr) * 128 + ((2 * lk) ^ x8) * 16;      // 16-bit: coordinates 8 lk .. + 3
    const int aoff1 = (rg * W::WR + lr) * 128 + ((2 * lk + 1) ^ x8) * 16;  // and 8 lk + 4 .. + 7
    const int foff = (rg * W::WR + lr) * 128 + lk * 4;                     // FP32: coordinate 4 ks + lk
    const int boff = W::A_BYTES + (cg * 8 + wn) * W::PIECES * 1024 + lane * 16;

    // One stage.  MASK zeroes the operand past the dimension (the last stage: M
    // is zero there, the rows may hold anything); UNIT drops the multiplication by a rate of 1, which is exact.
    auto compute = [&](int s, int buf, auto mask, auto unit) __attribute__((always_inline)) {
        // (the split's remainder is that of the rounded product, whatever the
        // including file's contraction mode)
#pragma clang fp contract(off)
        constexpr bool MASK = decltype(mask)::value, UNIT = decltype(unit)::value;
        const char *st = lds + buf * W::STAGE;
        if constexpr (F32) {
            // every row value of the stage is read before the first step needs one
            float a[8][W::RTW];
            {
                float ov[8];
#pragma unroll
                for (int ks = 0; ks < 8; ++ks) {
                    ov[ks] = shs[s * 32 + 4 * ks + lk];
#pragma unroll
                    for (int i = 0; i < W::RTW; ++i)
                        a[ks][i] = *reinterpret_cast<const float *>(st + foff + ((ks ^ x8) << 4) + i * 2048);
                }
#pragma unroll
                for (int ks = 0; ks < 8; ++ks)
#pragma unroll
                    for (int i = 0; i < W::RTW; ++i) {
                        a[ks][i] = (a[ks][i] - ov[ks]) * rate;
                        if constexpr (MASK)
                            if (s * 32 + 4 * ks + lk >= dim) a[ks][i] = 0.f;
                    }
            }
            floatx4 b[2][W::TPW];
#pragma unroll
            for (int h = 0; h < 2; ++h)
#pragma unroll
                for (int t = 0; t < W::TPW; ++t)
                    b[h][t] = *reinterpret_cast<const floatx4 *>(st + boff + (t * W::NSPLIT * 2 + h) * 1024);
            __builtin_amdgcn_sched_barrier(0);
            __builtin_amdgcn_s_setprio(1);
#pragma unroll
            for (int ks = 0; ks < 8; ++ks) {
                if (MASK && s * 32 + 4 * ks >= dim) break;  // the rest are zeros
#pragma unroll
                for (int t = 0; t < W::TPW; ++t)
#pragma unroll
                    for (int i = 0; i < W::RTW; ++i)
                        acc[i][t] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[ks][i], b[ks >> 2][t][ks & 3],
                                                                         acc[i][t], 0, 0, 0);
            }
            __builtin_amdgcn_s_setprio(0);
        } else {
            const int k = s * 32 + 8 * lk;
            const floatx4 o0 = *reinterpret_cast<const floatx4 *>(shs + k);
            const floatx4 o1 = *reinterpret_cast<const floatx4 *>(shs + k + 4);
            const floatx8 ov = __builtin_shufflevector(o0, o1, 0, 1, 2, 3, 4, 5, 6, 7);
            vec8 a[W::RTW][P], bb[W::TPW][P];
#pragma unroll
            for (int i = 0; i < W::RTW; ++i) {
                const floatx4 x0 = *reinterpret_cast<const floatx4 *>(st + aoff0 + i * 2048);
                const floatx4 x1 = *reinterpret_cast<const floatx4 *>(st + aoff1 + i * 2048);
                // eight coordinates as one vector: the conversions pair up into
                // packed converts with no packing instructions after them
                const floatx8 d = __builtin_shufflevector(x0, x1, 0, 1, 2, 3, 4, 5, 6, 7) - ov;
                floatx8 rem = UNIT ? d * sa : d * rate * sa;
                if constexpr (MASK) {
#pragma unroll
                    for (int q = 0; q < 8; ++q)
                        if (k + q >= dim) rem[q] = 0.f;
                }
#pragma unroll
                for (int pp = 0; pp < P; ++pp) {
                    a[i][pp] = __builtin_convertvector(rem, vec8);
                    if (pp + 1 < P) rem -= __builtin_convertvector(a[i][pp], floatx8);
                }
            }
#pragma unroll
            for (int t = 0; t < W::TPW; ++t)
#pragma unroll
                for (int pp = 0; pp < P; ++pp)
                    bb[t][pp] = *reinterpret_cast<const vec8 *>(st + boff + (t * W::NSPLIT * P + pp) * 1024);
            __builtin_amdgcn_sched_barrier(0);
            __builtin_amdgcn_s_setprio(1);
#pragma unroll
            for (int t = 0; t < W::TPW; ++t)
#pragma unroll
                for (int i = 0; i < W::RTW; ++i) {
                    // small products first, then hi*hi (gemm_chunk's order)
#pragma unroll
                    for (int sum = P - 1; sum >= 0; --sum)
#pragma unroll
                        for (int pa = 0; pa <= sum; ++pa) {
                            const int pb = sum - pa;
                            if (pa < P && pb < P) {
                                if constexpr (H)
                                    acc[i][t] = __builtin_amdgcn_mfma_f32_16x16x32_f16(a[i][pa], bb[t][pb],
                                                                                       acc[i][t], 0, 0, 0);
                                else
                                    acc[i][t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[i][pa], bb[t][pb],
                                                                                        acc[i][t], 0, 0, 0);
                            }
                        }
                }
            __builtin_amdgcn_s_setprio(0);
        }
    };

    // Stages 0 .. NBUF - 2 (of the whole run over the chunks) are requested up
    // front.  At each stage a wave waits for its own loads of that stage (those
    // of the NBUF - 2 stages after it may stay in flight); after the barrier
    // every wave's loads of the stage have landed and every wave has finished
    // the stage before, whose buffer takes the stage NBUF - 1 ahead.
    const int total = nchunks * nst;
    int ic = chunk0, is = 0, ib = 0, issued = 0;  // the next stage to request
    auto issue_next = [&]() __attribute__((always_inline)) {
        if (issued < total) {
            issue(ic, is, ib);
            ++issued;
            if (++is == nst) {
                is = 0;
                ++ic;
            }
            if (++ib == W::NBUF) ib = 0;
        }
    };
#pragma unroll
    for (int u = 0; u < W::NBUF - 1; ++u) issue_next();
    auto run = [&](auto unit) __attribute__((always_inline)) {
        int buf = 0;
        for (int chunk = chunk0; chunk < chunk0 + nchunks; ++chunk) {
            for (int s = 0; s < nst - 1; ++s) {
                if (W::NBUF == 3)
                    wait_vm<W::NLD>();
                else
                    wait_vm<0>();
                stage_barrier();
                issue_next();
                compute(s, buf, std::false_type{}, unit);
                if (++buf == W::NBUF) buf = 0;
            }
            if (W::NBUF == 3 && chunk + 1 < chunk0 + nchunks)
                wait_vm<W::NLD>();
            else
                wait_vm<0>();
            stage_barrier();
            issue_next();
            compute(nst - 1, buf, std::true_type{}, std::false_type{});  // coordinates past dim
            if (++buf == W::NBUF) buf = 0;
            done(chunk + cg, acc);
            clear();
        }
    };
    if (!F32 && o.rate_is_one)
        run(std::true_type{});
    else
        run(std::false_type{});
}

// M in fragment order, zero padded: column tiles rounded up to a multiple of 16
// (two chunks), K to stages of 32.  FP32: column tile ct, stage s, half h, lane
// l (lr = l % 16, lk = l / 16), element e at (((ct nst + s) 2 + h) 64 + l) 4 +
// e, holding M[16 ct + lr][32 s + 16 h + 4 e + lk]; 16-bit, per part: lane l's
// eight values M[16 ct + lr][32 s + 8 lk ..] at ((ct nst + s) 64 + l) 8.
__host__ __device__ inline size_t wide_frag_elems(int dim) { return (size_t)round_up((dim + 15) / 16, 16) * 16 * round_up(dim, 32); }
// The kernels move through the three 16-bit parts by 32-bit byte offsets.
inline bool wide_frag_fits(int dim) { return 3 * 2 * wide_frag_elems(dim) < 0x7fffffffull; }
// f32 and the six of f16 (BF16 parts, FP16 parts): any may be null.
int wide_fragments(const float *B32, int ldb32, const uint16_t *const M16[6], int ldm16, int dim, float *f32,
                   uint16_t *const f16[6], hipStream_t s);

}  // namespace speo

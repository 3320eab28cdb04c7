// de.h -- DE operator building blocks shared by the standalone kernels and
// the fused generation kernel.
#pragma once

#include "common.h"

namespace speo {

// One island of the engine's batch, as the kernels see it.
struct IslandDesc {
    int64_t elem_off;  // first element of row 0 in X / U
    int row_off;       // first row in the fitness arrays
    int np, dim, ld;   // rows, coordinates, row stride (ld % 4 == 0)
    int problem;       // index into the problem table
    float F, CR;
};

struct GenArgs {
    float *U;
    const float *X;
    int ld, n, dim;
    int S;  // sub-island size
    const int *perm;
    const DEInfo *de_info;
    const int *best;
    float lo, hi;
    uint64_t seed;
    uint32_t gen, row_base;
    const float *inj_r;
    int n_inj;
    const float *inj_cr;
    int *r_out, *jrand_out;
    // set: each sub-island's best member (fit [n] over rows) is found first and
    // stored in best_out, `best` is not read
    const float *fit = nullptr;
    int *best_out = nullptr;
};

// Sequential donor-phase draws of one row: draw k is word k%4 of Philox block
// {k/4, row, gen, purpose}; the first n_inj draws may be injected.  Blocks 0
// and 1 (the eight draws that cover the five donors and j_rand unless a row
// redraws more than twice) are computed up front, independently of each other.
struct DonorStream {
    uint64_t seed;
    uint32_t row, gen, k, cached, purpose;
    U4 w0, w1, cw;
    __host__ __device__ DonorStream(uint64_t s, uint32_t r, uint32_t g, uint32_t pur = kPurposeDonor)
        : seed(s), row(r), gen(g), k(0), cached(0xffffffffu), purpose(pur), cw{0, 0, 0, 0} {
        w0 = philox_block(s, 0u, r, g, pur);
        w1 = philox_block(s, 1u, r, g, pur);
    }
    __host__ __device__ __forceinline__ float next(const float *inj, int n_inj) {
        // (the words move up by one a draw, so that none is picked by an index
        // the compiler would put in memory)
        const uint32_t kk = k++, head = w0.x;
        w0 = U4{w0.y, w0.z, w0.w, w1.x};
        w1 = U4{w1.y, w1.z, w1.w, 0u};
        if (inj && (int)kk < n_inj) return inj[kk];
        if (kk < 8u) return u01(head);
        const uint32_t blk = kk >> 2;
        if (blk != cached) {
            cw = philox_block(seed, blk, row, gen, purpose);
            cached = blk;
        }
        return u01(word(cw, kk & 3u));
    }
};

// (int)(u S), clamped to [0, S] so that injected draws outside (0, 1] cannot
// index outside the sub-island; u in (0, 1] is unaffected.
__host__ __device__ __forceinline__ int scale_draw(float u, int S) {
    const int v = (int)(u * (float)S);
    return v < 0 ? 0 : (v > S ? S : v);
}

// kernel_DE_CUDA.cu:187-222: five sub-island-local donors, each redrawn while
// it equals an earlier one (earlier ones are not rechecked after a redraw),
// "== S" decremented before and after the redraw loop, then j_rand = (int)(u D)
// with no "== D" guard.  The target is not excluded.  Written with one draw
// site per donor: j walks the earlier donors, a collision redraws and stays
// on j, so the sequence of draws is that of the nested loops.
__host__ __device__ __forceinline__ void draw_donors(DonorStream &s, const float *inj, int n_inj, int S,
                                            int D, int (&r)[kMaxR], int &jr) {
    // (the i-th donor, with the earlier ones by value: they stay in registers)
    auto donor = [&](int i, int p0, int p1, int p2, int p3) {
        int v = 0, j = 0;
        bool draw = true, first = true;
        for (;;) {
            if (draw) {
                v = scale_draw(s.next(inj, n_inj), S);
                if (first && v == S) v--;
                first = false;
                draw = false;
            }
            if (j >= i) break;
            const int rj = j == 0 ? p0 : j == 1 ? p1 : j == 2 ? p2 : p3;
            if (v == rj && s.k < (uint32_t)kMaxDraws)
                draw = true;
            else
                ++j;
        }
        return v == S ? v - 1 : v;
    };
    const int r0 = donor(0, 0, 0, 0, 0), r1 = donor(1, r0, 0, 0, 0), r2 = donor(2, r0, r1, 0, 0);
    const int r3 = donor(3, r0, r1, r2, 0), r4 = donor(4, r0, r1, r2, r3);
    r[0] = r0;
    r[1] = r1;
    r[2] = r2;
    r[3] = r3;
    r[4] = r4;
    static_assert(kMaxR == 5, "five donors");
    jr = (int)(s.next(inj, n_inj) * (float)D);
}

// (f ascending, row ascending, NaN last): whether (a, ia) comes before (b, ib).
__device__ __forceinline__ bool before(float a, int ia, float b, int ib) {
    const bool an = isnan(a), bn = isnan(b);
    if (an != bn) return bn;
    if (!an && a != b) return a < b;
    return ia < ib;
}

// Block argmin of (f[slot], slot) over members t in [0, count): slot =
// perm ? perm[base + t] : base + t.  Valid on thread 0; sf and si hold one
// entry per wave.
__device__ __forceinline__ int block_argmin(const float *f, const int *perm, int base, int count,
                                            float *sf, int *si) {
    float bf = NAN;
    int bi = 0x7fffffff;
    for (int t = threadIdx.x; t < count; t += blockDim.x) {
        const int slot = perm ? perm[base + t] : base + t;
        const float v = f[slot];
        if (bi == 0x7fffffff || before(v, slot, bf, bi)) {
            bf = v;
            bi = slot;
        }
    }
    for (int off = 32; off > 0; off >>= 1) {
        const float of = __shfl_xor(bf, off, 64);
        const int oi = __shfl_xor(bi, off, 64);
        if (oi != 0x7fffffff && (bi == 0x7fffffff || before(of, oi, bf, bi))) {
            bf = of;
            bi = oi;
        }
    }
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    if (lane == 0) {
        sf[wave] = bf;
        si[wave] = bi;
    }
    __syncthreads();
    if (threadIdx.x == 0)
        for (int w = 1; w < (int)(blockDim.x >> 6); ++w)
            if (si[w] != 0x7fffffff && (bi == 0x7fffffff || before(sf[w], si[w], bf, bi))) {
                bf = sf[w];
                bi = si[w];
            }
    return bi;
}

// ceil(2^32 / ng), ng = ceil(dim / 4), for e / ng = mulhi(e, inverse): with it
// e * inverse / 2^32 exceeds e / ng by less than e / 2^32, which reaches no next
// whole number while e * ng < 2^32.  For e < 64 ng; 0 where that does not hold
// or ng == 1.
inline uint32_t group_inverse(int dim) {
    const uint64_t ng = ((uint64_t)dim + 3) / 4;
    return ng > 1 && 64 * ng * ng < (1ull << 32) ? (uint32_t)((0x100000000ull + ng - 1) / ng) : 0u;
}

int init_population(float *X, int ld, int n, int dim, float lo, float hi, uint64_t seed,
                    uint32_t row_base, hipStream_t s);
int de_generate(const GenArgs &a, hipStream_t s);
int de_select(float *X, float *fX, const float *U, float *fU, int ld, int n, int dim,
              uint8_t *accept_out, int clear_trials, hipStream_t s);
int segment_argmin(const float *f, const int *off, int nseg, int *best_out, hipStream_t s);
// Best slot of each of `subs` sub-islands of size S (members perm[s S ..]),
// ties to the lower slot, NaN last.
int subisland_best(const float *f, const int *perm, int S, int subs, int *best_out, hipStream_t s);
int migrate_ring(float *X, float *fX, const IslandDesc *isl_desc_dev, const int *row_off_dev,
                 const int *dst_dev, int *best_buf, int *worst_buf, int I, int max_np, int k,
                 hipStream_t s);  // max_np: rows of the largest island

}  // namespace speo

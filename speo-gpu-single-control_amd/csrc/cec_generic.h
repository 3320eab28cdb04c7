// cec_generic.h -- the CEC2014 objectives outside the fused FP32 epilogues:
// Rosenbrock, Weierstrass, Griewank, Katsuura, Griewank-Rosenbrock, expanded
// Schaffer F6, the hybrid functions (shuffled z cut into segments of different
// objectives) and compositions over any of them (F4, F6, F7, F12, F15-F23,
// F26-F30 of CEC2014.cc:14-145; kernel_CEC2014_CUDA.cu:355-1671).
//
// One block per tile of 16 rows: z = M ((x - o) rate) for each component on
// v_mfma_f64_16x16x4f64 with FP64 accumulation into an LDS-resident Z tile,
// then each row's objective by one wave from that tile (segment objectives
// over the shuffled z for hybrids), then the composition weights.  The same
// kernel gives the FP64 values of every problem (re-verification).  FP64
// throughout: Weierstrass scales z + 1/2 by 3^20 and Katsuura z by 2^32
// before taking a cosine or a fractional part, so an FP32 z (relative error
// ~1e-7) would leave those terms with no correct digits.
#pragma once

#include "problem.h"

namespace speo {

constexpr int kGenMaxDim = 1024;  // Z tile of 16 rows in LDS
constexpr int kGenMaxSeg = 5;
constexpr int kGenRows = 16;
constexpr int kGenThreads = 64 * kGenRows;  // one wave per row

// One segment of a component: objective `obj` (SPEO_OBJ_*, 1..14) over
// `len` consecutive coordinates of the (shuffled) z, scaled by `rate`.
struct GenSeg {
    int obj;
    int len;
    double rate;
    double par;  // Katsuura: its exponent 10 / len^1.2
};
GenSeg gen_seg(int objective, int len, double rate);

struct GenComp {
    int nseg;                  // 1: one objective over all coordinates
    GenSeg seg[kGenMaxSeg];
    const int *perm;           // hybrids: 1-based shuffle [dim] (the shuffle_data format), or null
    double rate;               // applied to x - o before the rotation (sr_func's sh_rate)
    int rotate;                // 0: z = (x - o) rate
    const double *o64;         // shift [dim]
    const double *M64f;        // M in fragment order (gen_fragments)
    double lambda, bias, sigma;  // fit = lambda g + bias; composition weight width
};

struct GenProblem {
    int dim, ncomp;
    GenComp comp[kMaxComp];
};

// Launch arguments: the problem's description lies in device memory (its
// fields are then L2 hits; as a 2 KB argument every 64-byte line of it was a
// scalar load from the host's argument memory at its first use).
struct GenLaunch {
    const GenProblem *P;       // device
    int dim, ncomp;            // of *P
    const float *X;            // rows of stride ld
    int ld, n;
    const int *rows;           // optional: launch row i reads row rows[i] - row_base of X
    int row_base;
    float *f32;                // outputs (either may be null)
    double *f64;
    double out_bias;           // added to every output
    int block_rows;            // set by eval_generic
    // The drop-in call's arrays, component c at c * stride (M^T: c * stride *
    // dim): used in place of the description's shift, rotation, shuffle and
    // sigma when o32 is set.
    const float *o32, *B32, *sigma32;
    const int *perm;
    int stride;
};

// SPEO_OBJ_HYBRID_1..6 -> the component's segments at `dim` (CEC2014.cc:954-1207):
// lengths ceil(p_i dim) in FP64 and the rest for the last segment.  Returns
// false for another objective.
bool hybrid_segments(int objective, int dim, GenComp &c);

// One component of CEC2014 function func_id (1..30) as the reference defines
// it (CEC2014.cc:14-145, 954-1371): objective, rate, rotation, lambda, bias,
// sigma; component count in *ncomp.  Returns false for an unknown function.
struct CecComp {
    int objective;   // SPEO_OBJ_* (hybrids: SPEO_OBJ_HYBRID_k)
    double rate;
    int rotate;
    double lambda, bias, sigma;
};
bool cec_function(int func_id, int *ncomp, CecComp comp[kMaxComp]);

// True when the problem needs this path (an objective outside 1..8, i.e.
// not one the fused FP32 epilogues take).
bool generic_objective(int objective);

// M (row-major, z_i = sum_j M_ij y_j) in the kernel's fragment order, zero
// padded: for 16-column tile t of z and K step s of 8, lane l's two doubles
// M[16 t + l % 16][8 s + 2 (l / 16) + 0..1] lie at ((t S + s) 64 + l) 2, S =
// ceil(dim / 8), so that a wave's operand is 1 KB contiguous.
inline size_t gen_fragment_doubles(int dim) { return (size_t)((dim + 15) / 16) * ((dim + 7) / 8) * 128; }
int gen_fragments(const double *M64, int dim, double *out, hipStream_t s);

// The components of *g, before it is uploaded: segments that cover dim <=
// kGenMaxDim, and a shift and a rotation where they are needed (`arrays`: the
// launch brings its own).
int check_gen_problem(const GenProblem &g, bool arrays);

// Evaluates n rows.
int eval_generic(const GenLaunch &p, hipStream_t s);

}  // namespace speo

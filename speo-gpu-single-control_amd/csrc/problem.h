// problem.h -- device-resident shifted-rotated problem (objective host wrapper).
// Counterpart of the reference's CEC2014_CUDA (CUDA_EA_library/CEC2014_CUDA.h:
// 38-82): owns the shift vectors and rotation matrices on the device, in every
// layout the kernels use, instead of loading CEC text files.
#pragma once

#include <vector>

#include "eval_core.h"
#include "workspace.h"

namespace speo {

constexpr int kMaxComp = 8;

// Column weights w_j of the weighted-sphere objectives, sum_j w_j z_j^2:
// elliptic 10^(6 j / (D - 1)), bent cigar (1, 10^6, 10^6, ...), discus
// (10^6, 1, 1, ...).  The FP32 kernels evaluate all three through one path.
bool weighted_sphere(int objective);
// The column that outweighs all others together (index), or -1; *w_out its
// FP64 weight.  column_weights gives it weight 0: the kernels add its term
// in FP64 (CompDev::heavy).
int heavy_column(int objective, int dim, double *w_out);
void column_weights(int objective, int dim, float *w);

struct CompHost {
    int objective = SPEO_OBJ_RASTRIGIN;
    float rate = 1.0f;     // FP32 kernels
    double rate64 = 1.0;   // FP64 verifier (a rate such as 0.0512 is not a float)
    double sigma = 10.0, bias = 0.0, lambda = 1.0;
    float *shift32 = nullptr;   // [dim]
    double *shift64 = nullptr;  // [dim]
    float *B32 = nullptr;       // [dim][ldb32]: B[k][c] = M[c][k]
    uint16_t *Mbf[3] = {nullptr, nullptr, nullptr};  // BF16 parts of M, [dim][ldm16]
    uint16_t *Mh[3] = {nullptr, nullptr, nullptr};   // FP16 parts of 2^14 M
    double *M64 = nullptr;      // [dim][dim]
    double *M64f = nullptr;     // M64 in the FP64 kernel's fragment order (dim <= 1024, rotated)
    // dim <= 128 only: zero-padded layouts of the register-resident-B path
    float *B32s = nullptr;                                   // 128 x 128, fragment order
    uint16_t *Mbfs[3] = {nullptr, nullptr, nullptr};         // [128][round_up(dim,32)]
    uint16_t *Mhs[3] = {nullptr, nullptr, nullptr};
    // dim > 128, FP32 epilogues only: M in the wide kernels' fragment order (wide_core.h):
    float *wide32 = nullptr;    // FP32,
    uint16_t *wide_bf = nullptr, *wide_h = nullptr;  // the three BF16 and the three FP16 parts
    float *colw = nullptr;      // [dim] bent cigar / discus weights (elliptic: ProblemHost::colw)
    int heavy_j = -1;           // heavy_column of the objective, found once (it takes dim
    double heavy_w = 0.0;       // powers, more host time than the launch of a small evaluation)
    bool unrotated = false;     // M = I: evaluated in FP32 whatever the requested precision,
                                // where the identity GEMM is exact
};

// Per-component parameters of the FP64 path and of the composition combine,
// stored on the device as an array.
struct CompParams {
    int objective;
    double rate;
    double sigma, bias, lambda;
    const float *shift32;
    const double *shift64;
    const double *M64;
};

struct GenProblem;

struct ProblemHost {
    int dim = 0, ncomp = 0;
    int ldb32 = 0, ldm16 = 0;
    float *colw = nullptr;          // [dim] elliptic weights
    CompParams *params_dev = nullptr;  // [ncomp]
    CompHost comp[kMaxComp];
    CompDev view(int c, int precision) const;
    // Objectives outside the fused FP32 epilogues (Rosenbrock, Weierstrass,
    // Griewank, Katsuura, Griewank-Rosenbrock, Schaffer F6, hybrids): the
    // whole problem is evaluated by the FP64 generic kernel (cec_generic.h).
    bool generic = false;
    int *perm[kMaxComp] = {};       // hybrids: 1-based shuffle [dim] on the device
    GenProblem *gen = nullptr;      // the FP64 kernel's description, on the device (dim <= 1024)
    // Every array above lies in one of two device allocations, the data and the
    // tables that point into it (params_dev, gen); the data of components of more
    // than 4 MiB in one each.
    void *data[kMaxComp + 1] = {}, *tables = nullptr;
};

}  // namespace speo

struct speo_problem_s {
    speo::ProblemHost h;
    // speo_evaluate's: the sums of eval_problem, and rows copied to an aligned
    // stride (a buffer of its own, so that a captured evaluation of aligned rows
    // keeps its sums' addresses when rows of another stride come)
    speo::Workspace scratch, packed;
};

// eval.h -- host entry points of the evaluation kernels.
#pragma once

#include "problem.h"

namespace speo {

struct EvalLaunch {
    CompDev comp;
    const float *X;
    int ld, n, dim;
    float *f_out;   // [n]
    float *part;    // [nchunks][2][n] when nchunks > 1
    int nchunks;
    float lambda, bias;
    int raw;        // 1: write g (composition component), 0: lambda * g + bias
    int small;      // dim <= 128 with the padded layouts: register-resident-B path
};

// One component over n rows; `part` is needed when dim > 128.
int eval_component(const CompDev &comp, const float *X, int ld, int n, int dim, float *f_out,
                   float *part, float lambda, float bias, int raw, int precision,
                   int rows_per_block, hipStream_t s);

// Scratch (floats) eval_problem needs for n rows; with eval_scratch_batched
// floats a wide composition's components run in one launch.
size_t eval_scratch_floats(int ncomp, int dim, int n);
size_t eval_scratch_batched(int ncomp, int dim, int n);

// Whole problem (single component or composition) over n rows; scratch holds
// scratch_floats floats; packed: null, or room for eval_pack_floats (16-byte
// aligned), to which the rows are copied first.
int eval_problem(const ProblemHost &P, const float *X, int ld, int n, float *f_out, float *scratch,
                 size_t scratch_floats, float *packed, int precision, int rows_per_block, hipStream_t s);

// FP64 evaluation: the generic kernel up to its 1024 columns, else one block
// per row (eval_rows_f64).
int eval_rows_f64(const CompParams *comps, int ncomp, int dim, const float *X, int ld, int n,
                  double *f_out, hipStream_t s);
int eval_problem_f64(const ProblemHost &P, const float *X, int ld, int n, double *f_out,
                     hipStream_t s);

// Floats of an aligned copy of rows wider than 128 columns that 16-byte accesses
// cannot take as they are (0: they can, or the copy would pass 1 GiB).
size_t eval_pack_floats(const ProblemHost &P, const float *X, int ld, int n);
// kept: the rotation is kept in a problem's layouts (the drop-in call's is not).
int default_rows_per_block(int n, int dim, int precision, bool kept);

// The tile kernels of wide problems are switched on (speo_wide_eval).
bool wide_eval_enabled();

// k_eval_wide: the evaluation of components wider than 128 columns with
// k_eval<64, precision>'s bits: component k's partial sums into part + k
// nchunks 2 n, finalized by the caller; applies when X and its stride allow
// 16-byte loads and, in FP32, when the rows fill the chip.
bool eval_wide_applies(const CompDev &c, const float *X, int ld, int n, int dim, int precision);
int eval_wide(const CompDev *c, int ncomp, const float *X, int ld, int n, int dim, float *part,
              int precision, hipStream_t s);

// Problems with objectives outside the fused FP32 epilogues (ProblemHost::
// generic): the FP64 generic kernel, FP32 and/or FP64 outputs; rows (device,
// optional) select rows[i] - row_base of X for launch row i.
int eval_problem_generic(const ProblemHost &P, const float *X, int ld, int n, float *f32,
                         double *f64, const int *rows, int row_base, hipStream_t s);

}  // namespace speo

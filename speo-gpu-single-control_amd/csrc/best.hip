// best.hip -- FP64 values of single rows: each island's best row
// (EA_CUDA::FindBestIndividual, EA_CUDA.cc:104-120, with the FP64 forms of
// CEC2014.cc) and rows wider than the generic kernel takes.
#include <algorithm>

#include "engine.h"
#include "eval.h"
#include "eval_f64.h"

namespace speo {

// FP64 values of rows wider than the generic kernel's 1024 columns: one block
// per row.
__global__ __launch_bounds__(256) void k_eval_f64(const CompParams *comps, int ncomp, int dim,
                                                  const float *X, int ld, int n, double *f_out) {
    extern __shared__ __align__(16) char lds_raw[];
    double *a = reinterpret_cast<double *>(lds_raw);
    double *red = a + dim;  // [4][3]
    const int row = blockIdx.x, tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
    if (row >= n) return;
    const float *x = X + (size_t)row * ld;
    double fit = 0.0, dist = 0.0, sigma = 1.0;  // lane c: component c's
    for (int c = 0; c < ncomp; ++c) {
        const CompParams cp = comps[c];
        double s1 = 0.0, s2 = 0.0, d = 0.0;
        __syncthreads();
        for (int j = tid; j < dim; j += 256) {
            const double v = (double)x[j] - cp.shift64[j];
            a[j] = v * cp.rate;
            d = fma(v, v, d);
        }
        __syncthreads();
        for (int c0 = 8 * wave; c0 < dim; c0 += 32) {
            const double z = gemv8(cp.M64, a, dim, c0, lane);
            const int col = c0 + (lane >> 3);
            if ((lane & 7) == 0 && col < dim) add_terms64(cp.objective, col, dim, z, s1, s2);
        }
        s1 = wave_sum64(s1);
        s2 = wave_sum64(s2);
        d = wave_sum64(d);
        if (lane == 0) {
            red[wave * 3 + 0] = s1;
            red[wave * 3 + 1] = s2;
            red[wave * 3 + 2] = d;
        }
        __syncthreads();
        s1 = s2 = d = 0.0;
        for (int w = 0; w < 4; ++w) {
            s1 += red[w * 3 + 0];
            s2 += red[w * 3 + 1];
            d += red[w * 3 + 2];
        }
        if (lane == c) {
            fit = cp.lambda * finish_objective64(cp.objective, s1, s2, dim) + cp.bias;
            dist = d;
            sigma = cp.sigma;
        }
    }
    const double f = ncomp == 1 ? __shfl(fit, 0, 64) : combine64(ncomp, dim, fit, dist, sigma, lane);
    if (tid == 0) f_out[row] = f;
}

// Each island's best row (ties to the lower row, NaN last) and its FP64 value.
// A block of 16 waves takes 128 columns of z = M (x - o) rate, eight per wave
// (gemv8).  Islands of at most 128 columns are finished by their one block,
// component by component; wider ones have a block per (chunk, component) whose
// sums k_best_combine adds in chunk order, so that the rows of M (8 dim^2
// bytes per component) come in over many compute units.  One block of four
// waves per island, each reducing one column at a time, took 40 us for 64
// islands of D = 100 and 4.6 ms for 8 islands of a three-function composition
// at D = 1000 (latency; one compute unit read 24 MB); with the results written
// straight to pinned host memory instead of three copies back, a call is
// 55-75 us shorter on the small runs and 4.7 ms on the wide one.
constexpr int kBestThreads = 1024;
__global__ __launch_bounds__(kBestThreads) void k_best(BestArgs p) {
    extern __shared__ __align__(16) char lds_raw[];
    double *a = reinterpret_cast<double *>(lds_raw);
    __shared__ float sf[kBestThreads / 64];
    __shared__ int si[kBestThreads / 64];
    __shared__ double red[kBestThreads / 64][3];
    const int isl = blockIdx.x, chunk = blockIdx.y;
    const IslandDesc I = p.isl[isl];
    const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
    const bool first = chunk == 0 && blockIdx.z == 0;
    const FusedProblem *P = p.probs + I.problem;
    const int dim = I.dim, nc = P->ncomp;
    // the generic kernel evaluates the rows of generic problems
    const bool evaluates = !P->generic && chunk * kBestCols < dim && (int)blockIdx.z < nc;
    if (!first && !evaluates) return;
    const int b = block_argmin(p.fX, nullptr, I.row_off, I.np, sf, si);
    if (tid == 0) si[0] = b;
    __syncthreads();
    const int row = si[0];
    if (first && tid == 0) {
        p.best_row[isl] = row;
        p.out[isl].row = row;
        p.out[isl].f32 = p.fX[row];
    }
    if (!evaluates) return;
    const float *x = p.X + I.elem_off + (size_t)(row - I.row_off) * I.ld;
    const int c0 = p.chunks > 1 ? (int)blockIdx.z : 0, c1 = p.chunks > 1 ? c0 + 1 : nc;
    double fit = 0.0, dist = 0.0, sigma = 1.0;  // lane c: component c's
    for (int c = c0; c < c1; ++c) {
        const CompParams cp = p.comps[I.problem][c];
        double s1 = 0.0, s2 = 0.0, d = 0.0;
        __syncthreads();
        for (int j = tid; j < dim; j += kBestThreads) {
            const double v = (double)x[j] - cp.shift64[j];
            a[j] = v * cp.rate;
            d = fma(v, v, d);
        }
        __syncthreads();
        const int col0 = chunk * kBestCols + 8 * wave;
        if (col0 < dim) {
            const double z = gemv8(cp.M64, a, dim, col0, lane);
            const int col = col0 + (lane >> 3);
            if ((lane & 7) == 0 && col < dim) add_terms64(cp.objective, col, dim, z, s1, s2);
        }
        s1 = wave_sum64(s1);
        s2 = wave_sum64(s2);
        d = wave_sum64(d);
        if (lane == 0) {
            red[wave][0] = s1;
            red[wave][1] = s2;
            red[wave][2] = d;
        }
        __syncthreads();
        s1 = s2 = d = 0.0;
        for (int w = 0; w < kBestThreads / 64; ++w) {
            s1 += red[w][0];
            s2 += red[w][1];
            d += red[w][2];
        }
        if (p.chunks > 1) {
            double *o = p.part + (((size_t)isl * kMaxComp + c) * p.chunks + chunk) * 3;
            if (tid == 0) {
                o[0] = s1;
                o[1] = s2;
                o[2] = d;
            }
        } else if (lane == c) {
            fit = cp.lambda * finish_objective64(cp.objective, s1, s2, dim) + cp.bias;
            dist = d;
            sigma = cp.sigma;
        }
    }
    if (p.chunks > 1 || wave != 0) return;
    const double f = nc == 1 ? __shfl(fit, 0, 64) : combine64(nc, dim, fit, dist, sigma, lane);
    if (lane == 0) p.out[isl].f64 = f;
}

// One wave per island: the chunks' sums of every component, then the value.
__global__ __launch_bounds__(64) void k_best_combine(BestArgs p) {
    const int isl = blockIdx.x, lane = threadIdx.x;
    const IslandDesc I = p.isl[isl];
    const FusedProblem *P = p.probs + I.problem;
    if (P->generic) return;
    const int dim = I.dim, nc = P->ncomp, chunks = (dim + kBestCols - 1) / kBestCols;
    double fit = 0.0, dist = 0.0, sigma = 1.0;
    for (int c = 0; c < nc; ++c) {
        const CompParams cp = p.comps[I.problem][c];
        const double *o = p.part + ((size_t)isl * kMaxComp + c) * p.chunks * 3;
        double s1 = 0.0, s2 = 0.0;
        for (int k = lane; k < chunks; k += 64) {
            s1 += o[3 * k];
            s2 += o[3 * k + 1];
        }
        s1 = wave_sum64(s1);
        s2 = wave_sum64(s2);
        if (lane == c) {
            fit = cp.lambda * finish_objective64(cp.objective, s1, s2, dim) + cp.bias;
            dist = o[2];  // every chunk holds the row's distance
            sigma = cp.sigma;
        }
    }
    const double f = nc == 1 ? __shfl(fit, 0, 64) : combine64(nc, dim, fit, dist, sigma, lane);
    if (lane == 0) p.out[isl].f64 = f;
}

int eval_rows_f64(const CompParams *comps, int ncomp, int dim, const float *X, int ld, int n,
                  double *f_out, hipStream_t s) {
    const size_t lds = sizeof(double) * ((size_t)dim + 16);
    if (lds > 48 * 1024)
        SPEO_TRY_HIP(hipFuncSetAttribute(reinterpret_cast<const void *>(&k_eval_f64),
                                         hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
    hipLaunchKernelGGL(k_eval_f64, dim3(n), dim3(256), lds, s, comps, ncomp, dim, X, ld, n, f_out);
    return check_launch("k_eval_f64");
}

int best_rows(const BestArgs &p, int islands, int ncomp, int max_dim, hipStream_t s) {
    const size_t lds = sizeof(double) * (size_t)max_dim;
    if (lds > 48 * 1024)
        SPEO_TRY_HIP(hipFuncSetAttribute(reinterpret_cast<const void *>(&k_best),
                                         hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
    hipLaunchKernelGGL(k_best, p.chunks > 1 ? dim3(islands, p.chunks, ncomp) : dim3(islands),
                       dim3(kBestThreads), lds, s, p);
    SPEO_TRY(check_launch("k_best"));
    if (p.chunks == 1) return SPEO_OK;
    hipLaunchKernelGGL(k_best_combine, dim3(islands), dim3(64), 0, s, p);
    return check_launch("k_best_combine");
}

}  // namespace speo

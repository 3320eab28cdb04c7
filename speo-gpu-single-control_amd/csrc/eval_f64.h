// eval_f64.h -- FP64 building blocks of the objectives (generic evaluation and
// re-verification), following the reference's FP64 CPU forms: elliptic
// CEC2014.cc:481-497, bent cigar 499-516, discus 518-530, Ackley 590-612,
// Rastrigin 668-683, Schwefel 705-738, HappyCat 907-929, HGBat 931-953,
// composition weights cf_cal 1481-1519.
#pragma once

#include "problem.h"

namespace speo {

constexpr double kPi64 = 3.1415926535897932384626433832795029;
constexpr double kE64 = 2.7182818284590452353602874713526625;

// cos x and sin x with an absolute error of a few 1e-16:
// x = n pi + r, |r| <= pi / 2, with pi as the sum of two doubles for |x| < 2^45
// (the first fused multiply-add rounds x - n pi_hi at the size of r, and n is
// exact), then r's Taylor polynomial (the first dropped terms, r^22 / 22! and
// r^23 / 23!, are below 3e-17) with the sign of odd n.  About 20 FP64
// instructions; the math library's functions choose between two reductions
// and two polynomials per lane and cost several times as much here, where every
// coordinate of every row takes up to 21 of them (Weierstrass).
//
// Beyond 2^45: the fraction of x / (2 pi) from the bits of 1 / (2 pi) that the
// integer part does not swallow (Payne and Hanek, 1983).  x = m 2^e with a
// 53-bit m, so the bits of weight 2^-e and above only add whole turns; the next
// 128 bits times m, modulo one turn, are the fraction, of which 64 bits are kept
// (to 2^-63 of a turn).
constexpr int kTurnWords = 20;
__device__ inline double large_turns(double x) {
    static const __constant__ uint64_t kTurnBits[kTurnWords + 1] = {  // 1 / (2 pi), after 64 zero bits
    0ull,
    0x28be60db9391054aull, 0x7f09d5f47d4d3770ull, 0x36d8a5664f10e410ull, 0x7f9458eaf7aef158ull,
    0x6dc91b8e909374b8ull, 0x01924bba82746487ull, 0x3f877ac72c4a69cfull, 0xba208d7d4baed121ull,
    0x3a671c09ad17df90ull, 0x4e64758e60d4ce7dull, 0x272117e2ef7e4a0eull, 0xc7fe25fff7816603ull,
    0xfbcbc462d6829b47ull, 0xdb4d9fb3c9f2c26dull, 0xd3d18fd9a797fa8bull, 0x5d49eeb1faf97c5eull,
    0xcf41ce7de294a4baull, 0x9afed7ec47e35742ull, 0x1580cc11bf1edaeaull, 0xfc33ef0826bd0d87ull};
    const uint64_t bits = __builtin_bit_cast(uint64_t, x);
    const int ex = (int)((bits >> 52) & 0x7ff);
    if (ex == 0x7ff) return x - x;  // infinities and NaN
    const uint64_t m = (bits & 0xfffffffffffffull) | 0x10000000000000ull;
    const int pos = ex - 1075 + 64, w = pos >> 6, sh = pos & 63;  // 57 <= pos <= 1035
    const uint64_t b0 = kTurnBits[w], b1 = kTurnBits[w + 1], b2 = kTurnBits[w + 2];
    const uint64_t hi = sh ? (b0 << sh) | (b1 >> (64 - sh)) : b0, lo = sh ? (b1 << sh) | (b2 >> (64 - sh)) : b1;
    const uint64_t f = m * hi + __umul64hi(m, lo);  // modulo one turn
    const double t = (double)(int64_t)f * 0x1p-64;
    return (int64_t)bits < 0 ? -t : t;
}
__device__ __forceinline__ double trig_reduce(double x, bool *odd) {
    if (!(fabs(x) < 0x1p45)) x = 6.2831853071795864769 * large_turns(x);
    const double n = rint(x * 0.31830988618379067154);
    double r = fma(-n, 3.141592653589793116, x);
    r = fma(-n, 1.2246467991473531772e-16, r);
    const double h = 0.5 * n;
    *odd = h != rint(h);
    return r;
}
__device__ __forceinline__ double cos64(double x) {
    bool odd;
    const double r = trig_reduce(x, &odd), u = r * r;
    double c = 1.0 / 2432902008176640000.0;  // 1 / 20!
    c = fma(c, u, -1.0 / 6402373705728000.0);
    c = fma(c, u, 1.0 / 20922789888000.0);
    c = fma(c, u, -1.0 / 87178291200.0);
    c = fma(c, u, 1.0 / 479001600.0);
    c = fma(c, u, -1.0 / 3628800.0);
    c = fma(c, u, 1.0 / 40320.0);
    c = fma(c, u, -1.0 / 720.0);
    c = fma(c, u, 1.0 / 24.0);
    c = fma(c, u, -0.5);
    c = fma(c, u, 1.0);
    return odd ? -c : c;
}
__device__ __forceinline__ double sin64(double x) {
    bool odd;
    const double r = trig_reduce(x, &odd), u = r * r;
    double c = 1.0 / 51090942171709440000.0;  // 1 / 21!
    c = fma(c, u, -1.0 / 121645100408832000.0);
    c = fma(c, u, 1.0 / 355687428096000.0);
    c = fma(c, u, -1.0 / 1307674368000.0);
    c = fma(c, u, 1.0 / 6227020800.0);
    c = fma(c, u, -1.0 / 39916800.0);
    c = fma(c, u, 1.0 / 362880.0);
    c = fma(c, u, -1.0 / 5040.0);
    c = fma(c, u, 1.0 / 120.0);
    c = fma(c, u, -1.0 / 6.0);
    const double s = fma(c * u, r, r);
    return odd ? -s : s;
}

// x mod 500 for x >= 0: x - 500 q is exact in one fused multiply-add while q,
// the truncated quotient or one of its neighbours, is a whole double.
__device__ __forceinline__ double mod500(double x) {
    if (!(x < 0x1p52)) return fmod(x, 500.0);
    const double q = trunc(x * (1.0 / 500.0));
    double r = fma(-q, 500.0, x);
    if (r < 0.0) r += 500.0;
    if (r >= 500.0) r -= 500.0;
    return r;
}

// The modified Schwefel function's term of v = z + 420.97 (the value to add to
// the row's sum), folded beyond |v| = 500; n is the dimension.
__device__ __forceinline__ double schwefel64(double v, double n) {
    const double av = fabs(v);
    if (av <= 500.0) return -v * sin64(sqrt(av));
    const double m = 500.0 - mod500(av), t = (av - 500.0) / 100.0;
    return (v > 0.0 ? -m : m) * sin64(sqrt(m)) + t * t / n;
}

// One coordinate's terms of the objectives 1..8, added to s1 and s2.
__device__ __forceinline__ void add_terms64(int objective, int i, int dim, double z, double &s1,
                                            double &s2) {
    switch (objective) {
    case SPEO_OBJ_ELLIPTIC: s1 += exp10(6.0 * i / (dim - 1)) * z * z; break;
    case SPEO_OBJ_BENT_CIGAR: s1 += (i == 0 ? 1.0 : 1.0e6) * z * z; break;
    case SPEO_OBJ_DISCUS: s1 += (i == 0 ? 1.0e6 : 1.0) * z * z; break;
    case SPEO_OBJ_SCHWEFEL: s1 += schwefel64(z + 4.209687462275036e+002, dim); break;
    case SPEO_OBJ_HAPPYCAT:
    case SPEO_OBJ_HGBAT:
        s1 += (z - 1.0) * (z - 1.0);
        s2 += z - 1.0;
        break;
    case SPEO_OBJ_RASTRIGIN: s1 += z * z - 10.0 * cos64(2.0 * kPi64 * z) + 10.0; break;
    default:
        s1 += z * z;
        s2 += cos64(2.0 * kPi64 * z);
        break;
    }
}

// The objective's value from the two sums over a row's n coordinates.
__device__ __forceinline__ double finish_objective64(int objective, double s1, double s2, double n) {
    switch (objective) {
    case SPEO_OBJ_ACKLEY: return kE64 - 20.0 * exp(-0.2 * sqrt(s1 / n)) + 20.0 - exp(s2 / n);
    case SPEO_OBJ_SCHWEFEL: return s1 + 4.189828872724338e+002 * n;
    case SPEO_OBJ_HAPPYCAT: return sqrt(sqrt(fabs(s1 - n))) + (0.5 * s1 + s2) / n + 0.5;
    case SPEO_OBJ_HGBAT: return sqrt(fabs(s1 * s1 - s2 * s2)) + (0.5 * s1 + s2) / n + 0.5;
    default: return s1;
    }
}

__device__ __forceinline__ double wave_sum64(double v) {
    for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off, 64);
    return v;
}

// cf_cal (CEC2014.cc:1481-1519) by one wave: lane c < ncomp holds component
// c's value `fit` (lambda g + bias), squared distance d and width sigma; the
// composition's value is returned on every lane.
__device__ __forceinline__ double combine64(int ncomp, int dim, double fit, double d, double sigma,
                                            int lane) {
    double w = 0.0;
    if (lane < ncomp) w = d != 0.0 ? sqrt(1.0 / d) * exp(-d / 2.0 / dim / (sigma * sigma)) : 1.0e99;
    double wmax = 0.0, wsum = 0.0;
    for (int c = 0; c < ncomp; ++c) {
        const double wc = __shfl(w, c, 64);
        wmax = fmax(wmax, wc);
        wsum += wc;
    }
    if (wmax == 0.0) {
        w = 1.0;
        wsum = ncomp;
    }
    double f = 0.0;
    for (int c = 0; c < ncomp; ++c) f += __shfl(w, c, 64) / wsum * __shfl(fit, c, 64);
    return f;
}

// Columns [c0, c0 + 8) of z = M a for one row by one wave: a (dim doubles) in
// LDS, M row-major; lane l ends with column c0 + (l >> 3) (0 past the
// dimension).  Eight rows of M are read side by side, and the lanes' partial
// sums are halved and exchanged (4 + 2 + 1 values, then three steps of one)
// instead of eight full butterflies.
__device__ __forceinline__ double gemv8(const double *M, const double *a, int dim, int c0, int lane) {
    double z[8];
    const double *m[8];
#pragma unroll
    for (int u = 0; u < 8; ++u) {
        z[u] = 0.0;
        m[u] = M + (size_t)min(c0 + u, dim - 1) * dim;
    }
    for (int k = lane; k < dim; k += 64) {
        const double ak = a[k];
#pragma unroll
        for (int u = 0; u < 8; ++u) z[u] = fma(gld(m[u] + k), ak, z[u]);
    }
    // lane bits 5, 4, 3 choose the column: four, two, one of the sums kept
    auto halve = [&](double x, double y, int bit) {  // lanes with the bit set keep y
        const bool up = (lane & bit) != 0;
        const double keep = up ? y : x, send = up ? x : y;
        return keep + __shfl_xor(send, bit, 64);
    };
    const double p0 = halve(z[0], z[4], 32), p1 = halve(z[1], z[5], 32), p2 = halve(z[2], z[6], 32),
                 p3 = halve(z[3], z[7], 32);
    const double q0 = halve(p0, p2, 16), q1 = halve(p1, p3, 16);
    double v = halve(q0, q1, 8);
#pragma unroll
    for (int off = 4; off > 0; off >>= 1) v += __shfl_xor(v, off, 64);
    return c0 + (lane >> 3) < dim ? v : 0.0;
}

}  // namespace speo

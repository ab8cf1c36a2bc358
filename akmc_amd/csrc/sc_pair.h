// Pair physics of the Sutton-Chen kernels: coefficients, powers, minimum
// image, lane sums and the pair table in LDS.  Included by every kernel file
// that evaluates Sutton-Chen pairs, so they share one arithmetic.
#pragma once
#include "akmc_internal.h"

#include <math.h>

namespace {

template <typename T>
__device__ inline const SCCoef<T> &sc_coef(const SCPairDev &p);
template <>
__device__ inline const SCCoef<float> &sc_coef<float>(const SCPairDev &p) { return p.f; }
template <>
__device__ inline const SCCoef<double> &sc_coef<double>(const SCPairDev &p) { return p.d; }

// 1/x: the hardware reciprocal (1 ulp) on the FP32 path, an exact division
// on the FP64 verification path
template <typename T>
__device__ inline T recip(T x) { return T(1) / x; }
template <>
__device__ inline float recip<float>(float x) { return __builtin_amdgcn_rcpf(x); }

// u^x for non-integer exponents: libm pow on the FP64 path; on the FP32
// path the integer part of x by squaring and the fraction by libm log2f /
// exp2f (relative-accurate near u = 1, where (a/r)^2 lives), which keeps
// the error of u^x at a few ulp without the cost of a full powf
__device__ inline double pow_general(double u, double x) { return pow(u, x); }
__device__ inline float pow_general(float u, float x)
{
    if (!(x >= 0.0f && x < 64.0f)) return exp2f(x * log2f(u));  // outside the split's range
    const float xi = floorf(x);
    float r = 1.0f, base = u;
    for (int p = int(xi); p > 0; p >>= 1) {
        if (p & 1) r *= base;
        base *= base;
    }
    return r * exp2f((x - xi) * log2f(u));
}

// square root for the integer powers: the hardware instruction (1 ulp) on
// the FP32 path, whose arguments (a/r)^2 are normal numbers far from the
// denormal range the correctly rounded expansion guards; libm on FP64
__device__ inline double root(double x) { return sqrt(x); }
__device__ inline float root(float x) { return __builtin_amdgcn_sqrtf(x); }

// 1/sqrt(x) in FP64 for normal x > 0: the hardware estimate refined by two
// Newton steps y += y (1 - x y^2) / 2 (quadratic convergence), a few ulp
// from the correctly rounded value at a third of the cost of a division and
// a square root
__device__ inline double rsqrt_fp64(double x)
{
    double y = __builtin_amdgcn_rsq(x);
    double r = fma(-(x * y), y, 1.0);
    y = fma(0.5 * y, r, y);
    r = fma(-(x * y), y, 1.0);
    return fma(0.5 * y, r, y);
}

// The single-species power inputs of U pairs: ir2 = 1/r^2, u2 = (a/r)^2 and,
// in FP64, rt = a/r.  FP32: hardware reciprocal (the power takes sqrt(u2)
// from the hardware square root for odd exponents).  FP64: one refined 1/r,
// so that neither a division nor a square root is needed.
template <typename T, int U>
__device__ inline void sc_powers_in(const double (&r2)[U], T a, T (&ir2)[U], T (&u2)[U], T (&rt)[U])
{
    if constexpr (sizeof(T) == 8) {
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const double ir = rsqrt_fp64(r2[u]);
            ir2[u] = ir * ir;
            u2[u] = a * a * ir2[u];
            rt[u] = a * ir;
        }
    } else {
#pragma unroll
        for (int u = 0; u < U; ++u) {
            ir2[u] = recip<T>(T(r2[u]));
            u2[u] = a * a * ir2[u];
            rt[u] = T(0);  // the FP32 power takes its root from u2 itself
        }
    }
}

// (a/r)^9 and (a/r)^6 of the single-pair kernels from u2 = (a/r)^2, with
// the compile-time exponents of the Sutton-Chen pairs they serve: the
// products of the repeated squaring, u8 sqrt(u2) and u2 u4, without its
// loop
template <typename T, int U>
__device__ inline void pow_9_6(const T (&u2)[U], const T (&rt)[U], T (&u9)[U], T (&u6)[U])
{
#pragma unroll
    for (int u = 0; u < U; ++u) {
        const T u4 = u2[u] * u2[u];
        const T u8 = u4 * u4;
        u9[u] = u8 * (sizeof(T) == 8 ? rt[u] : root(u2[u]));
        u6[u] = u2[u] * u4;
    }
}
template <typename T, int U>
__device__ inline void pow_6(const T (&u2)[U], T (&u6)[U])
{
#pragma unroll
    for (int u = 0; u < U; ++u) u6[u] = u2[u] * (u2[u] * u2[u]);
}

// sqrt(x) from the hardware estimate and one Newton step on its exact
// residual: the correctly rounded square root but for 3 in 2^24 arguments,
// whose roots lie within 10^-7 of a unit from a rounding boundary, at half
// the instructions
__device__ inline float root_refined(float x)
{
    const float y = __builtin_amdgcn_rsqf(x), r = x * y;
    return __builtin_fmaf(__builtin_fmaf(-r, r, x), 0.5f * y, r);
}

// 1/r^2, (a/r)^9 and (a/r)^6 of a table pair: the products of pow_half's
// repeated squaring, without its loops (a pair table whose exponents are 9
// and 6 throughout).  FP64: 1/r^2 and a/r from one refined 1/r, each with a
// last Newton step on its own exact residual, which gives them the bits of
// the division and the square root of the general pairs (600 distances of
// 600; the pair energy's error 4.8 half-units rms, without the steps 7.6)
template <typename T>
__device__ inline void table_9_6(double r2, const SCCoef<T> &c, T &ir2, T &un, T &um)
{
    T u2, rt;
    if constexpr (sizeof(T) == 8) {
        const double ir = rsqrt_fp64(r2), q = ir * ir, s = c.a * ir;
        ir2 = fma(q, fma(-r2, q, 1.0), q);
        u2 = c.a * c.a * ir2;
        // (the residual is a few units of s: 1 / (2 s) to FP32's bits is enough)
        rt = fma(fma(-s, s, u2), double(0.5f * __builtin_amdgcn_rsqf(float(u2))), s);
    } else {
        ir2 = recip<T>(T(r2));
        u2 = c.a * c.a * ir2;
        rt = root_refined(u2);
    }
    const T u4 = u2 * u2;
    un = u4 * u4 * rt;
    um = u2 * u4;
}

template <typename T>
__device__ inline T pow_half(T u2, int k, T e)
{
    // u2^(e/2) with u2 = (a/r)^2; exact repeated squaring when e is an integer
    if (k >= 0) {
        T r = T(1), base = u2;
        int p = k >> 1;
        while (p) {
            if (p & 1) r *= base;
            base *= base;
            p >>= 1;
        }
        if (k & 1) r *= sqrt(u2);
        return r;
    }
    return pow_general(u2, e * T(0.5));
}

__device__ inline void min_image(double &dx, double &dy, double &dz, const WalkerDev &w)
{
    dx -= w.L[0] * rint(dx * w.invL[0]);
    dy -= w.L[1] * rint(dy * w.invL[1]);
    dz -= w.L[2] * rint(dz * w.invL[2]);
}

// sum over the LPA consecutive lanes that share one atom
template <int LPA>
__device__ inline double lane_group_sum(double v)
{
    for (int o = LPA / 2; o > 0; o >>= 1) v += __shfl_xor(v, o);
    return v;
}

// The Sutton-Chen pair table (nspec^2 entries) staged in LDS by every
// workgroup before any thread leaves, so the coefficient lookup of a pair is
// an LDS read instead of a third dependent global load.
__device__ inline void stage_sc_table(const FieldDev &F, SCPairDev *tab)
{
    static_assert(sizeof(SCPairDev) % 4 == 0, "table staged in 4-byte words");
    const int nw = F.nspec * F.nspec * int(sizeof(SCPairDev) / 4);
    const uint32_t *src = reinterpret_cast<const uint32_t *>(F.sc);
    uint32_t *dst = reinterpret_cast<uint32_t *>(tab);
    for (int w = threadIdx.x; w < nw; w += blockDim.x) dst[w] = src[w];
    __syncthreads();
}

}  // namespace

// FP64 sine and cosine for the network models' phase differences: few instructions and few
// live registers.
//
// The library sin/cos carry an argument reduction for huge |x| (a multi-word product
// with 2/pi) whose temporaries set the register count of every kernel that inlines them,
// although the network models never reach it: a fused vertex kernel with one inlined
// library sin per entry needs 106 VGPRs (4 waves per SIMD), 65 without.  Here:
//
//   * Cody-Waite reduction by pi/2: k = rint(x * 2/pi), r = ((x - k*P1) - k*P2) - k*P3,
//     where P1 and P2 hold the leading 33 significant bits each of pi/2 (so k*P1 and
//     k*P2 are exact for |k| < 2^20) and P3 the next 53 bits;
//   * on |r| <= pi/4 sin r = r + r^3 S(r^2) and cos r = 1 - r^2/2 + r^4 C(r^2), S and C the
//     minimax polynomials of degrees 6 and 5 of the relative error (Remez exchange in 60
//     digits: 2.0e-21 and 5.6e-20 before the coefficients are rounded);
//   * |x| >= 2^20 * pi/2 and non-finite x go to the library function, out of line.
//
// Reduction and polynomials are explicit fused multiply-adds: the build compiles with
// -ffp-contract=off (which keeps the models' own arithmetic unfused), and a v_fma_f64 issues
// as fast as a product or a sum alone.  About 35 vector instructions a sine; with separate
// products and sums and Taylor polynomials it was 55.  One polynomial on |r| <= pi/2 would
// take 18, but its error is larger (0.30 ulp on average and 1.7 at most for |x| < pi).
//
// Largest and mean error in ulp against 80-bit sines of 1.6e7 random arguments (in brackets
// the Taylor form this replaced):
//   |x| < 0.8    1.05 (1.08)   0.253 (0.257)
//   |x| < 2 pi   1.32 (1.33)   0.286 (0.289)
//   |x| < 1e4    2.17 (2.17)   0.309 (0.311)
// and of the cosine (4e6 arguments a range):
//   pi/4 .. 0.8  1.01 (0.76)   0.381 (0.258)
//   |x| < 0.8    1.00 (0.75)   0.256 (0.253)
//   |x| < 2 pi   1.39 (1.44)   0.300 (0.302)
//   |x| < 1e4    2.28 (2.28)   0.309 (0.311)
// (just above pi/4 the rounding of the reduced argument is the same for all x, a bias of a third
// of an ulp, and the Taylor form's own error there had the other sign)
#pragma once

#include <hip/hip_runtime.h>

#include <cmath>

namespace nd {

constexpr double kTwoOverPi = 0x1.45f306dc9c883p-1;
constexpr double kPio2_1 = 0x1.921fb54400000p+0;    // pi/2, leading 33 bits
constexpr double kPio2_2 = 0x1.0b4611a600000p-34;   // the next 33 bits
constexpr double kPio2_3 = 0x1.3198a2e037073p-69;   // the next 53 bits
constexpr double kReduceMax = 1647099.3291652855;   // 2^20 * pi/2

__host__ __device__ __forceinline__ double fma_(double a, double b, double c) { return __builtin_fma(a, b, c); }

// sin(r) and cos(r) for |r| <= pi/4 (Horner in z = r^2)
__host__ __device__ __forceinline__ double sin_kernel(double r) {
    const double z = r * r;
    double q = fma_(z, -0x1.aaa24723321d2p-41, 0x1.61208c47f6473p-33);
    q = fma_(z, q, -0x1.ae64528d7eb79p-26);
    q = fma_(z, q, 0x1.71de3a53308bep-19);
    q = fma_(z, q, -0x1.a01a01a018a6dp-13);
    q = fma_(z, q, 0x1.111111111110bp-7);
    q = fma_(z, q, -0x1.5555555555555p-3);
    return fma_(r * z, q, r);
}

__host__ __device__ __forceinline__ double cos_kernel(double r) {
    const double z = r * r;
    double q = fma_(z, -0x1.8fa4996919a9fp-37, 0x1.1ee9d7b3b4e7ep-29);
    q = fma_(z, q, -0x1.27e4f7eac303bp-22);
    q = fma_(z, q, 0x1.a01a019c844cfp-16);
    q = fma_(z, q, -0x1.6c16c16c14f91p-10);
    q = fma_(z, q, 0x1.555555555554bp-5);
    // 1 - z/2 + z^2 q, with the leading subtraction done first for accuracy near pi/4
    const double w = fma_(-0.5, z, 1.0);
    return w + fma_(z * z, q, fma_(-0.5, z, 1.0 - w));
}

#if defined(__HIP_DEVICE_COMPILE__)
__device__ __noinline__ double sin_far(double x) { return ::sin(x); }
__device__ __noinline__ double cos_far(double x) { return ::cos(x); }
#else
inline double sin_far(double x) { return std::sin(x); }
inline double cos_far(double x) { return std::cos(x); }
#endif

// quadrant q = k mod 4 of x = k*pi/2 + r: sin(x) = sin r, cos r, -sin r, -cos r.  Both
// polynomials, then selects: no branch, so several arguments' chains overlap
__host__ __device__ __forceinline__ double quadrant_value(int q, double r) {
    const double s = sin_kernel(r), c = cos_kernel(r);
    const double v = (q & 1) ? c : s;
#if defined(__HIP_DEVICE_COMPILE__)
    return __hiloint2double(__double2hiint(v) ^ ((q << 30) & static_cast<int>(0x80000000u)), __double2loint(v));
#else
    return (q & 2) ? -v : v;
#endif
}

__host__ __device__ __forceinline__ double reduce_pio2(double x, int* q) {
    const double k = rint(x * kTwoOverPi);
    *q = static_cast<int>(k);
    return fma_(-k, kPio2_3, fma_(-k, kPio2_2, fma_(-k, kPio2_1, x)));
}

// within the fast range; elsewhere some value, finite or not
__host__ __device__ __forceinline__ double sin_near(double x) {
    int q;
    const double r = reduce_pio2(x, &q);
    return quadrant_value(q, r);
}
__host__ __device__ __forceinline__ double cos_near(double x) {
    int q;
    const double r = reduce_pio2(x, &q);
    return quadrant_value(q + 1, r);
}

// y[i] = sin(x[i]).  The fast path of all N arguments runs without a branch between them, so
// their dependent chains overlap; arguments outside its range are redone afterwards.
template <int N>
__host__ __device__ __forceinline__ void nd_sin_n(const double (&x)[N], double (&y)[N]) {
    bool far = false;
#pragma unroll
    for (int i = 0; i < N; ++i) {
        far |= !(fabs(x[i]) < kReduceMax);
        y[i] = sin_near(x[i]);
    }
    if (__builtin_expect(far, 0))
#pragma unroll
        for (int i = 0; i < N; ++i)
            if (!(fabs(x[i]) < kReduceMax)) y[i] = sin_far(x[i]);
}

__host__ __device__ __forceinline__ double nd_sin(double x) {
    if (!(fabs(x) < kReduceMax)) return sin_far(x);
    return sin_near(x);
}

__host__ __device__ __forceinline__ double nd_cos(double x) {
    if (!(fabs(x) < kReduceMax)) return cos_far(x);
    return cos_near(x);
}

}  // namespace nd

// FP64 divisions, square roots and WENO5-Z of the drop-in, with fewer VALU
// cycles than the compiler's expansions and the same bits.
//
// The FP64 stages are bound by VALU issue, and in cycles most of a WENO5-Z
// stage is division: on gfx950 an add, multiply or fma in FP64 issues every
// ~5 cycles per wavefront, a reciprocal estimate every 18 and the compiler's
// division takes 63 (a square root 85), measured at 8 wavefronts per SIMD.
//
// Division a/b (Markstein, "Computation of elementary functions on the IBM
// RISC System/6000 processor", 1990): r approximates 1/b to within a hair over
// half an ulp, q = a r, and q + (a - b q) r with the exact remainder from an
// fma rounds to the nearest double. r comes from the hardware estimate r0
// (relative error e below 2^-24) by one cubic step r0 (1 + e + e^2), whose
// error e^3 < 2^-72 is far below the rounding: one fma fewer than two Newton
// steps.
//
// Three forms, by what is known of the operands:
//   div_ieee   any operands (div_scale / div_fmas / div_fixup around it);
//   Recip      one divisor for several dividends, no scaling: exact when b and
//              a/b stay within 2^+-900 and |a| > 2^-900 (or 0); zeros,
//              infinities and NaN come out as IEEE's (div_fixup);
//   div_plain  no special cases: WENO5-Z's tau / (beta + eps). The divisor is
//              at least 1e-36, and a quotient below 2^-27 leaves the weight
//              1 + ind^2 = 1 whatever its last bits, so a tiny or zero tau
//              needs no care.
//
// With them a WENO5-Z + HLLC stage issues 1572 VALU instructions per row of
// the march instead of 1917; the KH step at 2048^2 takes 0.80 ms instead of
// 0.93 and the one at 512^2 134 us instead of 156.
#pragma once

#include <hip/hip_runtime.h>

namespace mh {

#if defined(__HIP_DEVICE_COMPILE__)
__device__ inline double recip_refined(double b) {
    const double r0 = __builtin_amdgcn_rcp(b);
    const double e = __builtin_fma(-b, r0, 1.0);
    return __builtin_fma(r0, __builtin_fma(e, e, e), r0);
}
__device__ inline double div_plain(double a, double b) {
    const double r = recip_refined(b);
    const double q = a * r;
    return __builtin_fma(__builtin_fma(-b, q, a), r, q);
}
__device__ inline double div_ieee(double a, double b) {
    bool scaled, unused;
    const double bs = __builtin_amdgcn_div_scale(a, b, false, &unused);
    const double as = __builtin_amdgcn_div_scale(a, b, true, &scaled);
    const double r = recip_refined(bs);
    const double q = as * r;
    return __builtin_amdgcn_div_fixup(__builtin_amdgcn_div_fmas(__builtin_fma(-bs, q, as), r, q, scaled), b, a);
}
// sqrt(x) for x zero, negative (NaN) or above 2^-900 and finite (smaller ones
// come out to 1e-14): Goldschmidt's iteration (Goldschmidt, "Applications of
// division by convergence", MIT, 1964) from the hardware 1/sqrt(x) and two
// residual corrections, without the scaling that smaller arguments need.
__device__ inline double sqrt_plain(double x) {
    double y = __builtin_amdgcn_rsq(x);
    y = x == 0.0 ? 0x1p+500 : y;  // 0 * finite = 0 below instead of 0 * inf
    double g = x * y, h = 0.5 * y;
    const double r = __builtin_fma(-g, h, 0.5);
    g = __builtin_fma(g, r, g);
    h = __builtin_fma(h, r, h);
    g = __builtin_fma(__builtin_fma(-g, g, x), h, g);
    return __builtin_fma(__builtin_fma(-g, g, x), h, g);
}
// ... and infinity (inf * 0 above)
__device__ inline double sqrt_inf(double x) {
    const double g = sqrt_plain(x);
    return x == __builtin_inf() ? x : g;
}
#else
__host__ inline double div_plain(double a, double b) { return a / b; }
__host__ inline double div_ieee(double a, double b) { return a / b; }
__host__ inline double sqrt_plain(double x) { return __builtin_sqrt(x); }
__host__ inline double sqrt_inf(double x) { return __builtin_sqrt(x); }
#endif

// A divisor used more than once.
template <typename T>
struct Recip {
    T b;
    __host__ __device__ explicit Recip(const T& x) : b(x) {}
    __host__ __device__ T div(const T& a) const { return a / b; }
    __host__ __device__ T mul(const T& a) const { return a / b; }
};
template <>
struct Recip<double> {
    double b;
#if defined(__HIP_DEVICE_COMPILE__)
    double r;
    __device__ explicit Recip(double x) : b(x), r(recip_refined(x)) {}
    __device__ double div(double a) const {
        const double q = a * r;
        return __builtin_amdgcn_div_fixup(__builtin_fma(__builtin_fma(-b, q, a), r, q), b, a);
    }
    __device__ double mul(double a) const { return a * r; }  // a / b to an ulp
#else
    __host__ __device__ explicit Recip(double x) : b(x) {}
    __host__ __device__ double div(double a) const { return a / b; }
    __host__ __device__ double mul(double a) const { return a / b; }
#endif
};

// reconstruct<Weno5Z> (Reconstruct.hpp:217-274) in FP64: the reference's
// operations in its order. Multiplying by a power of two is exact, so a
// product by 2, 4 or 1/4 and the add that follows it are one fma (14 of 85
// operations per cell and variable fewer); nothing else is fused.
template <typename S>
__host__ __device__ inline void weno5z_f64(const S& s, double& wL, double& wR) {
    constexpr double b0c = 13.0 / 12.0;
    constexpr double eps = 1e-36;  // Reconstruct.hpp:237-239
    const double sm2 = s(-2), sm1 = s(-1), s0 = s(0), sp1 = s(1), sp2 = s(2);
    const double s3 = 3.0 * s0, s5 = 5.0 * s0, s11 = 11.0 * s0;
    const double a0 = __builtin_fma(-2.0, sm1, sm2) + s0;
    const double a1 = __builtin_fma(-2.0, s0, sm1) + sp1;
    const double a2 = __builtin_fma(-2.0, sp1, s0) + sp2;
    const double c0 = __builtin_fma(-4.0, sm1, sm2) + s3;
    const double c1 = sm1 - sp1;
    const double c2 = __builtin_fma(-4.0, sp1, s3) + sp2;
    const double beta0 = __builtin_fma(0.25, c0 * c0, b0c * (a0 * a0));
    const double beta1 = __builtin_fma(0.25, c1 * c1, b0c * (a1 * a1));
    const double beta2 = __builtin_fma(0.25, c2 * c2, b0c * (a2 * a2));
    const double tau5 = __builtin_fabs(beta0 - beta2);
    const double ind0 = div_plain(tau5, beta0 + eps);
    const double ind1 = div_plain(tau5, beta1 + eps);
    const double ind2 = div_plain(tau5, beta2 + eps);
    const double q0 = 1.0 + ind0 * ind0;
    const double q1 = 1.0 + ind1 * ind1;
    const double q2 = 1.0 + ind2 * ind2;
    const double w1 = 6.0 * q1;
    {
        const double e0 = __builtin_fma(2.0, s0, 5.0 * sm1) - sm2;
        const double e1 = __builtin_fma(2.0, sm1, s5 - sp1);
        const double e2 = __builtin_fma(2.0, sp2, -(7.0 * sp1)) + s11;
        const double w0 = 3.0 * q0;
        wL = div_ieee(e0 * w0 + e1 * w1 + e2 * q2, 6.0 * (w0 + w1 + q2));
    }
    {
        const double e0 = __builtin_fma(2.0, s0, 5.0 * sp1) - sp2;
        const double e1 = __builtin_fma(2.0, sp1, s5 - sm1);
        const double e2 = __builtin_fma(2.0, sm2, -(7.0 * sm1)) + s11;
        const double w0 = 3.0 * q2;
        wR = div_ieee(e0 * w0 + e1 * w1 + e2 * q0, 6.0 * (w0 + w1 + q0));
    }
}

}  // namespace mh

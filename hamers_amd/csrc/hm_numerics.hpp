// hm_numerics.hpp -- pointwise numerics of the convective-flux RHS on the GPU.
//
// Every expression keeps the association order and reciprocal forms of the
// reference source lines it cites, so that a build without multiply-add
// contraction (-ffp-contract=off) rounds exactly as the reference's
// uncontracted x86-64 build does.  The knife-edge predicates of the scheme
// (R_tau > alpha_tau, s* > 0, sensor > 0.65, positivity) then take the same
// branch as the reference on identical inputs.
#pragma once

// Host+device so that host-side checks can compile the same pointwise code.
#if defined(__HIPCC__)
#include <hip/hip_runtime.h>
#define HM_HD __host__ __device__ __forceinline__
#else
#define HM_HD inline
#endif
#include <cmath>

namespace hm {

constexpr double kEps = 1.0e-15;  // HAMERS_EPSILON, include/HAMeRS_config.hpp.in:16

// The hardware reciprocal estimate.  A host build divides, unless it defines
// HM_RCP_ESTIMATE(b), an estimate of its own: then it follows the device's
// division step by step.
#if defined(__HIP_DEVICE_COMPILE__)
#define HM_RCP_ESTIMATE(b) __builtin_amdgcn_rcp(b)
#endif

// Correctly rounded FP64 division in fewer instructions than the compiler's
// general sequence, for operands whose quotient and remainder are normal
// numbers (every quotient of the scheme: denominators are state values or
// sums with a positive floor).  rcp_rn refines the hardware reciprocal
// estimate (relative error below 2^-24.3, measured) by one cubic Newton step
// r <- r + r (e + e^2), e = 1 - b r: the residual e^3 is below 2^-72, so it is
// as accurate as two quadratic steps (one FMA more) and the result is rounded
// once.  quot forms q0 = a r and returns q0 + r (a - b q0) with two FMAs
// (Markstein's correction, IBM J. Res. Develop. 34 (1990) 111-119), which
// rounds to the nearest FP64 number like a / b.  One reciprocal serves every
// quotient with the same denominator.  It skips the general sequence's range
// scaling and special-value fixup, so a zero dividend gives +0 for -0 and a
// zero divisor gives NaN; neither reaches a branch of the scheme.  Checked bit
// for bit against a / b on the GPU over 1e10 random operand pairs (exponents
// -80..79), on the host with a perturbed estimate over 2e7 pairs (all-ones
// significands and near-midpoint quotients included) and by the parity tests
// against the oracle's IEEE divisions.  Reciprocals of several denominators
// from one estimate of their product (each then 2 or 3 units off) gave other
// last places for significands of all ones and overflowed for indicators past
// 1e100; they saved 1 % of a right-hand side.
HM_HD double rcp_rn(double b) {
#if defined(HM_RCP_ESTIMATE)
    const double r = HM_RCP_ESTIMATE(b);
    const double e = fma(-b, r, 1.0);
    return fma(r, fma(e, e, e), r);
#else
    return double(1) / b;
#endif
}

HM_HD double quot(double a, double b, double r) {
#if defined(HM_RCP_ESTIMATE)
    const double q0 = a * r;
    return fma(fma(-b, q0, a), r, q0);
#else
    (void)r;
    return a / b;
#endif
}

// Reciprocal by two quadratic steps, for the adjoint's reverse sweep, which
// multiplies by it.  It equals rcp_rn except for a last place now and then; in
// stencils just above the indicators' rounding noise the sweep magnifies that
// to 1e-3 of the gradient of a random final adjoint.  Neither form is known to
// be the better one there; this one keeps the gradients as they were.
HM_HD double rcp_two(double b) {
#if defined(HM_RCP_ESTIMATE)
    double r = HM_RCP_ESTIMATE(b);
    double e = fma(-b, r, 1.0);
    r = fma(r, e, r);
    e = fma(-b, r, 1.0);
    return fma(r, e, r);
#else
    return double(1) / b;
#endif
}

HM_HD double div_rn(double a, double b) { return quot(a, b, rcp_rn(b)); }

// Whether cond holds on every active lane of the wavefront (host builds: cond).
HM_HD bool wave_all(bool cond) {
#if defined(__HIP_DEVICE_COMPILE__)
    return __builtin_amdgcn_ballot_w64(!cond) == 0;
#else
    return cond;
#endif
}

// ipow of ConvectiveFluxReconstructorWCNS6-LD-HLLC-HLL.cpp:9-18: repeated
// multiplication, so base^4 is ((b*b)*b)*b.  E < 0 means "exponent known only
// at run time".
template <int E>
HM_HD double rep_pow(double b, int e_rt) {
    if constexpr (E > 0) {
        double r = b;
#pragma unroll
        for (int i = 1; i < E; i++) r *= b;
        return r;
    } else {
        double r = b;
        for (int i = 1; i < e_rt; i++) r *= b;
        return r;
    }
}

// The six stencil values of one characteristic field at one face, cells
// i-3 .. i+2 of the face between cells i-1 and i.
struct Six {
    double v[6];
};

HM_HD Six flip(const Six& s) { return Six{{s.v[5], s.v[4], s.v[3], s.v[2], s.v[1], s.v[0]}}; }

// Smoothness indicators of the three 3-point sub-stencils
// (WCNS6-LD-HLLC-HLL.cpp:55-68, identical in WCNS5-JS-HLLC-HLL.cpp:32-44).  A
// product by a power of two is exact, so an FMA that takes it in rounds once,
// as the product and the sum do: the same bits in one instruction less.
HM_HD void beta3(const Six& s, double& b0, double& b1, double& b2) {
    b0 = double(1) / double(3) *
         (s.v[0] * (fma(double(4), s.v[0], -(double(19) * s.v[1])) + double(11) * s.v[2]) +
          s.v[1] * (double(25) * s.v[1] - double(31) * s.v[2]) + double(10) * s.v[2] * s.v[2]);
    b1 = double(1) / double(3) *
         fma(double(4), s.v[3] * s.v[3],
             s.v[1] * (fma(double(4), s.v[1], -(double(13) * s.v[2])) + double(5) * s.v[3]) +
                 double(13) * s.v[2] * (s.v[2] - s.v[3]));
    b2 = double(1) / double(3) *
         fma(double(4), s.v[4] * s.v[4],
             s.v[2] * (double(10) * s.v[2] - double(31) * s.v[3] + double(11) * s.v[4]) +
                 s.v[3] * (double(25) * s.v[3] - double(19) * s.v[4]));
}

// Six-point smoothness indicator (WCNS6-LD-HLLC-HLL.cpp:70-83).
HM_HD double beta6(const Six& s) {
    return double(1) / double(232243200) *
           (s.v[0] * (double(525910327) * s.v[0] - double(4562164630) * s.v[1] + double(7799501420) * s.v[2] -
                    double(6610694540) * s.v[3] + double(2794296070) * s.v[4] - double(472758974) * s.v[5]) +
            double(5) * s.v[1] *
                (double(2146987907) * s.v[1] - double(7722406988) * s.v[2] + double(6763559276) * s.v[3] -
                 double(2926461814) * s.v[4] + double(503766638) * s.v[5]) +
            double(20) * s.v[2] *
                (double(1833221603) * s.v[2] - double(3358664662) * s.v[3] + double(1495974539) * s.v[4] -
                 double(263126407) * s.v[5]) +
            double(20) * s.v[3] * (double(1607794163) * s.v[3] - double(1486026707) * s.v[4] + double(268747951) * s.v[5]) +
            double(5) * s.v[4] * (double(1432381427) * s.v[4] - double(536951582) * s.v[5]) +
            double(263126407) * s.v[5] * s.v[5]);
}

// Shock measure sigma (WCNS6-LD-HLLC-HLL.cpp:24-41); both sides use the
// unflipped stencil.
HM_HD double ld_sigma(const Six& s) {
    const double a1 = s.v[2] - s.v[1];
    const double a2 = s.v[3] - s.v[2];
    const double a3 = s.v[4] - s.v[3];
    const double t1 = div_rn(fabs(a1 - a2), fabs(a1) + fabs(a2) + kEps);
    const double t2 = div_rn(fabs(a2 - a3), fabs(a2) + fabs(a3) + kEps);
    return fmax(t1, t2);
}

// Scheme constants.  inv_thr: reciprocal of the ratio tau6 / (beta_k + eps)
// below which its q-th power vanishes in the sum C + ratio^q (ld_flat_limit);
// infinity: never.
struct LDConst {
    int p, q;
    double C, alpha_tau;
    double inv_thr = HUGE_VAL;
};

// LDConst::inv_thr of the constants (host).  With 0 <= x < half a unit in the
// last place of C, C + x rounds to C; then the four central weights are
// (C, 15 C, 15 C, C) / 32 over their sum.  Where those sums are exact the
// weights are 1/32, 15/32, 15/32, 1/32 to the bit.  R_tau is then below the
// same ratio (its denominator averages theirs), so it cannot exceed alpha_tau.
inline double ld_flat_limit(int q, double C, double alpha_tau) {
    const double never = HUGE_VAL;
    if (!(C >= 1.0 && C < 1.0e30) || q < 1) return never;
    const double s1 = C + 15.0 * C, s2 = s1 + 15.0 * C, s3 = s2 + C;
    if (C / s3 != 1.0 / 32.0 || 15.0 * C / s3 != 15.0 / 32.0) return never;
    const double half_ulp = std::ldexp(1.0, std::ilogb(C) - 53);
    const double thr = std::pow(half_ulp, 1.0 / q) * (1.0 - 1.0e-6);
    return thr > 0.0 && alpha_tau > 2.0 * thr ? 1.0 / thr : never;
}

// Midpoint value of one side from its stencil and the four weights.  .75 w is
// 2 (.375 w) to the bit and products by a power of two are exact (see beta3).
HM_HD double ld_combine(const Six& s, double w0, double w1, double w2, double w3) {
    const double a1 = double(3) / double(8) * w1, a2 = double(3) / double(8) * w2;
    return double(3) / double(8) * w0 * s.v[0] +
           fma(-double(1) / double(8), w1, -(double(10) / double(8) * w0)) * s.v[1] +
           (fma(double(2), a1, double(15) / double(8) * w0) + a2) * s.v[2] +
           (fma(double(2), a2, a1) + double(15) / double(8) * w3) * s.v[3] +
           fma(-double(1) / double(8), w2, -(double(10) / double(8) * w3)) * s.v[4] + double(3) / double(8) * w3 * s.v[5];
}

// One side of the WCNS6-LD nonlinear midpoint interpolation
// (WCNS6-LD-HLLC-HLL.cpp:133-223; the plus side 229-319 is this on flip(s)).
// The upwind weights u_k and the shock measure sigma enter only where the
// ratio R_tau = tau6 / (beta_avg + eps) exceeds alpha_tau, so they are formed
// only there (the same expressions, evaluated on demand): sigma of the
// unflipped stencil s0 is computed once per field, into sig (< 0: not yet).
// Where no lane of the wavefront has a ratio tau6 / (beta_k + eps) that
// reaches the sum C + ratio^q (resolved data: 30-50 % of the wavefronts of
// shear layers, mixing layers and smooth modes), the weights are constants and
// every quotient is left out.  Factors that are powers of two scale exactly:
// 1/32 of the outer central weights and 1/16 of the first upwind one are taken
// into the sum as an FMA (left out, the sums would overflow before the
// reference's do), 1/8 of beta_avg into the next operation.
template <int P, int Q>
HM_HD double ld_side(const Six& s, const Six& s0, double& sig, const LDConst& k) {
    double b0, b1, b2;
    beta3(s, b0, b1, b2);
    const double b3 = beta6(s);

    // e_k = b_k + eps divides both tau5 and tau6: one reciprocal each.
    const double e0 = b0 + kEps, e1 = b1 + kEps, e2 = b2 + kEps, e3 = b3 + kEps;
    const double b8 = b0 + b2 + double(6) * b1;  // 8 beta_avg
    const double tau6 = fabs(fma(-double(1) / double(8), b8, b3));

    const double lim = tau6 * k.inv_thr;
    if (wave_all(lim < e1)) {
        if (wave_all(lim < e0 && lim < e2 && lim < e3))
            return double(3) / double(256) * s.v[0] - double(25) / double(256) * s.v[1] +
                   double(150) / double(256) * s.v[2] + double(150) / double(256) * s.v[3] -
                   double(25) / double(256) * s.v[4] + double(3) / double(256) * s.v[5];
    }

    const double r0 = rcp_rn(e0), r1 = rcp_rn(e1), r2 = rcp_rn(e2);
    const double c32 = double(1) / double(32) * k.C;
    double w0 = fma(double(1) / double(32), rep_pow<Q>(quot(tau6, e0, r0), k.q), c32);
    double w1 = double(15) / double(32) * (k.C + rep_pow<Q>(quot(tau6, e1, r1), k.q));
    double w2 = double(15) / double(32) * (k.C + rep_pow<Q>(quot(tau6, e2, r2), k.q));
    double w3 = fma(double(1) / double(32), rep_pow<Q>(div_rn(tau6, e3), k.q), c32);
    const double ws = w0 + w1 + w2 + w3;
    const double rws = rcp_rn(ws);
    w0 = quot(w0, ws, rws);
    w1 = quot(w1, ws, rws);
    w2 = quot(w2, ws, rws);
    w3 = quot(w3, ws, rws);

    // RN(tau6 / den) > alpha_tau: the sign of tau6 - alpha_tau den is exact in
    // an FMA, and decides unless the two are within rounding of each other
    // (then, and for den <= 0, the quotient itself is formed).
    const double den = fma(double(1) / double(8), b8, kEps);  // beta_avg + eps
    const double over = fma(-k.alpha_tau, den, tau6);
    if (over > double(0) || !(den > double(0))) {
        if ((den > double(0) && over > double(8.8817841970012523e-16) * tau6) || div_rn(tau6, den) > k.alpha_tau) {
            const double tau5 = fabs(b0 - b2);
            double u0 = fma(double(1) / double(16), rep_pow<P>(quot(tau5, e0, r0), k.p), double(1) / double(16));
            double u1 = double(5) / double(8) * (double(1) + rep_pow<P>(quot(tau5, e1, r1), k.p));
            double u2 = double(5) / double(16) * (double(1) + rep_pow<P>(quot(tau5, e2, r2), k.p));
            const double us = u0 + u1 + u2;
            const double rus = rcp_rn(us);
            u0 = quot(u0, us, rus);
            u1 = quot(u1, us, rus);
            u2 = quot(u2, us, rus);
            if (sig < double(0)) sig = ld_sigma(s0);
            const double sigma = sig;
            w0 = sigma * u0 + (double(1) - sigma) * w0;
            w1 = sigma * u1 + (double(1) - sigma) * w1;
            w2 = sigma * u2 + (double(1) - sigma) * w2;
            w3 = (double(1) - sigma) * w3;
        }
    }
    return ld_combine(s, w0, w1, w2, w3);
}

// One side of WCNS5-JS (WCNS5-JS-HLLC-HLL.cpp:78-118; plus side 124-164 on
// flip(s)).
template <int P>
HM_HD double js_side(const Six& s, int p_rt) {
    double b0, b1, b2;
    beta3(s, b0, b1, b2);
    double w0 = div_rn(double(1.0) / double(16), rep_pow<P>((b0 + kEps), p_rt));
    double w1 = div_rn(double(5.0) / double(8), rep_pow<P>((b1 + kEps), p_rt));
    double w2 = div_rn(double(5.0) / double(16), rep_pow<P>((b2 + kEps), p_rt));
    const double ws = w0 + w1 + w2;
    const double rws = rcp_rn(ws);
    w0 = quot(w0, ws, rws);
    w1 = quot(w1, ws, rws);
    w2 = quot(w2, ws, rws);
    const double a1 = double(3) / double(8) * w1;
    return fma(-double(1) / double(8), w2 * s.v[4],
               double(3) / double(8) * w0 * s.v[0] +
                   fma(-double(1) / double(8), w1, -(double(10) / double(8) * w0)) * s.v[1] +
                   (fma(double(2), a1, double(15) / double(8) * w0) + double(3) / double(8) * w2) * s.v[2] +
                   (a1 + double(6) / double(8) * w2) * s.v[3]);
}

// Scheme selector: both sides of one characteristic field.
enum { kWCNS5_JS = 0, kWCNS6_LD = 1 };

template <int SCHEME, int P, int Q>
HM_HD void reconstruct_pair(const Six& s, const LDConst& k, double& um, double& up) {
    if constexpr (SCHEME == kWCNS6_LD) {
        double sig = double(-1);  // sigma >= 0, formed on the first side that blends
        // The two sides one after the other, kept apart from each other in
        // the schedule, so that only one side's indicators and weights are
        // live at a time (a runtime loop over the sides would select each
        // stencil value by the side: 24 moves per field).
        um = ld_side<P, Q>(s, s, sig, k);
        Six t = s;
#if defined(__HIP_DEVICE_COMPILE__)
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int m = 0; m < 6; m++) asm("" : "+v"(t.v[m]));
#endif
        up = ld_side<P, Q>(flip(t), t, sig, k);
    } else {
        um = js_side<P>(s, k.p);
        up = js_side<P>(flip(s), k.p);
    }
}

}  // namespace hm

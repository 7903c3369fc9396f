// Host check of hm_numerics.hpp: the midpoint values of one field against the
// reference's formulas written out term by term (WCNS6-LD-HLLC-HLL.cpp:24-223,
// WCNS5-JS-HLLC-HLL.cpp:32-118; no fused multiply-add, no constant weights),
// bit for bit, over stencils from rough to resolved and over scheme constants
// that do and do not admit the constant-weight rule, with the exponents at
// compile time and at run time.  Prints the number of differing values and how
// often the rule held; exits 1 on any difference.
//
// Built with -DDEVICE_DIVISION it runs the device's division instead of the
// host's: reciprocals refined from an estimate that is off by up to 2^-24.3
// either way (the bound measured on gfx950) and quotients corrected by FMAs.
// That division is checked by itself too, against a / b.
#include <cmath>
#include <cstdint>
#include <cstdio>
#include <cstring>

#if defined(DEVICE_DIVISION)
static uint64_t estimate_state = 0x9e3779b97f4a7c15ull;
static double estimate(double b) {
    estimate_state ^= estimate_state << 13;
    estimate_state ^= estimate_state >> 7;
    estimate_state ^= estimate_state << 17;
    const double off = 2.0 * (double(estimate_state >> 11) / 9007199254740992.0) - 1.0;
    return 1.0 / b * (1.0 + off * 4.84e-8);  // 2^-24.3 = 4.84e-8
}
#define HM_RCP_ESTIMATE(b) estimate(b)
#endif
#include "../hamers_amd/csrc/hm_numerics.hpp"

using namespace hm;

static uint64_t state = 88172645463325252ull;
static double rnd() {
    state ^= state << 13;
    state ^= state >> 7;
    state ^= state << 17;
    return 2.0 * (double(state >> 11) / 9007199254740992.0) - 1.0;
}

static double ipow(double b, int e) {
    double r = b;
    for (int i = 1; i < e; i++) r *= b;
    return r;
}

static void betas(const double* u, double* b) {
    b[0] = 1.0 / 3.0 * (u[0] * (4.0 * u[0] - 19.0 * u[1] + 11.0 * u[2]) + u[1] * (25.0 * u[1] - 31.0 * u[2]) + 10.0 * u[2] * u[2]);
    b[1] = 1.0 / 3.0 * (u[1] * (4.0 * u[1] - 13.0 * u[2] + 5.0 * u[3]) + 13.0 * u[2] * (u[2] - u[3]) + 4.0 * u[3] * u[3]);
    b[2] = 1.0 / 3.0 * (u[2] * (10.0 * u[2] - 31.0 * u[3] + 11.0 * u[4]) + u[3] * (25.0 * u[3] - 19.0 * u[4]) + 4.0 * u[4] * u[4]);
}

static double sum_terms(const double* u, const double* w) {
    return 3.0 / 8.0 * w[0] * u[0] + (-10.0 / 8.0 * w[0] - 1.0 / 8.0 * w[1]) * u[1] +
           (15.0 / 8.0 * w[0] + 6.0 / 8.0 * w[1] + 3.0 / 8.0 * w[2]) * u[2] +
           (3.0 / 8.0 * w[1] + 6.0 / 8.0 * w[2] + 15.0 / 8.0 * w[3]) * u[3] +
           (-1.0 / 8.0 * w[2] - 10.0 / 8.0 * w[3]) * u[4] + 3.0 / 8.0 * w[3] * u[5];
}

static double plain_ld(const double* u, double sigma, const LDConst& k) {
    double b[4], w[4], v[3];
    betas(u, b);
    Six s;
    std::memcpy(s.v, u, sizeof s.v);
    b[3] = beta6(s);
    const double avg = 1.0 / 8.0 * (b[0] + b[2] + 6.0 * b[1]), tau6 = std::fabs(b[3] - avg);
    const double d[4] = {1.0 / 32.0, 15.0 / 32.0, 15.0 / 32.0, 1.0 / 32.0}, e[3] = {1.0 / 16.0, 5.0 / 8.0, 5.0 / 16.0};
    for (int i = 0; i < 4; i++) w[i] = d[i] * (k.C + ipow(tau6 / (b[i] + kEps), k.q));
    const double ws = w[0] + w[1] + w[2] + w[3];
    for (int i = 0; i < 4; i++) w[i] = w[i] / ws;
    if (tau6 / (avg + kEps) > k.alpha_tau) {
        const double tau5 = std::fabs(b[0] - b[2]);
        for (int i = 0; i < 3; i++) v[i] = e[i] * (1.0 + ipow(tau5 / (b[i] + kEps), k.p));
        const double vs = v[0] + v[1] + v[2];
        for (int i = 0; i < 3; i++) w[i] = sigma * (v[i] / vs) + (1.0 - sigma) * w[i];
        w[3] = (1.0 - sigma) * w[3];
    }
    return sum_terms(u, w);
}

static double plain_js(const double* u, int p) {
    double b[3], w[4] = {0, 0, 0, 0};
    betas(u, b);
    const double d[3] = {1.0 / 16.0, 5.0 / 8.0, 5.0 / 16.0};
    for (int i = 0; i < 3; i++) w[i] = d[i] / ipow(b[i] + kEps, p);
    const double ws = w[0] + w[1] + w[2];
    for (int i = 0; i < 3; i++) w[i] /= ws;
    return 3.0 / 8.0 * w[0] * u[0] + (-10.0 / 8.0 * w[0] - 1.0 / 8.0 * w[1]) * u[1] +
           (15.0 / 8.0 * w[0] + 6.0 / 8.0 * w[1] + 3.0 / 8.0 * w[2]) * u[2] + (3.0 / 8.0 * w[1] + 6.0 / 8.0 * w[2]) * u[3] -
           1.0 / 8.0 * w[2] * u[4];
}

static bool differs(double a, double b) { return std::memcmp(&a, &b, 8) != 0 && !(a != a && b != b); }

// Both sides of a field against the plain values pm, pp.
template <int SCHEME, int P, int Q>
static int wrong(const Six& s, const LDConst& k, double pm, double pp) {
    double um, up;
    reconstruct_pair<SCHEME, P, Q>(s, k, um, up);
    return differs(um, pm) + differs(up, pp);
}

#if defined(DEVICE_DIVISION)
// A positive number of random exponent in [-range, range]; a quarter of them
// with all ones below the leading bits, or nearly so.
static double operand(int range) {
    double m = 1.0 + 0.5 * (rnd() + 1.0);
    uint64_t b;
    std::memcpy(&b, &m, 8);
    const int how = int(state >> 40) & 7;
    if (how == 0) b |= (uint64_t(1) << 52) - 1;
    if (how == 1) b |= (uint64_t(1) << 50) - 1, b ^= (state >> 20) & 3;
    std::memcpy(&m, &b, 8);
    return std::ldexp(m, int(range * rnd()));
}

// The quotient by a refined reciprocal is a / b to the last place, all-ones
// significands and quotients made to lie next to the midpoint of two numbers
// (a within half a unit of b times it) among them.
static int check_division() {
    long bad = 0;
    const long count = 10000000;
    for (long it = 0; it < count; it++) {
        const int range = it % 2 ? 60 : 420;
        const double a = operand(range), b = operand(range), q = operand(3);
        bad += differs(quot(a, b, rcp_rn(b)), a / b);
        const double near = double(((long double)q + 0.5L * (std::nextafter(q, 1e300) - q)) * b);
        bad += differs(div_rn(near, b), near / b);
    }
    std::printf("division: %ld of %ld quotients differ\n", bad, 2 * count);
    return bad != 0;
}
#endif

int main() {
#if defined(DEVICE_DIVISION)
    if (check_division()) return 1;
#endif
    struct Set {
        int p, q;
        double C, alpha;
    };
    const Set sets[] = {{2, 4, 1e9, 35.0}, {2, 4, 1e3, 35.0}, {2, 4, 1.0, 35.0}, {3, 1, 1e9, 35.0}, {1, 8, 1e6, 2.0},
                        {2, 4, 123456789.123, 35.0}, {2, 4, 1e9, 1e-3}, {2, 4, 1e9, -1.0}, {2, 4, 1e31, 35.0}, {2, 4, 0.0, 35.0}};
    long bad = 0, total = 0;
    for (const Set& c : sets) {
        LDConst k{c.p, c.q, c.C, c.alpha, ld_flat_limit(c.q, c.C, c.alpha)};
        const bool off = !(k.inv_thr < HUGE_VAL);
        long flat = 0;
        for (int it = 0; it < 200000; it++) {
            // polynomial data of a random resolution, noise of a random size and offset
            const double h = std::pow(10.0, -3.0 * std::fabs(rnd())), noise = it % 3 ? std::pow(10.0, -16.0 * std::fabs(rnd())) : 0.0;
            const double off0 = it % 5 ? rnd() : 0.0, a1 = rnd(), a2 = rnd(), a3 = rnd();
            // (indicators of 1e120 and 1e156: no product of two of them, or of their squares, is a number)
            const double scale = it % 7 == 0 ? 1e8 : it % 77 == 1 ? 1e60 : it % 77 == 2 ? 1e78 : 1.0;
            Six s;
            for (int m = 0; m < 6; m++) {
                const double x = (m - 2.5) * h;
                s.v[m] = scale * (off0 + a1 * x + a2 * x * x + a3 * x * x * x * x * x + noise * rnd());
            }
            double r[6];
            for (int m = 0; m < 6; m++) r[m] = s.v[5 - m];
            const double sigma = ld_sigma(s);
            const double lm = plain_ld(s.v, sigma, k), lp = plain_ld(r, sigma, k);
            bad += wrong<kWCNS6_LD, -1, -1>(s, k, lm, lp);
            if (c.p == 2 && c.q == 4) bad += wrong<kWCNS6_LD, 2, 4>(s, k, lm, lp);
            total += c.p == 2 && c.q == 4 ? 4 : 2;
            double b[3];
            betas(s.v, b);
            const double tau6 = std::fabs(beta6(s) - 1.0 / 8.0 * (b[0] + b[2] + 6.0 * b[1]));
            flat += tau6 * k.inv_thr < b[1] + kEps;
            if (scale < 1e70) {  // (squares of the indicators are beyond the numbers there)
                const double jm = plain_js(s.v, c.p), jp = plain_js(r, c.p);
                bad += wrong<kWCNS5_JS, -1, -1>(s, k, jm, jp);
                if (c.p == 2) bad += wrong<kWCNS5_JS, 2, 4>(s, k, jm, jp);
                total += c.p == 2 ? 4 : 2;
            }
        }
        // powers up to the largest number: one jump beside equal values (differing floors only)
        for (double a = 1e10; a < 1e60; a *= 1.02) {
            const double u[6] = {0, 0, 0, 0, 0, a}, r[6] = {a, 0, 0, 0, 0, 0};
            Six s;
            std::memcpy(s.v, u, sizeof s.v);
            const double sigma = ld_sigma(s), lm = plain_ld(u, sigma, k), lp = plain_ld(r, sigma, k);
            bad += wrong<kWCNS6_LD, -1, -1>(s, k, lm, lp);
            if (c.p == 2 && c.q == 4) bad += wrong<kWCNS6_LD, 2, 4>(s, k, lm, lp);
            total += c.p == 2 && c.q == 4 ? 4 : 2;
        }
        std::printf("p %d q %d C %g alpha %g: rule %s, held about %ld times\n", c.p, c.q, c.C, c.alpha, off ? "off" : "on", flat);
        const bool expect_off = c.C == 1e31 || c.C == 0.0 || c.alpha < 0.01;
        if (off != expect_off || (!off && flat == 0)) {
            std::printf("rule: unexpected\n");
            return 1;
        }
    }
    std::printf("%ld of %ld values differ\n", bad, total);
    return bad != 0;
}

// Host check of hm_numerics.hpp: the midpoint values of one field against the
// reference's formulas written out term by term (WCNS6-LD-HLLC-HLL.cpp:24-223,
// WCNS5-JS-HLLC-HLL.cpp:32-118; no fused multiply-add, no constant weights),
// bit for bit, over stencils from rough to resolved and over scheme constants
// that do and do not admit the constant-weight rule.  Prints the number of
// differing values and how often the rule held; exits 1 on any difference.
#include <cstdint>
#include <cstdio>
#include <cstring>

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

int main() {
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
            const double off0 = it % 5 ? rnd() : 0.0, a1 = rnd(), a2 = rnd(), a3 = rnd(), scale = it % 7 ? 1.0 : 1e8;
            Six s;
            for (int m = 0; m < 6; m++) {
                const double x = (m - 2.5) * h;
                s.v[m] = scale * (off0 + a1 * x + a2 * x * x + a3 * x * x * x * x * x + noise * rnd());
            }
            double um, up, pm, pp;
            reconstruct_pair<kWCNS6_LD, -1, -1>(s, k, um, up);
            double r[6];
            for (int m = 0; m < 6; m++) r[m] = s.v[5 - m];
            pm = plain_ld(s.v, ld_sigma(s), k);
            pp = plain_ld(r, ld_sigma(s), k);
            bad += std::memcmp(&um, &pm, 8) != 0;
            bad += std::memcmp(&up, &pp, 8) != 0;
            double b[3];
            betas(s.v, b);
            const double tau6 = std::fabs(beta6(s) - 1.0 / 8.0 * (b[0] + b[2] + 6.0 * b[1]));
            flat += tau6 * k.inv_thr < b[1] + kEps;
            reconstruct_pair<kWCNS5_JS, -1, -1>(s, k, um, up);
            pm = plain_js(s.v, c.p);
            pp = plain_js(r, c.p);
            bad += std::memcmp(&um, &pm, 8) != 0;
            bad += std::memcmp(&up, &pp, 8) != 0;
            total += 4;
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

// Host-side check of fast_setup (pp_pmt_bounds.h): what it admits, its relative error
// bound covers. The approximate weight of an antipode is taken with its partner's
// direction turned round, so that directions which are not quite opposite change the
// weight; in 64 bits, that change alone may not exceed f.rel.
// Built by tests/test_pmt_bounds_host.py.
//   usage: pmt_bounds_check <sigma1> <sigma2> <shift>
//   prints: set-ups tried, admitted, the largest (relative change / f.rel)
#include <cstdio>
#include <cstdlib>
#include <random>

#include "../../photonpropagation.jl_amd/csrc/pp_pmt_bounds.h"

using namespace pp;

static double log_weight(const double p[3], const double d[3], double k) {
    const double c = p[0] * d[0] + p[1] * d[1] + p[2] * d[2];
    const double pt = std::acos(std::min(c, 1.0));
    return -k * pt * pt + (pt > 0.0 ? std::log(pt / std::sin(pt)) : 0.0);
}

int main(int argc, char** argv) {
    if (argc < 4) return 2;
    const float sigma[2] = {(float)atof(argv[1]), (float)atof(argv[2])};
    const float shift = (float)atof(argv[3]);
    std::mt19937_64 rng(7);
    std::uniform_real_distribution<double> U(-1.0, 1.0);
    double th[kPmts], ph[kPmts];
    pom_angles(th, ph);
    long tried = 0, admitted = 0;
    double worst = 0.0;
    for (int trial = 0; trial < 50; ++trial) {
        // a rotation about a random axis
        double a[3], l = 0.0;
        for (double& x : a) x = U(rng);
        for (double x : a) l += x * x;
        for (double& x : a) x /= std::sqrt(l);
        const double w = 3.1 * U(rng), cw = std::cos(w), sw = std::sin(w);
        PmtSetup s{};
        s.acc_ok = true;
        for (int g = 0; g < 2; ++g) s.inv_s2[g] = 1.0f / (sigma[g] * sigma[g]);
        for (int j = 0; j < kPmts; ++j) {
            const double v[3] = {std::sin(th[j]) * std::cos(ph[j]), std::sin(th[j]) * std::sin(ph[j]),
                                 std::cos(th[j])};
            const double av = a[0] * v[0] + a[1] * v[1] + a[2] * v[2];
            const double x[3] = {a[1] * v[2] - a[2] * v[1], a[2] * v[0] - a[0] * v[2],
                                 a[0] * v[1] - a[1] * v[0]};
            for (int r = 0; r < 3; ++r)
                s.dir[j][r] = (float)(cw * v[r] + sw * x[r] + (1.0 - cw) * av * a[r]);
        }
        for (int j = 0; j < 8; ++j)
            for (int r = 0; r < 3; ++r) s.dir[kAntipode[j]][r] += shift * (U(rng) < 0.0 ? -1.0f : 1.0f);
        PmtFast f{};
        ++tried;
        if (!fast_setup(s, &f)) continue;
        ++admitted;
        for (int j = 0; j < 8; ++j) {
            const double k = 0.5 * s.inv_s2[(j >> 2) & 1];
            double own[3], turned[3];
            for (int r = 0; r < 3; ++r) {
                own[r] = s.dir[kAntipode[j]][r];
                turned[r] = -(double)s.dir[j][r];
            }
            for (int i = 0; i < 2000; ++i) {  // positions on the antipode's hemisphere
                double p[3], n = 0.0;
                for (double& x : p) x = U(rng);
                for (double x : p) n += x * x;
                if (n > 1.0 || n < 1e-3) continue;
                const double side = p[0] * own[0] + p[1] * own[1] + p[2] * own[2] < 0.0 ? -1.0 : 1.0;
                for (double& x : p) x *= side / std::sqrt(n);
                const double e = std::fabs(std::expm1(log_weight(p, turned, k) - log_weight(p, own, k)));
                worst = std::max(worst, e / f.rel);
            }
        }
    }
    std::printf("%ld %ld %.6f\n", tried, admitted, worst);
    return 0;
}

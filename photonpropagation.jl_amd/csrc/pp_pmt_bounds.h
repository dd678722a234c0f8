// pp_pmt_bounds.h - geometry of the POM's PMTs and the error bounds of the PMT
// detection kernel's approximate weights (pp_pmt.hip). Host code only.
#pragma once

#include <algorithm>
#include <cmath>

#include "pp_hits.h"

namespace pp {

constexpr int kPmts = 16;
// PMT group of PMT j (src/pom.jl:172-174): PMTs 0-3 and 8-11 (25 deg from the
// equator) are group 1, 4-7 and 12-15 (57.5 deg) group 2: index (j >> 2) & 1

// PMT (theta, phi) of the POM, src/pom.jl:108-128
inline void pom_angles(double th[kPmts], double ph[kPmts]) {
    const double d2r = M_PI / 180.0;
    for (int k = 0; k < 4; ++k) {
        th[k] = (90.0 - 25.0) * d2r;
        ph[k] = k * M_PI / 2;
        th[4 + k] = (90.0 - 57.5) * d2r;
        ph[4 + k] = M_PI / 4 + k * M_PI / 2;
        th[8 + k] = (90.0 + 25.0) * d2r;
        th[12 + k] = (90.0 + 57.5) * d2r;
    }
    const double lower2[4] = {M_PI / 2, 0.0, 3 * M_PI / 2, M_PI};
    const double lower[4] = {M_PI / 4, 7 * M_PI / 4, 5 * M_PI / 4, 3 * M_PI / 4};
    for (int k = 0; k < 4; ++k) {
        ph[8 + k] = lower2[k];
        ph[12 + k] = lower[k];
    }
}

// The 16 PMT directions are 8 antipodal pairs of one group each: PMT j and
// kAntipode[j], j < 8 (the layout of pom_angles; fast_setup checks it).
constexpr int kAntipode[8] = {11, 10, 9, 8, 14, 13, 12, 15};

// Constants of the approximate weights (pmt_fast) of a set-up; false where they
// do not serve: a module orientation that is not a rotation (or reflection) to
// 1e-5, a negative acceptance, or widths whose error bounds leave too much to
// evaluate in full (sigma below 0.030 or above 0.347). With k = 1 / (2 sigma^2), a
// weight's relative error has three parts: the cosine times d ln p / dc <= pi k + 2;
// the fit of acos, 2e-7 times 1 + 2 k pt^2 <= 1 + 5 k; and 1e-5 for the roundings of
// both evaluations. The cosine is off by 2.5e-7 at most in either evaluation and by
// what a pair's directions fall short of opposite ones, since the approximate weight
// of an antipode is taken with its partner's direction.
// Per unit of acceptance a group's weight is at most scale, at its PMTs' axes,
// and falls with the angle. The near weights of both groups, each in units of its
// own largest, add up to at most 1.1455 for widths up to 0.3 and 1.7101 up to
// 0.4 (the sum grows with either width; the largest value over the sphere, at
// 0.075 degree steps), so that no position's sum exceeds that times the larger
// group's acceptance x scale: reach, with 1% to spare.
inline bool fast_setup(const PmtSetup& s, PmtFast* f) {
    if (!s.acc_ok) return false;
    double apart = 0.0;
    for (int j = 0; j < 8; ++j) {
        double d2 = 0.0;
        for (int r = 0; r < 3; ++r) {
            const double d = (double)s.dir[j][r] + s.dir[kAntipode[j]][r];
            if (!(std::fabs(d) <= 1e-6)) return false;
            d2 += d * d;
        }
        apart = std::max(apart, std::sqrt(d2));
    }
    double th[kPmts], ph[kPmts];
    pom_angles(th, ph);
    for (int j = 0; j < 8; ++j)
        for (int k = 0; k <= j; ++k) {
            double want = std::cos(th[j]) * std::cos(th[k]) +
                          std::sin(th[j]) * std::sin(th[k]) * std::cos(ph[j] - ph[k]);
            for (int r = 0; r < 3; ++r) want -= (double)s.dir[j][r] * s.dir[k][r];
            if (!(std::fabs(want) <= 1e-5)) return false;
        }
    const float width = std::max(1.0f / std::sqrt(s.inv_s2[0]), 1.0f / std::sqrt(s.inv_s2[1]));
    if (!(width <= 0.4f)) return false;
    f->rel = 0.0f;
    for (int g = 0; g < 2; ++g) {
        const double k = 0.5 * s.inv_s2[g];
        f->k2[g] = (float)(-k * 1.4426950408889634);
        f->scale[g] = s.inv_s2[g] * 0.25f;
        f->reach[g] = f->scale[g] * (width <= 0.3f ? 1.16f : 1.73f);
        f->rel = std::max(f->rel, (float)((2.5e-7 + apart) * (M_PI * k + 2.0) +
                                          2e-7 * (1.0 + 5.0 * k) + 1e-5));
        // four far PMTs a group, each at most pt exp(-k pt^2) / sin(pt) per unit
        // of scale and acceptance: up to 3 pi/4, and from there to the pole that
        // is left out (sin pt >= 1.41e-3)
        const double most = std::max(3.34 * std::exp(-2.467 * k), 2222.0 * std::exp(-5.55 * k));
        f->far[g] = (float)(4.0 * 0.25 * s.inv_s2[g] * most);
    }
    return f->rel <= 1e-3f && f->far[0] <= 1e-3f && f->far[1] <= 1e-3f;
}

}  // namespace pp

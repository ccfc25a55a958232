// The automatic skin of candidate lists that steps run on (host-only C++, no HIP): which skin the next build should take,
// from what the lists in force show of their gaps and of the speed.
#pragma once

#include <algorithm>
#include <cmath>
#include <cstdint>

namespace deme_int {

constexpr uint32_t SKIN_BUCKETS = 16;
// The automatic skin's widest value (mean radii), and the steps that lists have to last: those that die sooner at the
// widest skin give way to the cell sweep.
constexpr double SKIN_WIDEST = 0.8;
constexpr double SKIN_MIN_LIFE = 4.0;

// Seconds of a step on k candidates and of a build, fitted to 600 spheres to 1M clumps: the launches, then 70 ps a
// candidate; a build some 25 launches and three waits, then about three steps over its candidates.
inline double direct_step_s(double k) { return 14e-6 + 70e-12 * k; }
inline double direct_build_s(double k) { return 300e-6 + 3.0 * 70e-12 * k; }

struct SkinView {
    double skin, meanRadius;
    double nCand;          // candidates of the lists in force
    const uint32_t* gaps;  // a sample of their gaps, in sixteenths of the skin
    double move;           // the largest displacement of a step
    double least;          // thinner skins are not kept (the build positions' unit)
};
struct SkinChoice {
    double skin;
    double ratio;  // its candidates over the current lists'
    double life;   // steps its lists last
};

// The smallest time per step, builds included, among the skins whose lists last SKIN_MIN_LIFE steps; a build comes every
// time the fastest sphere moves half the skin. In view are sixteenths of the current skin, itself, and 1.25 and 1.5 times
// it. Where none of them lasts -- a calm system made fast, its lists thin -- the wider ones up to SKIN_WIDEST are looked
// at too, and the widest is taken where none lasts at all: a list that lives a step costs a build at any skin, so the
// thinnest would look cheapest, and neither a wider skin nor the cell sweep would ever be tried.
// (1M clumps moving at 0.02 m/s: 0.2 r lists 4.95M candidates, 343 us a step; the skin chosen 2.98M, 247 to 288 us.)
inline SkinChoice choose_skin(const SkinView& v) {
    const double s = v.skin, m = v.meanRadius, widest = SKIN_WIDEST * m;
    auto life = [&](double skin) { return 0.5 * skin / v.move; };
    SkinChoice best{s, 1.0, life(s)};
    double total = 0.0;
    for (uint32_t k = 0; k < SKIN_BUCKETS; k++) total += v.gaps[k];
    if (!(total > 0.0) || !std::isfinite(v.move) || !(v.move > 0.0)) return best;
    double bestCost = INFINITY;
    auto look = [&](double skin, double ratio) {
        const double L = life(skin);
        if (L < SKIN_MIN_LIFE) return;
        const double cost = direct_step_s(ratio * v.nCand) + direct_build_s(ratio * v.nCand) / L;
        if (cost < bestCost) {
            bestCost = cost;
            best = {skin, ratio, L};
        }
    };
    look(s, 1.0);
    double below = 0.0;
    for (uint32_t j = 1; j < SKIN_BUCKETS; j++) {
        below += v.gaps[j - 1] / total;
        const double skin = s * j / SKIN_BUCKETS;
        if (skin >= std::max(0.01 * m, v.least)) look(skin, below);
    }
    // beyond the skin the lists say nothing: the count grows on as over their last quarter, somewhat faster, and with the
    // area of the shell
    double last = 0.0;
    for (uint32_t j = SKIN_BUCKETS - SKIN_BUCKETS / 4; j < SKIN_BUCKETS; j++) last += v.gaps[j] / total;
    auto beyond = [&](double skin) {
        const double shell = (2.0 * m + skin) / (2.0 * m + s);
        return 1.0 + last * (skin - s) / (0.25 * s) * std::max(1.2, 0.5 * (1.0 + shell * shell));
    };
    for (int q = 1; q <= 2; q++) {
        const double skin = s * (1.0 + 0.25 * q);
        if (skin <= widest) look(skin, beyond(skin));
    }
    if (bestCost < INFINITY) return best;
    for (double skin = 1.25 * 1.5 * s; skin < widest; skin *= 1.25) look(skin, beyond(skin));
    if (s < widest) look(widest, beyond(widest));
    if (bestCost < INFINITY || s >= widest) return best;
    return {widest, beyond(widest), life(widest)};
}

}  // namespace deme_int

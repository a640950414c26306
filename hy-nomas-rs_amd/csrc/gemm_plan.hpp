// Which GEMM kernel and tile height a forward takes (host code, no device
// state: a function of the sizes alone).
//
// gemm_mfma's 256 x 256 tiles reach the chip's matrix rate once there are
// enough of them; gemm_rows' 16 / 32 / 64 x 64 tiles spread small problems
// over all CUs and stream weights for few rows.  The choice is the least
// estimated time of each GEMM, from what both kernels measured
// on one MI355X (stage times, weights in the last-level cache, expert widths
// 64 x 128 to 1536 x 4096, 1 to 8,192 rows, 1 to 64 experts):
//  - gemm_mfma: 4 us (f32: 15 us, the first fetch of its code), and for each
//    round of 256 tiles 16 us plus 0.58 us per k step (f32: 45 us plus 1.7 us
//    per 16 k); past one round, 0.75 of a round for the last, uneven one; 10 us
//    (f32: 20 us) for the partial sums where tiles are split along K.
//  - gemm_rows: 5 us, per k step of one tile 0.05 / 0.06 / 0.07 us for 16 / 32 /
//    64 rows (f32: 0.13 / 0.16 / 0.23), and per tile, with the chip full, 3.8 +
//    0.27 kt / 5 + 0.31 kt / 5.3 + 0.47 kt ns for kt k steps (f32: 12 + 0.25 kt /
//    7.5 + 0.44 kt / 8 + 0.8 kt).  64-row tiles take two waves instead of four
//    once there are 400 (f32: 700) of them (up to 1.35 times faster there).
// Over 70 drawn calls (both GEMMs, each choice timed) the picks take 2.3% more
// time than the best ones would, the worst of them 15 us or more 1.56 times.
// The two GEMMs choose on their own, each with its tile table: 1,111 rows of
// 1000 x 2667, 6 experts, in bf16 take 36 + 53 us on gemm_mfma, 64 + 35 us on
// 64-row tiles, 36 + 35 us on one of each.  Where the two meet either is within
// 15% of the other.
#pragma once

#include <algorithm>

#include "kernels.hpp"

namespace nomas {

// gemm_rows' smaller tiles are taken up to these mean rows per expert
constexpr int kRows16Mean = 1024, kRows32Mean = 2048;

// GEMM tiles that a tile table must hold for A routed rows (or fewer) over E
// experts, whatever gemm_plan picks.
inline int64_t max_gemm_tiles(int64_t A, int64_t E) {
    const int64_t small = std::max(std::min(A, kRows16Mean * E) / 16, std::min(A, kRows32Mean * E) / 32);
    return std::max((A + 63) / 64, small + 1) + E;
}

// A routed rows over E experts; Dk and Hp are the padded widths of D and H.
inline GemmPlan gemm_plan(DType dt, int64_t A, int64_t E, int64_t Dk, int64_t Hp, int64_t D, int64_t H) {
    // padded widths keep one order of summation at any row count: one wave
    const bool padded = D % kMfmaBN != 0 || H != Hp;
    const bool f32 = dt == DType::F32;
    const double kb = kKBlockBytes / (double)dtype_size(dt);
    // k steps of gate/up and down: gemm_mfma's, and gemm_rows' (kernels.hpp)
    const double kt1 = Dk / kb, kt2 = Hp / kb, kr1 = step_k(D) / kb, kr2 = step_k(H) / kb;
    const double live = (double)std::max<int64_t>(1, std::min(A, E)), mean = A / live;
    auto tiles = [&](int bm) { return live * std::max(1.0, mean / bm + 0.5); };  // row tiles, about
    auto cost_mfma = [&](double cols, double kt) {
        const double rounds = tiles(kMfmaBM) * cols / kMfmaBN / 256;
        const double fixed = f32 ? 45 : 16, step = f32 ? 1.7 : 0.58, once = f32 ? 15 : 4;
        // half a round or less: tiles split along K
        if (!padded && rounds <= 0.5)
            return once + fixed + step * kt / (rounds <= 0.25 ? 4 : 2) + (f32 ? 20 : 10);
        return once + (rounds <= 1 ? 1 : rounds + 0.75) * (fixed + step * kt);
    };
    const struct { int bm; double ns, ns_kt, ns_f32, ns_kt_f32; } opts[] = {
        {16, 3.8, 0.27, 12, 0.25}, {32, 5, 0.31, 7.5, 0.44}, {64, 5.3, 0.47, 8, 0.8}};
    // the least cost of a GEMM over the choices (all of them, or those of one tile height)
    auto pick = [&](double cols_mfma, double kt_mfma, double cols, double kt, int only, int* bm, int* waves) {
        double least = 1e30;
        *bm = kMfmaBM;
        if (!only || only == kMfmaBM) {
            least = cost_mfma(cols_mfma, kt_mfma);
            *waves = 0;
        }
        for (const auto& o : opts) {
            if ((o.bm == 16 && mean > kRows16Mean) || (o.bm == 32 && mean > kRows32Mean)) continue;
            if (only && only != o.bm) continue;
            const double lat = (f32 ? 0.1 + 0.002 * o.bm : 0.045 + 0.0004 * o.bm) * (padded ? 2.5 : 1);
            const double units = tiles(o.bm) * cols / 64;
            const double c = 5 + lat * kt + units * (f32 ? o.ns_f32 + o.ns_kt_f32 * kt : o.ns + o.ns_kt * kt) * 1e-3;
            // (between gemm_rows' heights, the smaller where it is within 1 us)
            if (c >= least - (*bm < o.bm ? 1.0 : 0.0)) continue;
            least = c;
            *bm = o.bm;
            *waves = padded ? 1 : o.bm == 64 && units >= (f32 ? 700 : 400) ? 2 : 4;
        }
        return least;
    };
    auto both = [&](int only, GemmPlan* p) {
        const double c = pick(2.0 * Hp, kt1, 2.0 * step_k(H), kr1, only, &p->bm1, &p->waves1);
        return c + pick((double)round_up(D, kMfmaBN), kt2, (double)round_up(D, 64), kr2, only, &p->bm2, &p->waves2);
    };
    GemmPlan plan, one;
    double least = both(0, &plan);
    if (plan.bm1 == plan.bm2) return plan;
    // a second tile table costs the dispatch 2 us, and nearly equal estimates
    // say little: one tile height unless two are better by 4 us
    least += 4;
    for (int bm : {kMfmaBM, 64, 32, 16}) {
        const double c = both(bm, &one);
        if (c < least) {
            least = c;
            plan = one;
        }
    }
    return plan;
}

}  // namespace nomas

// Which GEMM kernel and tile height a forward takes (host code, no device
// state: a function of the sizes alone).
//
// gemm_mfma's 256 x 256 tiles reach the chip's matrix rate once there are
// enough of them; gemm_rows' 16 / 32 / 64 x 64 tiles spread small problems
// over all CUs and stream weights for few rows.  The choice is the least
// estimated time of each GEMM.  The estimates (the tables below) are fitted to the
// stage times of 9,900 drawn calls with every choice timed (one MI355X, weights
// in the last-level cache, widths 16 to 3,072, 16 to 150,000 routed rows, 1 to 64
// experts evenly and unevenly loaded); they are within 10 to 20% (one standard
// deviation), which is mostly the tile counts that an uneven load makes.
//  - gemm_mfma: a time per tile where all run at once, less where tiles are
//    split along K, and beyond that one per round of 256 tiles.
//  - gemm_rows: the time of one tile's k steps and the time of all tiles with
//    the chip full, t = (a^1.5 + b^1.5)^(2/3).
// Over these calls the picks take 0.6% (whole-tile widths) and 1.1% (padded) more
// GEMM time than the best ones.  At whole-tile widths gemm_rows must be estimated
// 10% better: 0.8% of the GEMMs then take more than 1.05 times gemm_mfma's time,
// 1.5 times at worst (1.0% at an equal estimate; an earlier fit to 70 calls: 6%, up
// to twice the time: 5,539 rows of 512 x 768 in bf16, gate/up 38.7 instead of 20 us).
// The two GEMMs choose on their own, each with its tile table: 1,111 rows of
// 1000 x 2667, 6 experts, in bf16 take 36 + 53 us on gemm_mfma, 64 + 35 us on
// 64-row tiles, 36 + 35 us on one of each.
#pragma once

#include <algorithm>
#include <cmath>

#include "kernels.hpp"
#include "tile_map.hpp"

namespace nomas {

// gemm_rows' smaller tiles are taken up to these mean rows per expert
constexpr int kRows16Mean = 1024, kRows32Mean = 2048;

// GEMM tiles that a tile table must hold for A routed rows (or fewer) over E
// experts, whatever gemm_plan picks.
inline int64_t max_gemm_tiles(int64_t A, int64_t E) {
    const int64_t small = std::max(std::min(A, kRows16Mean * E) / 16, std::min(A, kRows32Mean * E) / 32);
    return std::max((A + 63) / 64, small + 1) + E;
}

// Estimated times in us, kt the k steps of 64 bytes.
struct MfmaCost {
    double one, one_kt, split;        // all tiles at once: one + one_kt kt / parts, + split where parts > 1
    double many, uneven, round, round_kt;  // else many + (rounds + uneven) (round + round_kt kt)
};
struct RowsCost {
    int bm, waves;
    double lat, lat_kt;  // one tile: lat + lat_kt kt
    double ns, ns_kt;    // each of them, in ns: ns + ns_kt kt
};
// [padded widths][f32]
constexpr MfmaCost kMfmaCost[2][2] = {
    {{10.5, 0.608, 15.3, 12.0, 0.49, 7.8, 0.625}, {27.5, 1.80, 9.8, 34.9, 0.14, 22.3, 1.90}},
    {{10.7, 0.529, 0, 6.4, 0.47, 8.5, 0.618}, {24.5, 1.59, 0, 2.8, 0.53, 28.4, 1.85}}};
// (waves 0: no such choice)
constexpr RowsCost kRowsCost[2][2][4] = {
    {{{64, 2, 3.9, 0.102, 6.5, 0.483}, {64, 4, 4.0, 0.079, 9.8, 0.465}, {32, 4, 3.9, 0.062, 7.1, 0.323}, {16, 4, 4.0, 0.052, 6.0, 0.265}},
     {{64, 2, 4.9, 0.353, 8.7, 0.787}, {64, 4, 5.7, 0.178, 13.7, 0.772}, {32, 4, 3.9, 0.142, 7.1, 0.457}, {16, 4, 4.6, 0.085, 10.4, 0.326}}},
    {{{64, 1, 3.9, 0.152, 4.4, 0.499}, {32, 1, 3.8, 0.093, 4.1, 0.330}, {16, 1, 3.8, 0.108, 4.2, 0.259}, {0, 0, 0, 0, 0, 0}},
     {{64, 1, 4.4, 0.570, 7.0, 0.769}, {32, 1, 3.7, 0.401, 3.7, 0.455}, {16, 1, 3.6, 0.309, 3.6, 0.316}, {0, 0, 0, 0, 0, 0}}}};

// A routed rows over E experts; Dk and Hp are the padded widths of D and H.
// dense_copy: >= 0 in the dense feed-forward, the us of the K-blocked copy of x that
// it saves where gemm_rows runs both GEMMs.  shared: of the A rows, those of the shared
// dense branch, one of the E experts, which has every row of the call.
inline GemmPlan gemm_plan(DType dt, int64_t A, int64_t E, int64_t Dk, int64_t Hp, int64_t D, int64_t H,
                          double dense_copy = -1, int64_t shared = 0) {
    // padded widths keep one order of summation at any row count: one wave, no K split
    const bool padded = D % kMfmaBN != 0 || H != Hp;
    const bool f32 = dt == DType::F32;
    const double kb = kKBlockBytes / (double)dtype_size(dt);
    // k steps of gate/up and down: gemm_mfma's, and gemm_rows' (kernels.hpp)
    const double kt1 = Dk / kb, kt2 = Hp / kb, kr1 = step_k(D) / kb, kr2 = step_k(H) / kb;
    const double live = (double)std::max<int64_t>(1, std::min(A, E)), mean = A / live;
    // row tiles: of evenly loaded experts, and on average over uneven ones (of one: the
    // same); the shared branch's exactly
    const double routed = (double)(A - shared), on = (double)std::min(A - shared, E - (shared ? 1 : 0));
    auto even = [&](int bm) {
        return (on > 0 ? on * std::ceil(routed / on / bm) : 0) + std::ceil((double)shared / bm);
    };
    auto tiles = [&](int bm) {
        return on <= 1 ? even(bm) : on * std::max(1.0, routed / on / bm + 0.5) + std::ceil((double)shared / bm);
    };
    auto cost_mfma_of = [&](double all, double kt) {
        const MfmaCost& c = kMfmaCost[padded][f32];
        const double rounds = all / kRound;
        if (rounds > 1) return c.many + (rounds + c.uneven) * (c.round + c.round_kt * kt);
        const int parts = padded ? 1 : split_parts((long long)std::min(all + 0.5, kRound - 1.0), (int)kt / kStages);
        return c.one + c.one_kt * kt / parts + (parts > 1 ? c.split : 0);
    };
    auto cost_mfma = [&](double cols, double kt) {  // a few tiles more or less can halve or double it
        return (cost_mfma_of(even(kMfmaBM) * cols / kMfmaBN, kt) + cost_mfma_of(tiles(kMfmaBM) * cols / kMfmaBN, kt)) / 2;
    };
    auto cost_rows = [&](const RowsCost& c, double cols, double kt) {
        const double one = c.lat + c.lat_kt * kt, full = tiles(c.bm) * cols / 64 * (c.ns + c.ns_kt * kt) * 1e-3;
        return std::pow(std::pow(one, 1.5) + std::pow(full, 1.5), 2.0 / 3.0);
    };
    // the least cost of a GEMM over the choices (0: all of them, -1: gemm_rows', else those of one tile height)
    auto pick = [&](double cols_mfma, double kt_mfma, double cols, double kt, int only, int* bm, int* waves) {
        double least = 1e30;
        *bm = kMfmaBM;
        if (!only || only == kMfmaBM) {
            least = cost_mfma(cols_mfma, kt_mfma) / (padded ? 1.0 : 1.1);
            *waves = 0;
        }
        for (const RowsCost& o : kRowsCost[padded][f32]) {
            if (!o.waves || (o.bm == 16 && mean > kRows16Mean) || (o.bm == 32 && mean > kRows32Mean)) continue;
            if (only > 0 && only != o.bm) continue;
            const double c = cost_rows(o, cols, kt);
            // (between gemm_rows' heights, the smaller of two about as good)
            if (c >= least + (o.bm < *bm && *bm != kMfmaBM ? 0.2 : 0.0)) continue;
            least = c;
            *bm = o.bm;
            *waves = o.waves;
        }
        return least;
    };
    auto both = [&](int only, GemmPlan* p) {
        const double c = pick(2.0 * Hp, kt1, 2.0 * step_k(H), kr1, only, &p->bm1, &p->waves1);
        return c + pick((double)round_up(D, kMfmaBN), kt2, (double)round_up(D, 64), kr2, only, &p->bm2, &p->waves2);
    };
    GemmPlan plan, one;
    double least = both(0, &plan);
    if (dense_copy >= 0) {  // (no table to write twice)
        if ((plan.waves1 && plan.waves2) || least + dense_copy <= both(-1, &one)) return plan;
        return one;
    }
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

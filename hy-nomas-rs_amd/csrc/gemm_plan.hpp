// Which GEMM kernel and tile height a forward takes (host code, no device
// state: a function of the sizes alone).
//
// gemm_mfma's 256 x 256 tiles reach the chip's matrix rate once there are
// enough of them; gemm_rows' 16 / 32 / 64 x 64 tiles spread small problems
// over all CUs and stream weights for few rows.  The choice is the least
// estimated time of the two GEMMs together, from what both kernels measured
// on one MI355X (stage times, weights in the last-level cache, expert widths
// 64 x 128 to 1536 x 4096, 1 to 8,192 rows, 1 to 64 experts):
//  - gemm_mfma: 5 us (f32: 22 us, most of it the first fetch of its code), and
//    for each round of 256 tiles, full or not, 6 us plus 0.5 us per k step (f32:
//    12 us plus 2 us per 16 k).
//  - gemm_rows: 5 us, per k step of one tile 0.05 / 0.06 / 0.07 us for 16 / 32 /
//    64 rows (f32: 0.13 / 0.16 / 0.23), and per tile and k step, with the chip
//    full, 0.35 / 0.42 / 0.6 ns (f32: 0.37 / 0.52 / 0.9 ns).
// Where the two meet, at 64 rows per expert of 1536 x 4096 or 2,048 of 512 x
// 1024 in bf16, either is within 10% of the other.
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
    const double kt1 = Dk / kb, kt2 = Hp / kb;  // k steps of gate/up and down
    const double live = (double)std::max<int64_t>(1, std::min(A, E)), mean = A / live;
    auto tiles = [&](int bm) { return live * std::max(1.0, mean / bm + 0.5); };  // row tiles, about
    auto cost_mfma = [&](double cols, double kt) {
        const double rounds = tiles(kMfmaBM) * cols / kMfmaBN / 256;
        return (f32 ? 22 : 5) + (rounds <= 1 ? 1 : rounds + 0.5) * (f32 ? 12 + 2.0 * kt : 6 + 0.5 * kt);
    };
    GemmPlan best{kMfmaBM, 0, 0};
    double least = cost_mfma(2.0 * Hp, kt1) + cost_mfma((double)round_up(D, kMfmaBN), kt2);
    const struct { int bm; double ns, ns_f32; } opts[] = {{16, 0.35, 0.37}, {32, 0.42, 0.52}, {64, 0.6, 0.9}};
    for (const auto& o : opts) {
        if ((o.bm == 16 && mean > kRows16Mean) || (o.bm == 32 && mean > kRows32Mean)) continue;
        auto cost = [&](double cols, double kt) {
            const double lat = (f32 ? 0.1 + 0.002 * o.bm : 0.045 + 0.0004 * o.bm) * (padded ? 2.5 : 1);
            return 5 + lat * kt + tiles(o.bm) * cols / 64 * kt * (f32 ? o.ns_f32 : o.ns) * 1e-3;
        };
        // two waves per block (fewer partial sums) once 64-row tiles alone fill the chip
        auto waves = [&](double cols) { return padded ? 1 : o.bm == 64 && !f32 && tiles(64) * cols / 64 >= 2048 ? 2 : 4; };
        const double c = cost(2.0 * Hp, kt1) + cost((double)D, kt2);
        if (c < least) {
            least = c;
            best = GemmPlan{o.bm, waves(2.0 * Hp), waves((double)D)};
        }
    }
    return best;
}

}  // namespace nomas

// Grouped expert GEMMs for calls of few rows (bf16 / f16 / f32 in, f32
// accumulate): the same operands, layouts and epilogues as gemm_mfma.hip, on
// tiles of 16 NT token rows x 64 weight rows.
//
// What bounds these calls is the weights' way from HBM (few rows per expert)
// or how few 256 x 256 tiles there are (small widths), so the work is split
// finely and nothing waits for anything:
//  - A block's NW waves take the same tile, each its own 1/NW of the k steps;
//    the waves' partial sums meet in LDS once, at the end, and are added in
//    wave order.  There is no barrier in the k loop.  With one wave (padded
//    widths) a tile's sums run in gemm_mfma's order, from the bias through
//    ascending k with the same MFMAs: results then do not depend on which of
//    the two kernels, and so on how many rows, a call has.
//  - Operands go straight from global memory to registers: K-blocked, the 16
//    rows x 64 bytes of one MFMA fragment are 1 KB of consecutive memory, read
//    by one instruction, and no other wave of the block needs them.  A ring
//    of P steps of fragments per wave is in flight.
//  - Units run weight tile by weight tile, the row tiles of one expert next to
//    each other, in eight contiguous shares, one per XCD (block i runs on XCD
//    i % 8): the row tiles of an expert then find its weights in their XCD's
//    L2.
//  - Padding past a step of 32 columns, past the real columns (down) and past 32
//    hidden units that hold a real one (gate/up) is neither read nor computed.
// Measured (stage times of gate/up + down, one MI355X, against gemm_mfma's 256 x
// 256 tiles or, for padded widths, the earlier vector-unit kernel): 16 rows of 8
// experts of 1536 x 4096 in bf16 42 + 51 -> 33 + 18.5 us (6.1 and 5.4 TB/s of
// weights); 64 rows 43 + 53 -> 36 + 21 us; 512 rows of 512 x 1024, 4 experts, 37 +
// 29 -> 13 + 8 us; 208 rows of 64 x 128 in f32, 4 experts, 18 + 20 -> 5.5 + 6 us;
// 1,111 rows of 1000 x 2667, 6 experts, down 555 -> 35 us.
#include <type_traits>

#include "kernels.hpp"
#include "mfma.hpp"

namespace nomas {

namespace {

constexpr int kRowsBN = 64;  // weight rows per tile: 32 gate + 32 up rows, or 64 down rows

template <typename T, int MODE, int NT, int NW>
__global__ __launch_bounds__(NW * kWave) void gemm_rows_kernel(GemmArgs a) {
    using V = typename Mfma<T>::V;
    constexpr int BM = 16 * NT, BN = kRowsBN, NB = BN / 16;
    constexpr int BK = kblock_elems<T>();
    constexpr bool kSplit = sizeof(T) == 4;  // f32: bf16 planes (mfma.hpp), two K-blocks a step
    constexpr int KS = kSplit ? 2 : 1;       // weight K-blocks per step
    constexpr int XS = kSplit ? kPlanes : 1; // token blocks per step
    // steps in flight per wave
    constexpr int P = kSplit    ? (NT == 1 ? 3 : 2)
                      : NW == 1 ? (NT == 1 ? 8 : NT == 2 ? 6 : 4)
                                : (NT <= 2 ? 4 : 3);
    __shared__ f32x4_t s_part[NW][NB][NT][kWave];

    const int N = a.N, K = a.K;
    const int live = a.dense_rows ? (int)((a.dense_rows + BM - 1) / BM) : min(*a.tile_total, a.max_tiles);
    // down: weight tiles past the real columns have nothing to store
    const int ntn = (MODE == kDown ? a.n_out + BN - 1 : a.n_used) / BN;
    const long long units = (long long)live * ntn;
    const long long share = (units + kNumXcd - 1) / kNumXcd;
    const long long q = blockIdx.x / kNumXcd, u = (blockIdx.x % kNumXcd) * share + q;
    if (q >= share || u >= units) return;
    const int mt = (int)(u % live), n0 = (int)(u / live) * BN;
    TileInfo ti = {0, mt * BM, (int)min<int64_t>(BM, a.dense_rows - (int64_t)mt * BM), 0};
    if (!a.dense_rows) ti = a.tiles[mt];
    const int e = ti.expert, row0 = ti.row0, nrows = ti.rows;
    if (e < 0 || e >= a.num_experts || nrows < 1 || nrows > BM || row0 < 0 ||
        row0 + (int64_t)nrows > a.a_cap)
        return;
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int l16 = lane & 15, lq = lane >> 4;

    // this wave's k steps (none in gate/up tiles that hold padding only)
    const int kt_all = K / BK, st_all = a.k_used / (BK * KS);
    const bool pad_tile = MODE == kGateUp && n0 / 2 >= a.n_out;
    const int s0 = pad_tile ? 0 : st_all * wave / NW, s1 = pad_tile ? 0 : st_all * (wave + 1) / NW;
    const int64_t wstep = (int64_t)N * BK, xstep = a.x_row ? kKBlockBytes : a.a_cap * kKBlockBytes;  // (elements, bytes)
    const int64_t xrow = a.x_row ? a.x_row : kKBlockBytes;
    const T* Wt = static_cast<const T*>(a.W) + ((int64_t)e * kt_all * N + n0) * BK;
    const char* Xt = static_cast<const char*>(a.X) + row0 * xrow;
    const uint32_t woff = (uint32_t)(l16 * kKBlockBytes + lq * 16);
    uint32_t xoff[NT];  // rows past the tile's end read its last row (never stored)
#pragma unroll
    for (int j = 0; j < NT; ++j)
        xoff[j] = (uint32_t)(min(j * 16 + l16, nrows - 1) * xrow + lq * 16);

    auto bias = [&](int i) -> f32x4_t {
        const float4 b = *reinterpret_cast<const float4*>(a.bias + (int64_t)e * N + n0 + i * 16 + 4 * lq);
        return f32x4_t{b.x, b.y, b.z, b.w};
    };
    f32x4_t acc[NB][NT];
#pragma unroll
    for (int i = 0; i < NB; ++i)
#pragma unroll
        for (int j = 0; j < NT; ++j) acc[i][j] = NW == 1 ? bias(i) : f32x4_t{0.0f, 0.0f, 0.0f, 0.0f};
    if constexpr (kSplit && NW == 1) {  // f32: the sums are scaled (mfma.hpp)
#pragma unroll
        for (int i = 0; i < NB; ++i)
#pragma unroll
            for (int j = 0; j < NT; ++j) acc[i][j] *= a.sum_up;
    }
    V fa[P][KS][NB], fb[P][XS][NT];
    auto load = [&](int st, V (&wa)[KS][NB], V (&xb)[XS][NT]) {  // the fragments of step st
#pragma unroll
        for (int c = 0; c < KS; ++c) {
            const char* w = reinterpret_cast<const char*>(Wt + (st * KS + c) * wstep);
#pragma unroll
            for (int i = 0; i < NB; ++i)
                wa[c][i] = *reinterpret_cast<const V*>(w + i * 16 * kKBlockBytes + woff);
        }
#pragma unroll
        for (int c = 0; c < XS; ++c) {
            const char* x = Xt + (st * XS + c) * xstep;
#pragma unroll
            for (int j = 0; j < NT; ++j) xb[c][j] = *reinterpret_cast<const V*>(x + xoff[j]);
        }
    };
    auto fetch = [&](int s, V (&wa)[KS][NB], V (&xb)[XS][NT]) {  // past the end: the last step again
        load(max(min(s, s1 - 1), 0), wa, xb);
    };
#pragma unroll
    for (int p = 0; p < P; ++p) fetch(s0 + p, fa[p], fb[p]);
    for (int st = s0; st < s1; st += P) {
#pragma unroll
        for (int p = 0; p < P; ++p) {
            if (st + p < s1) {
                if constexpr (kSplit) {
#pragma unroll
                    for (int i = 0; i < NB; ++i) {
                        u32x4_t pa[kPlanes];
                        split_all(fa[p][0][i], fa[p][KS - 1][i], pa);
#pragma unroll
                        for (int m = 0; m < kProducts; ++m)
#pragma unroll
                            for (int j = 0; j < NT; ++j)
                                acc[i][j] = mfma_plane(pa[product_a(m)],
                                                       __builtin_bit_cast(u32x4_t, fb[p][product_b(m)][j]), acc[i][j]);
                    }
                } else {
#pragma unroll
                    for (int i = 0; i < NB; ++i)
#pragma unroll
                        for (int j = 0; j < NT; ++j)
                            acc[i][j] = Mfma<T>::run(fa[p][0][i], fb[p][0][j], acc[i][j]);
                }
            }
            fetch(st + p + P, fa[p], fb[p]);
        }
    }
    if constexpr (kSplit) {
        // as in gemm_mfma: sums that are not finite again, with f32 MFMAs
        float t = 0.0f;
#pragma unroll
        for (int i = 0; i < NB; ++i)
#pragma unroll
            for (int j = 0; j < NT; ++j) t = not_finite(acc[i][j], t);
#pragma unroll
        for (int i = 0; i < NB; ++i)
#pragma unroll
            for (int j = 0; j < NT; ++j) acc[i][j] *= a.sum_down;
        if (a.all_f32 || __any(t != t)) {
            // (16 token rows at a time: all of them at once took 260 to 288
            // registers, which leaves a SIMD one wave)
#pragma unroll
            for (int j = 0; j < NT; ++j) {
                f32x4_t again[NB];
#pragma unroll
                for (int i = 0; i < NB; ++i) again[i] = NW == 1 ? bias(i) : f32x4_t{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll 1
                for (int st = s0; st < s1; ++st) {
                    u32x4_t pl[kPlanes];
#pragma unroll
                    for (int c = 0; c < kPlanes; ++c)
                        pl[c] = *reinterpret_cast<const u32x4_t*>(Xt + (st * XS + c) * xstep + xoff[j]);
#pragma unroll
                    for (int c = 0; c < KS; ++c)
#pragma unroll
                        for (int i = 0; i < NB; ++i) {
                            const f32x4_t w = *reinterpret_cast<const f32x4_t*>(
                                reinterpret_cast<const char*>(Wt + (st * KS + c) * wstep) + i * 16 * kKBlockBytes + woff);
#pragma unroll
                            for (int k4 = 0; k4 < 4; ++k4)
                                again[i] = mfma_f32(w[k4] * a.w_down, unsplit(pl, c * 4 + k4), again[i]);
                        }
                }
                if (a.all_f32) {
#pragma unroll
                    for (int i = 0; i < NB; ++i) acc[i][j] = again[i];
                } else if constexpr (MODE == kDown) {
#pragma unroll
                    for (int i = 0; i < NB; ++i) keep_finite(acc[i][j], again[i]);
                } else {
#pragma unroll
                    for (int i = 0; i < 2; ++i)
#pragma unroll
                        for (int s = 0; s < 4; ++s) {
                            const bool ok = unit_finite(acc[i][j][s], acc[i + 2][j][s]);
                            acc[i][j][s] = ok ? acc[i][j][s] : again[i][s];
                            acc[i + 2][j][s] = ok ? acc[i + 2][j][s] : again[i + 2][s];
                        }
                }
            }
        }
    }
    // Epilogue.  Lane (l16, lq) of block (i, j) holds token row 16 j + l16 and
    // weight rows 16 i + 4 lq + (0..3).  Blocks (i, j) and (i + 2, j) finish
    // together: a gate block and its up block, or two blocks of down columns.
    T* out = static_cast<T*>(a.out);
    typedef typename std::conditional<sizeof(T) == 2, uint2, uint4>::type Raw4;
    auto finish = [&](int i, int j, const f32x4_t (&v)[2]) {
        const int m = j * 16 + l16;
        if (m >= nrows) return;
        if constexpr (MODE == kGateUp) {
            const int hc = n0 / 2 + i * 16 + 4 * lq;
            float hv[4];
#pragma unroll
            for (int s = 0; s < 4; ++s) hv[s] = hc + s < a.n_out ? swiglu<T>(v[0][s], v[1][s]) : 0.0f;
            store_hidden<T>(a.out, a.a_cap, row0 + m, hc, hv);
        } else {
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                const int n = n0 + (i + 2 * h) * 16 + 4 * lq;
                if (n >= a.n_out) continue;  // (n_out % 8 == 0: 4 columns are real or padding)
                T ov[4];
#pragma unroll
                for (int s = 0; s < 4; ++s) ov[s] = Elt<T>::from_f32(v[h][s]);
                Raw4 raw;
                __builtin_memcpy(&raw, ov, sizeof(raw));
                *reinterpret_cast<Raw4*>(out + (int64_t)(row0 + m) * a.n_out + n) = raw;
            }
        }
    };
    if constexpr (NW == 1) {
#pragma unroll
        for (int j = 0; j < NT; ++j)
#pragma unroll
            for (int i = 0; i < 2; ++i) {
                const f32x4_t v[2] = {acc[i][j], acc[i + 2][j]};
                finish(i, j, v);
            }
    } else {
        // the waves' partial sums in wave order; wave w takes pairs w, w + NW, ...
#pragma unroll
        for (int i = 0; i < NB; ++i)
#pragma unroll
            for (int j = 0; j < NT; ++j) s_part[wave][i][j][lane] = acc[i][j];
        __syncthreads();
        for (int it = wave; it < 2 * NT; it += NW) {
            const int i = it & 1, j = it >> 1;
            f32x4_t v[2];
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                f32x4_t t = s_part[0][i + 2 * h][j][lane];
#pragma unroll
                for (int w = 1; w < NW; ++w) t += s_part[w][i + 2 * h][j][lane];
                v[h] = t + bias(i + 2 * h);
            }
            finish(i, j, v);
        }
    }
}

template <typename T, int MODE, int NT, int NW>
hipError_t launch_rows_t(const GemmArgs& a, hipStream_t s) {
    const int n_cols = MODE == kGateUp ? a.N / 2 : a.N;
    if (a.N % kMfmaBN != 0 || a.K % (kblock_elems<T>() * kStages) != 0 || a.n_out < 1 || a.n_out > n_cols ||
        (MODE == kDown && a.n_out % 8 != 0))
        return hipErrorInvalidValue;
    if (a.k_used < 1 || a.k_used % 32 != 0 || a.k_used > a.K ||
        (MODE == kGateUp && (a.n_used < a.n_out * 2LL || a.n_used % kRowsBN != 0 || a.n_used > a.N)))
        return hipErrorInvalidValue;
    if (a.x_row && (sizeof(T) != 2 || a.x_row % 16 != 0 || a.x_row < a.K * 2LL || a.x_row > (1LL << 26)))
        return hipErrorInvalidValue;
    if (a.max_tiles <= 0) return hipSuccess;
    const int64_t ntn = (MODE == kDown ? a.n_out + kRowsBN - 1 : a.n_used) / kRowsBN;
    const int64_t grid = round_up((int64_t)a.max_tiles * ntn, kNumXcd);
    if (grid > 0x7fffffff) return hipErrorInvalidValue;
    launch_kernel((gemm_rows_kernel<T, MODE, NT, NW>), dim3((unsigned)grid), dim3(NW * kWave), 0, s, a);
    return hipGetLastError();
}

template <typename T, int MODE>
hipError_t launch_rows(const GemmArgs& a, int bm, int waves, hipStream_t s) {
    switch (bm * 100 + waves) {
        case 1601: return launch_rows_t<T, MODE, 1, 1>(a, s);
        case 3201: return launch_rows_t<T, MODE, 2, 1>(a, s);
        case 6401: return launch_rows_t<T, MODE, 4, 1>(a, s);
        case 1604: return launch_rows_t<T, MODE, 1, 4>(a, s);
        case 3204: return launch_rows_t<T, MODE, 2, 4>(a, s);
        case 6404: return launch_rows_t<T, MODE, 4, 4>(a, s);
        case 6402: return launch_rows_t<T, MODE, 4, 2>(a, s);
    }
    return hipErrorInvalidValue;
}

}  // namespace

hipError_t launch_gemm_rows(DType dt, bool gate_up, const GemmArgs& a, int bm, int waves, hipStream_t s) {
    switch (dt) {
        case DType::F32:
            return gate_up ? launch_rows<float, kGateUp>(a, bm, waves, s) : launch_rows<float, kDown>(a, bm, waves, s);
        case DType::BF16:
            return gate_up ? launch_rows<__bf16, kGateUp>(a, bm, waves, s) : launch_rows<__bf16, kDown>(a, bm, waves, s);
        case DType::F16:
            return gate_up ? launch_rows<_Float16, kGateUp>(a, bm, waves, s)
                           : launch_rows<_Float16, kDown>(a, bm, waves, s);
    }
    return hipErrorInvalidValue;
}

}  // namespace nomas

// Host-side launch interface of the MoE feed-forward kernels.
//
// Pipeline of one forward (all on one stream):
//   router  -> topk_idx / topk_w / gap per row, per-chunk expert histogram
//   dispatch-> expert counts/offsets, GEMM tile table, stable permutation
//              (tok_pos) + gather of x rows (x_perm)
//   gemm_gate_up -> h = silu(x W_gate^T + b_gate) * (x W_up^T + b_up)
//   gemm_down    -> y_perm = h W_down^T + b_down
//   combine -> out[t] = sum over the row's slots (ascending expert) of w * y_perm
#pragma once

#include <hip/hip_ext.h>

#include "common.hpp"

namespace nomas {

constexpr int kMaxExperts = 256;  // router LDS holds 64 rows x E f64 logits

// Kernel-exact stage timing.  While a layer records a profiled forward, this
// thread's stage in progress is set here, and every launch of the stage
// carries its events: the runtime stamps the start event when the stage's
// first kernel starts and the stop event when each kernel ends (the last one
// counts).  Null when not profiling.
struct StageTiming {
    hipEvent_t start, stop;
    bool launched;
};
StageTiming*& stage_timing();

// Every kernel of the library is launched through here (errors are left for
// the caller's hipGetLastError).
template <typename F, typename... Args>
inline void launch_kernel(F kernel, dim3 grid, dim3 block, uint32_t lds, hipStream_t s,
                          Args... args) {
    StageTiming* t = stage_timing();
    hipEvent_t start = nullptr, stop = nullptr;
    if (t) {
        start = t->launched ? nullptr : t->start;
        stop = t->stop;
        t->launched = true;
    }
    hipExtLaunchKernelGGL(kernel, grid, block, lds, s, start, stop, 0u, args...);
}

// Output tile of the grouped GEMMs: token rows and weight rows.
constexpr int kMfmaBM = 256;
constexpr int kMfmaBN = 256;

// The FFN half of a DiT block around the MoE (block.rs:96-101):
//   h   = modulate(norm2(x), shift, scale)   (norm.rs:55-65, modulate.rs:69-79)
//   out = x + moe(h) * gate
// Row r belongs to sequence r / seq; shift, scale, gate are (sequences, D) f32.
// seam_h_kernel writes h (read by the router and the dispatch as their x);
// the combine applies the gated residual in its epilogue.
struct SeamArgs {
    const void* x;        // rows x D, model dtype
    void* h;              // rows x D, model dtype
    int64_t rows;
    int D;
    int64_t seq;          // rows per sequence
    const float* norm_w;  // D (null: no affine gain)
    double eps;
    const float* shift;   // sequences x D
    const float* scale;
};

struct RouterArgs {
    const void* x;
    const void* wr;
    int64_t rows;
    int D, E, k;
    int k_slots;        // k, or k + 1 with the shared dense slot
    float dense_coef;   // gate of the dense slot
    int32_t* topk_idx;  // rows x k_slots
    float* topk_w;      // rows x k_slots
    float* gap;         // rows
    int32_t* chunk_counts;  // ceil(rows / block_rows) x E_cols: one histogram per router block
    int block_rows;         // rows per router block: router_block_rows() of this launch
};


// K-blocked layout: a matrix of R rows and K columns is stored as
// column blocks of KB = 64 bytes of elements (32 for 16-bit types, 16 for
// f32), each R rows x KB contiguous elements, i.e. element (r, k) at
// ((k / KB) * R + r) * KB + k % KB.  One k step of a GEMM tile (256 rows x
// 64 bytes) is then a single contiguous 16 KB run of memory, fetched as whole
// 128-byte lines.
//
// Any dim and hidden width run on the same GEMMs: the operands are padded with
// zeros when they are laid out (weights at upload, x_perm by the dispatch, h
// by the gate/up epilogue), K to whole turns of the GEMM's LDS ring and the
// weight rows to whole tiles, so no GEMM loop has a remainder.  gemm_rows needs
// whole steps of 32 only (step_k), and neither computes nor reads the rest of the
// padding; where it runs the GEMM that reads an operand, the rest is not written.
constexpr int kKBlockBytes = 64;
constexpr int kStages = 4;  // K steps (K-blocks) per turn of the ring
template <typename T>
__host__ __device__ constexpr int kblock_elems() { return kKBlockBytes / (int)sizeof(T); }
__host__ __device__ constexpr int64_t round_up(int64_t n, int64_t m) { return (n + m - 1) / m * m; }
// f32 activations (x_perm, h) are stored as their three bf16 planes (mfma.hpp):
// columns in blocks of 32, each block's planes one after another, each plane's
// row 64 bytes.  Within a row the 16-byte chunk c holds columns 4c..4c+3 and
// 16 + 4c..16 + 4c + 3 of the block, the order in which a GEMM lane holds the
// weights of two 16-column f32 K-blocks.  Element (r, k) of plane p:
//   ((k / 32 * 3 + p) * R + r) * 32 + (k / 4 % 4) * 8 + (k / 16 % 2) * 4 + k % 4
constexpr int kActPlanes = 3;  // mfma.hpp's kPlanes
constexpr float kPlaneScale = 0x1p24f;  // the planes add up to the value times this (mfma.hpp)
// Bytes of one element of x_perm or h.
__host__ __device__ constexpr int act_bytes(DType dt) { return dt == DType::F32 ? 2 * kActPlanes : 2; }
// Columns of a K-blocked operand with K = `k` columns of es-byte elements.
__host__ __device__ constexpr int64_t padded_k(int64_t k, int es) {
    return round_up(k, kStages * kKBlockBytes / es);
}

// Columns that gemm_rows reads of an operand of `k` columns.
__host__ __device__ constexpr int64_t step_k(int64_t k) { return round_up(k, 32); }

struct DispatchArgs {
    const void* x;
    int64_t rows;
    int D, E_cols, k_slots;
    const int32_t* topk_idx;
    const int32_t* chunk_counts;  // ceil(rows / count_rows) x E_cols, from the router
    int nchunks;            // 64-row chunks
    int count_rows;         // rows per histogram (the router's rows per block: 64 or 32)
    int BM, BM2;            // GEMM tile rows: gate/up, down
    int max_tiles, max_tiles2;
    int32_t* expert_count;  // E_cols
    int32_t* expert_off;    // E_cols + 1
    TileInfo* tiles;        // max_tiles
    TileInfo* tiles2;       // max_tiles2 (written where BM2 != BM)
    int32_t* tile_total;    // 4: the tile count, the two GEMMs' tail counters (cleared), the second count
    int32_t* tok_pos;  // rows x k_slots
    void* x_perm;      // a_cap x Dk, K-blocked (R = a_cap; f32: planes)
    int Dk;            // padded_k(D) or step_k(D): columns D .. Dk - 1 are written as zeros
    int64_t a_cap;     // rows of x_perm (positions must stay below)
};

struct GemmArgs {
    const void* X;     // token rows (a_cap x K), expert-contiguous (f32: planes)
    const void* W;     // expert weights
    const float* bias; // expert biases (f32)
    void* out;
    const TileInfo* tiles;
    const int32_t* tile_total;
    int max_tiles;
    int N;  // weight rows, whole tiles (2 x padded H for gate/up, padded D for down)
    int K;  // padded to whole ring turns
    // real output columns: H (hidden units past it are written as zeros, which
    // the down GEMM multiplies with zero weights) or D (columns past it are not
    // stored; also the row stride of out)
    int n_out;
    int num_experts;  // experts with weights (tiles naming others are skipped)
    int64_t a_cap;    // rows of X / out (tiles reaching beyond are skipped)
    // gemm_rows: the columns of K that it walks (step_k of the real ones), and in
    // gate/up the weight rows that it computes (those of step_k(H) hidden units,
    // or N where gemm_mfma reads h)
    int k_used = 0, n_used = 0;
    // gemm_rows: where X is not K-blocked (rows of x in place, whole K-blocks
    // of 16-bit elements): bytes from row to row; 0: K-blocked
    int64_t x_row = 0;
    // gemm_rows, dense feed-forward: its rows, all of expert 0, with no tile
    // table (tiles and tile_total are not read); 0: the table
    int64_t dense_rows = 0;
    // f32: W holds the weights times a power of two (kPlaneScale or 1) and the sums
    // of planes come out times sum_up; their inverses; and whether every sum is
    // made with f32 MFMAs (weights too large to be scaled, others too small not to be)
    float w_down = 1.0f, sum_up = 1.0f, sum_down = 1.0f;
    bool all_f32 = false;
    // f32 partial sums of tiles split along K (kSplitUnits units of
    // kSplitUnitFloats each; null: no tile is split) and one arrival counter per
    // split tile (zero between launches: the last part to arrive resets it)
    float* split_ws;
    int32_t* split_cnt;
    // the ticket counter of the tail units handed out at run time
    // (zero before the launch: the kernel that writes the tile table clears it)
    int32_t* tail_cnt = nullptr;
    // down GEMM: write `out` with the nontemporal hint.  For
    // outputs larger than the chip's last-level cache, which the combine reads
    // back once: their lines then go to HBM as they are written instead of
    // being evicted dirty while the combine streams them in.
    int out_nt = 0;
};
// MI355X's last-level cache (the Infinity Cache in front of HBM).
constexpr int64_t kLastLevelCacheBytes = (int64_t)256 << 20;
// MI355X's L2 caches together (8 XCDs x 4 MB).
constexpr int64_t kL2TotalBytes = (int64_t)32 << 20;
// One split unit's partial tile: 256 x 256 f32.
constexpr int64_t kSplitUnitFloats = 256 * 256;
constexpr int kSplitUnits = 256;

// Which kernels run a forward's two GEMMs (gemm_plan.hpp).
struct GemmPlan {
    // gate/up and down: token rows per tile, and waves per block of gemm_rows
    // (0: gemm_mfma, with its 256 rows)
    int bm1, waves1;
    int bm2, waves2;
};

struct CombineArgs {
    const void* y_perm;
    const int32_t* tok_pos;
    const float* topk_w;
    int64_t rows;
    int D, k_slots;
    void* out;
    int64_t a_cap;  // rows of y_perm
    // gated residual (gate non-null): out = x + out_moe * gate[row / seq]
    const void* resid_x;  // rows x D, model dtype
    const float* gate;    // sequences x D
    int64_t seq;
    // write `out` with the nontemporal hint: when y_perm is larger than the
    // last-level cache, its reads stream through it and would evict the
    // output's dirty lines into the middle of them anyway
    int out_nt = 0;
};

size_t router_lds_bytes(int E);
// Rows per router block (and per histogram it writes) for a launch of
// `rows` rows: 64, or 32 for small launches that 64-row blocks would leave
// short of bytes in flight.
int router_block_rows(DType dt, int64_t rows, int D, int E);
// Smallest rows per router block: the histogram buffer holds
// ceil(rows / kMinRouterBlockRows) histograms.
constexpr int kMinRouterBlockRows = 32;
// Whether the dispatch kernel's LDS holds E_cols experts and k_slots slots per row.
bool dispatch_supported(int E_cols, int k_slots);

hipError_t launch_seam_h(DType dt, const SeamArgs& a, hipStream_t s);
hipError_t launch_gated_residual(DType dt, const void* x, const void* y, const float* gate,
                                 void* out, int64_t rows, int D, int64_t seq, hipStream_t s);
hipError_t launch_router(DType dt, const RouterArgs& a, hipStream_t s);
hipError_t launch_dispatch(DType dt, const DispatchArgs& a, hipStream_t s);
// Grouped GEMMs: W packed as described in moe_layer.cpp, the tile tables in
// tiles of plan.bm1 and plan.bm2 rows.
hipError_t launch_gemm_gate_up(DType dt, const GemmArgs& a, const GemmPlan& plan, hipStream_t s);
hipError_t launch_gemm_down(DType dt, const GemmArgs& a, const GemmPlan& plan, hipStream_t s);
hipError_t launch_gemm_mfma(DType dt, bool gate_up, const GemmArgs& a, hipStream_t s);
hipError_t launch_gemm_rows(DType dt, bool gate_up, const GemmArgs& a, int bm, int waves, hipStream_t s);
hipError_t launch_combine(DType dt, const CombineArgs& a, hipStream_t s);
// Dense feed-forward (no routing): x re-laid out K-blocked with Dk columns
// (padded_k(D) or step_k(D)) for the gate/up GEMM, and the tile table of `rows` rows
// of one expert in BM-row tiles (max_tiles entries written).
hipError_t launch_kblock(DType dt, const void* x, void* xk, int64_t rows, int D, int Dk,
                         int64_t a_cap, int BM, int max_tiles, TileInfo* tiles, int32_t* tile_total,
                         hipStream_t s);

}  // namespace nomas

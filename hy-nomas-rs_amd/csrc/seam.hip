// norm2 + modulate of a DiT block on gfx950 (block.rs:96):
//   h = modulate(norm2(x), shift, scale)      (norm.rs:55-65, modulate.rs:69-79)
// for rows x D activations, row r in sequence r / seq.
//
// One block of 256 threads takes 16 rows in two phases.
//  1. The sum of squares of each row, added in the reference's order: x*x
//     rounded to f32, then one add per element in ascending d -- a serial chain
//     of D adds per row that no reordering may shorten.  Waves 1..3 make the
//     squares, 256 columns of the 16 rows at a time, into one half of a double
//     buffer in LDS (f32, rows padded by 16 bytes so the lanes' 16-byte reads at
//     one column spread over all banks); meanwhile lane r of wave 0 adds row
//     r's squares out of the other half.  The chain then costs one add per
//     element and never waits on HBM.
//  2. h: a thread takes a 16-byte column chunk of 8 rows, its norm_w, shift and
//     scale in registers (read again where the sequence changes).
// Bytes per row: D*b read twice (the second time mostly from cache), D*b
// written.  The chain (about 8 us at D = 3072) bounds a call whose blocks run
// once, so blocks are small: there are enough of them for all CUs from 4,096
// rows on, and several on a CU hide each other's chains.  Measured against
// blocks of 64 rows and 1,024 threads (75 blocks for 4,744 rows): 4,744 rows of
// 3,072 bf16 46 -> 31 us, 4,872 rows of 1,024 f32 19 -> 17 us, 14,232 rows of
// 1,536 bf16 31 -> 30 us (131 MB, 4.4 TB/s; a large copy reaches 4.9).
#include <algorithm>

#include "kernels.hpp"
#include "seam.hpp"

namespace nomas {

namespace {

constexpr int kSeamRows = 16;
constexpr int kSeamThreads = 256;
constexpr int kStageCols = 256;                           // columns per stage
constexpr int kRowStride = kStageCols * 4 + 16;           // bytes, padded
constexpr int kStageBytes = kSeamRows * kRowStride;       // 16,640
constexpr int kRowGroup = 8;                              // rows per thread in phase 2

template <typename T>
__global__ __launch_bounds__(kSeamThreads) void seam_h_kernel(SeamArgs a) {
    __shared__ __align__(16) unsigned char s_buf[2 * kStageBytes];
    __shared__ float s_inv[kSeamRows];   // inverse RMS per row
    __shared__ int s_seqidx[kSeamRows];  // sequence per row, from the block's first
    constexpr int EPC = 16 / sizeof(T);
    constexpr int kChunks = kSeamRows * kStageCols / EPC;   // 16-byte chunks per stage
    constexpr int kRowChunks = kStageCols / EPC;
    // waves 1..3 produce the squares, wave 0 adds them up
    constexpr int kProducers = kSeamThreads - kWave;
    constexpr int kLoads = (kChunks + kProducers - 1) / kProducers;  // 3 (16-bit) or 6 (f32)
    constexpr int kRing = kLoads == 3 ? 4 : 3;  // stages of x in flight (32 or 48 KB a block)
    const T* x = static_cast<const T*>(a.x);  // h may alias x: no restrict
    T* h = static_cast<T*>(a.h);
    const int D = a.D, nck = D / EPC;  // D % 8 == 0
    const int64_t row0 = (int64_t)blockIdx.x * kSeamRows;
    const int nrows = (int)min<int64_t>(kSeamRows, a.rows - row0);
    const int tid = threadIdx.x;
    const int pi = tid - kWave;  // producer index (negative in wave 0)
    const int nstage = (D + kStageCols - 1) / kStageCols;

    // ---- phase 1: inverse RMS of each row ----
    // x arrives through a ring of kRing stages in registers (the loads of a
    // stage are issued kRing - 1 stages before its squares go to LDS).  The
    // loads are unconditional (chunks outside the rows, past D or past the
    // stage read a valid chunk instead) and the stash zeroes or skips what
    // lies outside: a load under a branch is waited for at the branch's join.
    uint4 ring[kRing][kLoads];
    auto inside = [&](int st, int j) {
        const int i = pi + j * kProducers;
        return i < kChunks && i / kRowChunks < nrows && st * kRowChunks + i % kRowChunks < nck;
    };
    auto fetch = [&](int st, uint4* ld) {
#pragma unroll
        for (int j = 0; j < kLoads; ++j) {
            const int i = min(pi + j * kProducers, kChunks - 1);
            const int r = min(i / kRowChunks, nrows - 1);
            const int c = inside(st, j) ? st * kRowChunks + i % kRowChunks : 0;
            ld[j] = *reinterpret_cast<const uint4*>(x + (row0 + r) * (int64_t)D + (int64_t)c * EPC);
        }
    };
    auto stash = [&](const uint4* ld, int st) {  // the squares, rounded to f32
#pragma unroll
        for (int j = 0; j < kLoads; ++j) {
            const int i = pi + j * kProducers;
            const bool in = inside(st, j);
            Vec16<T> t;
            __builtin_memcpy(&t, &ld[j], 16);
            float sq[EPC];
#pragma unroll
            for (int e = 0; e < EPC; ++e) {
                const float v = Elt<T>::to_f32(t.v[e]);
                const float q = mul_rn(v, v);
                sq[e] = in ? q : 0.0f;  // zeros: acc + 0 == acc
            }
            if (i < kChunks) {
                unsigned char* dst = s_buf + (st & 1) * kStageBytes + (i / kRowChunks) * kRowStride +
                                     (i % kRowChunks) * EPC * 4;
#pragma unroll
                for (int q = 0; q < EPC / 4; ++q)
                    *reinterpret_cast<float4*>(dst + 16 * q) =
                        make_float4(sq[4 * q], sq[4 * q + 1], sq[4 * q + 2], sq[4 * q + 3]);
            }
        }
    };
    // Producers and the adder run separate loops with the same barriers (one
    // per stage): a branch inside one loop would hide from the compiler that
    // a producer's ring slot had kRing - 1 stages of loads issued after it.
    float acc = 0.0f;
    if (tid >= kWave) {
#pragma unroll
        for (int p = 0; p < kRing; ++p) fetch(p, ring[p]);
        stash(ring[0], 0);
        fetch(kRing, ring[0]);
        __syncthreads();
        // stage st sits in ring slot st % kRing, LDS half st & 1.  Stages past the
        // end stash zeros nobody reads and load a valid chunk.
        for (int st0 = 0; st0 < nstage; st0 += kRing) {
#pragma unroll
            for (int p = 0; p < kRing; ++p) {
                const int st = st0 + p;
                if (st >= nstage) break;
                stash(ring[(p + 1) % kRing], st + 1);
                fetch(st + 1 + kRing, ring[(p + 1) % kRing]);
                __syncthreads();
            }
        }
    } else {
        if (tid < kSeamRows) s_seqidx[tid] = (int)((row0 + min(tid, nrows - 1)) / a.seq - row0 / a.seq);
        __syncthreads();
        for (int st0 = 0; st0 < nstage; st0 += kRing) {
#pragma unroll
            for (int p = 0; p < kRing; ++p) {
                const int st = st0 + p;
                if (st >= nstage) break;
                const unsigned char* rowp = s_buf + (st & 1) * kStageBytes + (tid % kSeamRows) * kRowStride;
                // the reads of the next 8 pieces go out before 8 are added
                constexpr int kP = 8;
                float4 q[2][kP];
#pragma unroll
                for (int i = 0; i < kP; ++i) q[0][i] = *reinterpret_cast<const float4*>(rowp + i * 16);
#pragma unroll
                for (int c = 0; c < kStageCols / 4; c += kP) {
                    const int b = c / kP % 2;
                    if (c + kP < kStageCols / 4) {
#pragma unroll
                        for (int i = 0; i < kP; ++i)
                            q[b ^ 1][i] = *reinterpret_cast<const float4*>(rowp + (c + kP + i) * 16);
                    }
                    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                    for (int i = 0; i < kP; ++i) {
                        acc = add_nc(acc, q[b][i].x);
                        acc = add_nc(acc, q[b][i].y);
                        acc = add_nc(acc, q[b][i].z);
                        acc = add_nc(acc, q[b][i].w);
                    }
                }
                __syncthreads();
            }
        }
    }
    if (tid < kSeamRows) s_inv[tid] = seam_inv_rms(acc, D, a.eps);
    __syncthreads();

    // ---- phase 2: h ----
    // Chunk c of rows g kRowGroup .. + kRowGroup - 1, the rows' loads in flight
    // together; each thread reads only the chunks it writes (h may alias x).
    const int64_t b0 = row0 / a.seq;
    for (int q = tid; q < nck * (kSeamRows / kRowGroup); q += kSeamThreads) {
        const int g = q / nck, col = (q - g * nck) * EPC, r0 = g * kRowGroup;
        if (r0 >= nrows) break;
        uint4 v[kRowGroup];
#pragma unroll
        for (int u = 0; u < kRowGroup; ++u)  // past the end: the last row again, not stored
            v[u] = *reinterpret_cast<const uint4*>(x + (row0 + min(r0 + u, nrows - 1)) * (int64_t)D + col);
        float w[EPC], sc[EPC], sh[EPC];
#pragma unroll
        for (int e = 0; e < EPC; ++e) w[e] = 1.0f;  // norm_w null: gain 1
        if (a.norm_w) load_f32s<EPC>(a.norm_w + col, w);
        int seq = -1;
#pragma unroll
        for (int u = 0; u < kRowGroup; ++u) {
            const int r = r0 + u;
            if (r >= nrows) break;
            if (s_seqidx[r] != seq) {
                seq = s_seqidx[r];
                load_f32s<EPC>(a.scale + (b0 + seq) * D + col, sc);
                load_f32s<EPC>(a.shift + (b0 + seq) * D + col, sh);
            }
            const float inv = s_inv[r];
            Vec16<T> t;
            __builtin_memcpy(&t, &v[u], 16);
#pragma unroll
            for (int e = 0; e < EPC; ++e)
                t.v[e] = Elt<T>::from_f32(seam_h<T>(Elt<T>::to_f32(t.v[e]), inv, w[e], sc[e], sh[e]));
            uint4 o;
            __builtin_memcpy(&o, &t, 16);
            *reinterpret_cast<uint4*>(h + (row0 + r) * (int64_t)D + col) = o;
        }
    }
}

template <typename T>
hipError_t launch_seam_h_t(const SeamArgs& a, hipStream_t s) {
    const int64_t nblk = (a.rows + kSeamRows - 1) / kSeamRows;
    if (nblk == 0) return hipSuccess;
    if (nblk > 0x7fffffff) return hipErrorInvalidValue;
    launch_kernel(seam_h_kernel<T>, dim3((unsigned)nblk), dim3(kSeamThreads), 0, s, a);
    return hipGetLastError();
}

// out = x + y * gate (block.rs:101) on its own, for a feed-forward whose last
// kernel does not apply it: 16 bytes of each operand per thread; each thread
// reads the elements it writes, so out may alias x or y.
template <typename T>
__global__ __launch_bounds__(256) void gated_residual_kernel(const T* x, const T* y,
                                                             const float* __restrict__ gate,
                                                             T* out, int64_t rows, int D,
                                                             int64_t seq) {
    constexpr int EPC = 16 / sizeof(T);
    const int nck = D / EPC;
    const int64_t total = rows * nck;
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < total;
         i += (int64_t)gridDim.x * blockDim.x) {
        const int64_t row = i / nck;
        const int64_t off = row * D + (i % nck) * EPC;
        float xv[EPC], yv[EPC], g[EPC];
        load16(x + off, xv);
        load16(y + off, yv);
        load_f32s<EPC>(gate + row / seq * D + (i % nck) * EPC, g);
#pragma unroll
        for (int e = 0; e < EPC; ++e) xv[e] = seam_residual<T>(xv[e], yv[e], g[e]);
        store16(out + off, xv);
    }
}

template <typename T>
hipError_t launch_residual_t(const void* x, const void* y, const float* gate, void* out,
                             int64_t rows, int D, int64_t seq, hipStream_t s) {
    const int64_t total = rows * (D / (16 / (int)sizeof(T)));
    if (total == 0) return hipSuccess;
    const int64_t blocks = std::min<int64_t>((total + 255) / 256, 256 * 16);
    launch_kernel(gated_residual_kernel<T>, dim3((unsigned)blocks), dim3(256), 0, s,
                  (const T*)x, (const T*)y, gate, (T*)out, rows, D, seq);
    return hipGetLastError();
}

}  // namespace

hipError_t launch_gated_residual(DType dt, const void* x, const void* y, const float* gate,
                                 void* out, int64_t rows, int D, int64_t seq, hipStream_t s) {
    if (!x || !y || !gate || !out || seq < 1 || D <= 0 || D % 8 != 0 || rows < 0)
        return hipErrorInvalidValue;
    switch (dt) {
        case DType::F32: return launch_residual_t<float>(x, y, gate, out, rows, D, seq, s);
        case DType::BF16: return launch_residual_t<__bf16>(x, y, gate, out, rows, D, seq, s);
        case DType::F16: return launch_residual_t<_Float16>(x, y, gate, out, rows, D, seq, s);
    }
    return hipErrorInvalidValue;
}

hipError_t launch_seam_h(DType dt, const SeamArgs& a, hipStream_t s) {
    if (!a.x || !a.h || !a.shift || !a.scale || a.seq < 1 || a.D <= 0 || a.D % 8 != 0 ||
        a.rows < 0)
        return hipErrorInvalidValue;
    switch (dt) {
        case DType::F32: return launch_seam_h_t<float>(a, s);
        case DType::BF16: return launch_seam_h_t<__bf16>(a, s);
        case DType::F16: return launch_seam_h_t<_Float16>(a, s);
    }
    return hipErrorInvalidValue;
}

}  // namespace nomas

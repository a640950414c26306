// Copies between pageable host memory and the device for the host-tensor
// forward: through pinned staging buffers of one chunk each, so
// that the host-side memcpy of one chunk (spread over a small pool of worker
// threads) overlaps the DMA of earlier ones.  The first chunk's memcpy is what
// no DMA hides, and every chunk wakes the workers: 4 MB, 70 us on either side, and
// 8 MB where there are many (123 MB each way, both pageable: 4 MB 5,800, 8 MB 5,430, 16 MB
// 5,660 us; 55 MB 2,600 / 2,240 / 2,280; 29 MB 1,320 / 1,310 / 1,500, and 8 MB buffers take
// 1.2 ms more to allocate on a handle's first call).  hipMemcpy from pageable
// memory stages through the runtime's own buffers with one host thread and
// reached about 19 GB/s here; pinned-to-device DMA runs at about 55 GB/s.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstring>
#include <thread>

#include "host.hpp"

namespace nomas {

namespace {
// bytes per chunk (and staging buffer) of calls of up to kLongCall bytes, and of longer ones
constexpr size_t kChunk = (size_t)4 << 20, kLongChunk = (size_t)8 << 20, kLongCall = (size_t)40 << 20;
constexpr size_t kMinSplit = (size_t)1 << 20;  // smaller copies stay on the calling thread
}  // namespace

CopyPool::CopyPool(int workers) : parts_(workers + 1) {
    for (int i = 0; i < workers; ++i) threads_.emplace_back([this, i] { loop(i + 1); });
}

CopyPool::~CopyPool() {
    {
        std::lock_guard<std::mutex> l(m_);
        stop_ = true;
    }
    cv_work_.notify_all();
    for (std::thread& t : threads_) t.join();
}

// Part p of the current copy: 64-byte aligned slices, the last one takes the rest.
void CopyPool::range(int p, size_t* b, size_t* e) const {
    const size_t per = (n_ / parts_ + 63) & ~(size_t)63;
    *b = std::min(n_, (size_t)p * per);
    *e = p == parts_ - 1 ? n_ : std::min(n_, *b + per);
}

void CopyPool::loop(int p) {
    uint64_t seen = 0;
    for (;;) {
        {
            std::unique_lock<std::mutex> l(m_);
            cv_work_.wait(l, [&] { return stop_ || gen_ != seen; });
            if (stop_) return;
            seen = gen_;
        }
        size_t b, e;
        range(p, &b, &e);
        if (e > b) std::memcpy(dst_ + b, src_ + b, e - b);
        std::lock_guard<std::mutex> l(m_);
        if (--remaining_ == 0) cv_done_.notify_one();
    }
}

void CopyPool::copy(void* dst, const void* src, size_t n) {
    if (n < kMinSplit || parts_ == 1) {
        std::memcpy(dst, src, n);
        return;
    }
    {
        std::lock_guard<std::mutex> l(m_);
        dst_ = static_cast<unsigned char*>(dst);
        src_ = static_cast<const unsigned char*>(src);
        n_ = n;
        remaining_ = parts_ - 1;
        ++gen_;
    }
    cv_work_.notify_all();
    size_t b, e;
    range(0, &b, &e);
    if (e > b) std::memcpy(dst_ + b, src_ + b, e - b);
    std::unique_lock<std::mutex> l(m_);
    cv_done_.wait(l, [&] { return remaining_ == 0; });
}

// Host memory that is already pinned (hipHostMalloc'd, or a framework's pinned
// tensor) goes straight to the DMA engine.  hipPointerGetAttributes fails on
// pageable memory; that error is cleared so that a later launch check does
// not report it.
bool is_pinned(const void* p) {
    hipPointerAttribute_t at;
    const hipError_t e = hipPointerGetAttributes(&at, p);
    if (e != hipSuccess) {
        (void)hipGetLastError();
        return false;
    }
    return at.type == hipMemoryTypeHost;
}

HostStager::~HostStager() { release(); }

void HostStager::begin(size_t bytes) {
    chunk_ = bytes > kLongCall ? kLongChunk : kChunk;
    next_ = 0;
}

void HostStager::release() {
    for (int b = 0; b < kBufs; ++b) {
        if (ev_[b]) (void)hipEventDestroy(ev_[b]);
        if (pin_[b]) (void)hipHostFree(pin_[b]);
        ev_[b] = nullptr;
        pin_[b] = nullptr;
    }
    pool_.reset();
}

// All or nothing: a failed set-up leaves nothing behind, and the next call tries again.
int HostStager::ensure() {
    if (pool_ && cap_ >= chunk_) return NOMAS_OK;
    for (int b = 0; pool_ && b < kBufs; ++b) (void)hipEventSynchronize(ev_[b]);  // larger ones are needed
    release();
    cap_ = chunk_;
    for (int b = 0; b < kBufs; ++b) {
        hipError_t e = hipHostMalloc(&pin_[b], cap_, hipHostMallocDefault);
        if (e != hipSuccess) {
            pin_[b] = nullptr;
            release();
            return set_error(NOMAS_ERR_OUT_OF_MEMORY, "hipHostMalloc of a staging buffer failed: %s",
                             hipGetErrorString(e));
        }
        e = hipEventCreateWithFlags(&ev_[b], hipEventDisableTiming);
        if (e != hipSuccess) {
            ev_[b] = nullptr;
            release();
            return set_error(NOMAS_ERR_HIP, "hipEventCreate failed: %s", hipGetErrorString(e));
        }
    }
    const unsigned hw = std::thread::hardware_concurrency();
    pool_.reset(new CopyPool((int)std::min(7u, hw > 2 ? hw / 2 - 1 : 0u)));
    return NOMAS_OK;
}

#define STAGE_TRY(expr, what)                                                                  \
    do {                                                                                       \
        hipError_t _e = (expr);                                                                \
        if (_e != hipSuccess) return set_error(NOMAS_ERR_HIP, "%s failed: %s", what, hipGetErrorString(_e)); \
    } while (0)

int HostStager::to_device(void* dst, const void* src, size_t bytes, hipStream_t s) {
    if (is_pinned(src)) {
        STAGE_TRY(hipMemcpyAsync(dst, src, bytes, hipMemcpyHostToDevice, s), "hipMemcpyAsync H2D");
        return NOMAS_OK;
    }
    int rc = ensure();
    if (rc != NOMAS_OK) return rc;
    const unsigned char* in = static_cast<const unsigned char*>(src);
    unsigned char* out = static_cast<unsigned char*>(dst);
    for (size_t off = 0; off < bytes; off += chunk_) {
        const size_t n = std::min(chunk_, bytes - off);
        const int b = next_;
        next_ = (next_ + 1) % kBufs;
        // buffer b drained (its last DMA may belong to an earlier call: the
        // pieces of a host forward stage one after another)
        STAGE_TRY(hipEventSynchronize(ev_[b]), "hipEventSynchronize");
        pool_->copy(pin_[b], in + off, n);
        STAGE_TRY(hipMemcpyAsync(out + off, pin_[b], n, hipMemcpyHostToDevice, s), "hipMemcpyAsync H2D");
        STAGE_TRY(hipEventRecord(ev_[b], s), "hipEventRecord");
    }
    return NOMAS_OK;
}

int HostStager::to_host(void* dst, const void* src, size_t bytes, hipStream_t s) {
    if (is_pinned(dst)) {
        STAGE_TRY(hipMemcpyAsync(dst, src, bytes, hipMemcpyDeviceToHost, s), "hipMemcpyAsync D2H");
        STAGE_TRY(hipStreamSynchronize(s), "hipStreamSynchronize");
        return NOMAS_OK;
    }
    int rc = ensure();
    if (rc != NOMAS_OK) return rc;
    const unsigned char* in = static_cast<const unsigned char*>(src);
    unsigned char* out = static_cast<unsigned char*>(dst);
    // up to kBufs chunks' DMAs in flight; the host copies the oldest one out
    // when it has landed.  (The buffers' earlier DMAs, into the device, may
    // still be in flight on the first round.)
    const int64_t chunks = (int64_t)((bytes + chunk_ - 1) / chunk_);
    const int first = next_;
    next_ = (int)((next_ + chunks) % kBufs);
    auto len = [&](int64_t c) { return std::min(chunk_, bytes - (size_t)c * chunk_); };
    for (int64_t c = 0; c < chunks + kBufs - 1; ++c) {
        const int64_t done = c - (kBufs - 1);
        if (done >= 0) {
            const int b = (int)((first + done) % kBufs);
            STAGE_TRY(hipEventSynchronize(ev_[b]), "hipEventSynchronize");
            pool_->copy(out + (size_t)done * chunk_, pin_[b], len(done));
        }
        if (c < chunks) {
            const int b = (int)((first + c) % kBufs);
            if (c < kBufs) STAGE_TRY(hipEventSynchronize(ev_[b]), "hipEventSynchronize");
            STAGE_TRY(hipMemcpyAsync(pin_[b], in + (size_t)c * chunk_, len(c), hipMemcpyDeviceToHost, s),
                      "hipMemcpyAsync D2H");
            STAGE_TRY(hipEventRecord(ev_[b], s), "hipEventRecord");
        }
    }
    return NOMAS_OK;
}

#undef STAGE_TRY

}  // namespace nomas

// jy_stage.cpp — the pinned ring of jy_stage.h.
#include "jy_stage.h"

#include <algorithm>
#include <atomic>
#include <cstring>
#include <system_error>
#include <thread>

namespace jy {

namespace {

__global__ __launch_bounds__(256) void stage_copy16_kernel(const uint4* __restrict__ s, uint4* __restrict__ d, size_t n) {
    const size_t i = (size_t)blockIdx.x * 256 + threadIdx.x;
    if (i < n) d[i] = s[i];
}
__global__ __launch_bounds__(256) void stage_copy4_kernel(const uint32_t* __restrict__ s, uint32_t* __restrict__ d, size_t n) {
    const size_t i = (size_t)blockIdx.x * 256 + threadIdx.x;
    if (i < n) d[i] = s[i];
}

void launch_copy(const void* s, void* d, size_t bytes, hipStream_t st) {
    const bool w = bytes % 16 == 0 && (uintptr_t)d % 16 == 0;
    const size_t n = bytes / (w ? 16 : 4);
    const dim3 grid((unsigned)((n + 255) / 256));
    if (w)
        hipLaunchKernelGGL(stage_copy16_kernel, grid, dim3(256), 0, st, (const uint4*)s, (uint4*)d, n);
    else
        hipLaunchKernelGGL(stage_copy4_kernel, grid, dim3(256), 0, st, (const uint32_t*)s, (uint32_t*)d, n);
}

// The pieces of a transfer's chunks, claimed in order by whoever is free; a piece may be
// claimed once its chunk is opened.  Nothing but help() allocates.
template <class Copy>  // copy(chunk, offset in it, bytes)
class Team {
  public:
    static constexpr size_t PIECE = (size_t)64 << 10;

    Team(size_t chunk, size_t last, size_t nch, const Copy& copy)
        : chunk_(chunk), last_(last), nch_(nch), per_((chunk + PIECE - 1) / PIECE),
          total_((nch - 1) * per_ + (last + PIECE - 1) / PIECE), copy_(copy) {}
    ~Team() {
        next_.store(total_);  // (after an error: no more claims)
        for (std::thread& t : threads_)
            if (t.joinable()) t.join();
    }
    void help() {
        const int n = std::min(HostStage::HELPERS, (int)std::thread::hardware_concurrency() - 1);
        try {
            for (int i = 0; i < n; i++)
                threads_[i] = std::thread([this] {
                    for (int spin = 0; next_.load(std::memory_order_relaxed) < total_;) {
                        if (work())
                            spin = 0;
                        else if (++spin > 64)
                            std::this_thread::yield();
                    }
                });
        } catch (const std::system_error&) {  // no thread to be had: the caller copies alone
        }
    }
    // (the caller's thread) the next chunk, whose slot's last chunk is complete
    void open_next() {
        done_[opened_ % HostStage::SLOTS].store(0, std::memory_order_relaxed);
        opened_++;
        limit_.store(std::min(opened_ * per_, total_), std::memory_order_release);
    }
    size_t opened() const { return opened_; }
    // one piece, if an opened one is left
    bool work() {
        size_t i = next_.load(std::memory_order_relaxed);
        do {
            if (i >= limit_.load(std::memory_order_acquire)) return false;
        } while (!next_.compare_exchange_weak(i, i + 1));
        const size_t c = i / per_, off = (i - c * per_) * PIECE;
        copy_(c, off, std::min(PIECE, (c + 1 == nch_ ? last_ : chunk_) - off));
        done_[c % HostStage::SLOTS].fetch_add(1, std::memory_order_release);
        return true;
    }
    // (the caller's thread) whether chunk c, one of the last SLOTS opened or not opened yet, is copied
    bool complete(size_t c) const {
        const size_t n = ((c + 1 == nch_ ? last_ : chunk_) + PIECE - 1) / PIECE;
        return c < opened_ && done_[c % HostStage::SLOTS].load(std::memory_order_acquire) == n;
    }

  private:
    const size_t chunk_, last_, nch_, per_, total_;
    size_t opened_ = 0;
    std::atomic<size_t> next_{0}, limit_{0};
    std::atomic<unsigned> done_[HostStage::SLOTS] = {};  // pieces copied of the chunk in each slot
    const Copy& copy_;
    std::thread threads_[HostStage::HELPERS];
};

}  // namespace

bool HostStage::ready(size_t n, bool create) {
    if (ring_) return true;
    if (n <= SMALL) {
        if (!small_ && create && !tried_small_) {
            tried_small_ = true;
            void* p = nullptr;
            if (hipHostMalloc(&p, SMALL, hipHostMallocDefault) == hipSuccess)
                small_ = static_cast<unsigned char*>(p);
            else
                (void)hipGetLastError();
        }
        return small_ != nullptr;
    }
    if (!create || tried_) return false;
    tried_ = true;
    return init();
}

bool HostStage::init() {
    void* p = nullptr;
    bool ok = hipHostMalloc(&p, SLOT * SLOTS, hipHostMallocDefault) == hipSuccess;
    ring_ = ok ? static_cast<unsigned char*>(p) : nullptr;
    for (int i = 0; ok && i < SLOTS; i++) ok = hipEventCreateWithFlags(&ev_[i], hipEventDisableTiming) == hipSuccess;
    if (!ok) {
        free_ring();
        (void)hipGetLastError();
    }
    return ok;
}

void HostStage::free_ring() {
    for (hipEvent_t& e : ev_) {
        if (e) (void)hipEventDestroy(e);
        e = nullptr;
    }
    if (ring_) (void)hipHostFree(ring_);
    ring_ = nullptr;
}

void HostStage::release() {
    free_ring();
    if (small_) (void)hipHostFree(small_);
    small_ = nullptr;
}

// the ring free of an earlier transfer that ended in an error
hipError_t HostStage::idle(hipStream_t st) {
    if (!busy_) return hipSuccess;
    const hipError_t e = hipStreamSynchronize(st);
    if (e == hipSuccess) busy_ = false;
    return e;
}

hipError_t HostStage::to_device(void* dst, const void* src, size_t n, hipStream_t st, bool threads) {
    hipError_t e = idle(st);
    if (e != hipSuccess || n == 0) return e;
    busy_ = true;  // (until to_host has waited for the stream)
    const size_t nch = (n + SLOT - 1) / SLOT, last = n - (nch - 1) * SLOT;
    auto* d = static_cast<unsigned char*>(dst);
    auto* s = static_cast<const unsigned char*>(src);
    if (nch == 1) {
        memcpy(one(), s, n);
        launch_copy(one(), d, n, st);
        return hipGetLastError();
    }
    auto copy = [&](size_t c, size_t off, size_t len) {
        memcpy(ring_ + (c % SLOTS) * SLOT + off, s + c * SLOT + off, len);
    };
    Team<decltype(copy)> team(SLOT, last, nch, copy);
    while (team.opened() < std::min<size_t>(nch, SLOTS)) team.open_next();
    if (threads && n >= MT_BYTES) team.help();
    size_t sent = 0;
    while (sent < nch) {
        if (team.complete(sent)) {
            launch_copy(ring_ + (sent % SLOTS) * SLOT, d + sent * SLOT, sent + 1 == nch ? last : SLOT, st);
            if ((e = hipGetLastError()) != hipSuccess) return e;
            if ((e = hipEventRecord(ev_[sent % SLOTS], st)) != hipSuccess) return e;
            sent++;
        } else if (!team.work() && team.opened() == nch) {
            std::this_thread::yield();
        }
        // a slot is free again once the copy of the chunk it held has run
        while (team.opened() < nch && team.opened() - SLOTS < sent) {
            e = hipEventQuery(ev_[team.opened() % SLOTS]);
            if (e == hipErrorNotReady) {
                (void)hipGetLastError();  // (an answer, not an error to be found after the next launch)
                break;
            }
            if (e != hipSuccess) return e;
            team.open_next();
        }
    }
    return hipSuccess;
}

hipError_t HostStage::to_host(void* dst, size_t rows, size_t row_bytes, hipStream_t st, RowProducer produce,
                              bool threads) {
    if (row_bytes > SLOT) return hipErrorInvalidValue;
    hipError_t e = hipSuccess;
    busy_ = true;
    const size_t rpc = SLOT / row_bytes, nch = (rows + rpc - 1) / rpc;
    const size_t chunk = rpc * row_bytes, last = rows * row_bytes - (nch - 1) * chunk;
    auto* d = static_cast<unsigned char*>(dst);
    // (the slots' copies to the GPU are ahead of the producers on the stream)
    if (nch == 1) {
        produce(0, rows, one());
        if ((e = hipGetLastError()) != hipSuccess || (e = hipStreamSynchronize(st)) != hipSuccess) return e;
        busy_ = false;
        memcpy(d, one(), rows * row_bytes);
        return hipSuccess;
    }
    auto copy = [&](size_t c, size_t off, size_t len) {
        memcpy(d + c * chunk + off, ring_ + (c % SLOTS) * SLOT + off, len);
    };
    Team<decltype(copy)> team(chunk, last, nch, copy);
    size_t sent = 0, copied = 0;
    auto send = [&]() {
        produce(sent * rpc, std::min(rpc, rows - sent * rpc), ring_ + (sent % SLOTS) * SLOT);
        if ((e = hipGetLastError()) == hipSuccess) e = hipEventRecord(ev_[sent % SLOTS], st);
        sent++;
        return e == hipSuccess;
    };
    while (sent < std::min<size_t>(nch, SLOTS))
        if (!send()) return e;
    if ((e = hipEventSynchronize(ev_[0])) != hipSuccess) return e;  // (the call's work before it)
    team.open_next();
    if (threads && rows * row_bytes >= MT_BYTES) team.help();
    while (copied < nch) {
        while (team.opened() < sent) {
            e = hipEventQuery(ev_[team.opened() % SLOTS]);
            if (e == hipErrorNotReady) {
                (void)hipGetLastError();
                break;
            }
            if (e != hipSuccess) return e;
            team.open_next();
        }
        if (team.complete(copied)) {
            copied++;
            if (sent < nch && !send()) return e;
        } else if (!team.work()) {
            std::this_thread::yield();
        }
    }
    e = hipStreamSynchronize(st);
    if (e == hipSuccess) busy_ = false;
    return e;
}

}  // namespace jy

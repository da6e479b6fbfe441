// jy_stage.h — rows between the caller's (pageable) memory and the GPU through a small ring
// of pinned memory.
#pragma once

#include <hip/hip_runtime.h>

#include <cstddef>
#include <functional>

namespace jy {

// One ring per model: SLOTS slots of SLOT bytes.  The GPU side of a transfer is a kernel that
// reads or writes a slot (to_device's copy; to_host's producer, which may be the kernel that
// computes the rows), the host side memcpy by the calling thread and, from MT_BYTES on, up to
// HELPERS threads that live for the transfer; the two overlap chunk by chunk.
// The runtime's own copy of pageable memory stages it on one thread, copy after copy: 1024 x
// 4096 floats to the GPU and back took about 2.4 ms of a call, against 0.6 for the bytes over
// the bus.
class HostStage {
  public:
    static constexpr size_t SLOT = (size_t)512 << 10, MT_BYTES = (size_t)1 << 20;
    static constexpr int SLOTS = 8, HELPERS = 3;

    // allocates; false (and no ring: the calls below may not be made) where it cannot
    bool init();
    void release();
    bool ready() const { return ring_ != nullptr; }

    // dst (device) = src, n bytes (a multiple of 4), in order on st; src may be reused at once
    hipError_t to_device(void* dst, const void* src, size_t n, hipStream_t st);
    // dst = `rows` rows of row_bytes (a multiple of 4, at most SLOT), which produce(first row,
    // rows, where) writes by kernels it enqueues on st; all of it has arrived, and st is idle, on return
    hipError_t to_host(void* dst, size_t rows, size_t row_bytes, hipStream_t st,
                       const std::function<void(size_t, size_t, void*)>& produce);

  private:
    hipError_t idle(hipStream_t st);
    unsigned char* ring_ = nullptr;
    hipEvent_t ev_[SLOTS] = {};
    bool busy_ = false;  // a transfer was begun and not seen to its end
};

}  // namespace jy

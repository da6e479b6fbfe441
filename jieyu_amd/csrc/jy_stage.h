// jy_stage.h — rows between the caller's (pageable) memory and the GPU through a small ring
// of pinned memory.
#pragma once

#include <hip/hip_runtime.h>

#include <cstddef>

namespace jy {

// produce(first row, rows, where) of to_host: a callable by reference, for the length of the call
// (std::function may allocate)
class RowProducer {
  public:
    template <class F>
    RowProducer(const F& f)
        : ctx_(&f), call_([](const void* c, size_t r0, size_t n, void* where) {
              (*static_cast<const F*>(c))(r0, n, where);
          }) {}
    void operator()(size_t r0, size_t n, void* where) const { call_(ctx_, r0, n, where); }

  private:
    const void* ctx_;
    void (*call_)(const void*, size_t, size_t, void*);
};

// One ring per model: SLOTS slots of SLOT bytes (calls of one row or few: SMALL bytes).  The GPU side
// of a transfer is a kernel that reads or writes a slot (to_device's copy; to_host's producer,
// which may be the kernel that computes the rows), the host side memcpy by the calling thread
// and, with `threads` and from MT_BYTES on, up to HELPERS threads that live for the transfer; the
// two overlap chunk by chunk.
// Without `threads` a transfer allocates nothing.
// The runtime's own copy of pageable memory stages it on one thread, copy after copy: 1024 x
// 4096 floats to the GPU and back took about 2.4 ms of a call, against 0.6 for the bytes over
// the bus.
class HostStage {
  public:
    static constexpr size_t SLOT = (size_t)512 << 10, MT_BYTES = (size_t)1 << 20;
    static constexpr size_t SMALL = (size_t)64 << 10;
    static constexpr int SLOTS = 8, HELPERS = 3;

    // whether a transfer of n bytes has pinned memory (else the calls below may not be made).  With
    // `create` the first call that needs it makes it, and where it cannot no later one tries: one
    // row or few (n <= SMALL) take a small buffer, more the ring, and a model that never takes rows from
    // the host (generation, sessions) holds neither.  (20-50 us and 50-300 us of that call; the first
    // touch of its pages, ~0.4 us per KiB used, falls on the calls that use them either way.)
    bool ready(size_t n, bool create);
    void release();

    // dst (device) = src, n bytes (a multiple of 4), in order on st; src may be reused at once
    hipError_t to_device(void* dst, const void* src, size_t n, hipStream_t st, bool threads);
    // dst = `rows` rows of row_bytes (a multiple of 4, at most SLOT), which produce(first row,
    // rows, where) writes by kernels it enqueues on st; all of it has arrived, and st is idle, on return
    hipError_t to_host(void* dst, size_t rows, size_t row_bytes, hipStream_t st, RowProducer produce, bool threads);

  private:
    bool init();
    void free_ring();
    hipError_t idle(hipStream_t st);
    unsigned char* one() const { return ring_ ? ring_ : small_; }  // a transfer of one chunk
    unsigned char* small_ = nullptr;
    unsigned char* ring_ = nullptr;
    hipEvent_t ev_[SLOTS] = {};
    bool tried_small_ = false, tried_ = false;
    bool busy_ = false;  // a transfer was begun and not seen to its end
};

}  // namespace jy

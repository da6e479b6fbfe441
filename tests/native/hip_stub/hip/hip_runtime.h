// Just enough of the HIP runtime for jy_stage.cpp in a host build: one in-order stream whose
// operations wait in a queue until something waits for them (or hipEventQuery lets one run), so
// that host code that reuses memory too early finds it unread or unwritten.  Device memory is
// host memory.  The queue is fixed and the operations are stored in it: nothing here allocates.
#pragma once

#include <atomic>
#include <cstddef>
#include <cstdint>
#include <cstdlib>
#include <cstring>
#include <new>
#include <type_traits>

#define __global__ static
#define __launch_bounds__(n)
#define __restrict__ __restrict

struct uint4 {
    unsigned x, y, z, w;
};
struct dim3 {
    unsigned x, y, z;
    dim3(unsigned x_ = 1, unsigned y_ = 1, unsigned z_ = 1) : x(x_), y(y_), z(z_) {}
};
inline dim3 blockIdx, threadIdx;

enum hipError_t { hipSuccess = 0, hipErrorInvalidValue = 1, hipErrorOutOfMemory = 2, hipErrorNotReady = 600 };
typedef struct StubEvent {
    size_t at = 0;  // operations recorded before it
} * hipEvent_t;
typedef void* hipStream_t;
enum { hipHostMallocDefault = 0, hipEventDisableTiming = 2 };

namespace hip_stub {

struct Op {
    alignas(16) unsigned char data[128];
    void (*run)(void*);
};
inline Op g_ops[4096];
inline size_t g_put = 0, g_done = 0;
inline int g_host_allocs = 0, g_host_frees = 0, g_events = 0, g_live_events = 0;
inline int g_fail_host_malloc = 0, g_fail_event_at = 0, g_fail_record_in = 0;  // (0: never)

inline void run_to(size_t n) {
    while (g_done < n) {
        Op& o = g_ops[g_done % 4096];
        o.run(o.data);
        g_done++;
    }
}
template <class F>
void enqueue(const F& f) {
    static_assert(sizeof(F) <= sizeof(Op::data) && std::is_trivially_copyable<F>::value, "an operation");
    if (g_put - g_done == 4096) abort();
    Op& o = g_ops[g_put++ % 4096];
    new (o.data) F(f);
    o.run = [](void* p) { (*static_cast<F*>(p))(); };
}

}  // namespace hip_stub

#define hipLaunchKernelGGL(kernel, grid, block, lds, stream, ...)           \
    do {                                                                    \
        const dim3 g_ = (grid), b_ = (block);                               \
        hip_stub::enqueue([=]() {                                           \
            for (unsigned i_ = 0; i_ < g_.x; i_++)                          \
                for (unsigned t_ = 0; t_ < b_.x; t_++) {                    \
                    blockIdx.x = i_;                                        \
                    threadIdx.x = t_;                                       \
                    kernel(__VA_ARGS__);                                    \
                }                                                           \
        });                                                                 \
    } while (0)

inline hipError_t hipHostMalloc(void** p, size_t n, unsigned) {
    if (hip_stub::g_fail_host_malloc) return hipErrorOutOfMemory;
    hip_stub::g_host_allocs++;
    *p = aligned_alloc(4096, n);
    return hipSuccess;
}
inline hipError_t hipHostFree(void* p) {
    hip_stub::g_host_frees++;
    free(p);
    return hipSuccess;
}
inline hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) {
    if (hip_stub::g_fail_event_at && ++hip_stub::g_events == hip_stub::g_fail_event_at) return hipErrorOutOfMemory;
    *e = new StubEvent;
    hip_stub::g_live_events++;
    return hipSuccess;
}
inline hipError_t hipEventDestroy(hipEvent_t e) {
    delete e;
    hip_stub::g_live_events--;
    return hipSuccess;
}
inline hipError_t hipEventRecord(hipEvent_t e, hipStream_t) {
    if (hip_stub::g_fail_record_in && --hip_stub::g_fail_record_in == 0) return hipErrorInvalidValue;
    e->at = hip_stub::g_put;
    return hipSuccess;
}
inline hipError_t hipEventQuery(hipEvent_t e) {
    if (hip_stub::g_done < e->at) hip_stub::run_to(hip_stub::g_done + 1);
    return hip_stub::g_done < e->at ? hipErrorNotReady : hipSuccess;
}
inline hipError_t hipEventSynchronize(hipEvent_t e) {
    hip_stub::run_to(e->at);
    return hipSuccess;
}
inline hipError_t hipStreamSynchronize(hipStream_t) {
    hip_stub::run_to(hip_stub::g_put);
    return hipSuccess;
}
inline hipError_t hipGetLastError() { return hipSuccess; }

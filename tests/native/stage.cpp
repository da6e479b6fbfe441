// The pinned ring (jy_stage.cpp) over the stub runtime of hip_stub/: rows to the device and back,
// what it allocates, and what it does after a transfer that did not end.  Each check takes a case
// from the command line and exits 0.
#include <cstdio>
#include <vector>

#include "jy_stage.h"

using namespace jy;

static std::atomic<long> g_news{0};
void* operator new(size_t n) {
    g_news++;
    if (void* p = malloc(n ? n : 1)) return p;
    throw std::bad_alloc();
}
void operator delete(void* p) noexcept { free(p); }
void operator delete(void* p, size_t) noexcept { free(p); }

#define CHECK(x)                                                \
    do {                                                        \
        if (!(x)) {                                             \
            fprintf(stderr, "line %d: %s\n", __LINE__, #x);     \
            exit(1);                                            \
        }                                                       \
    } while (0)

static void fill(std::vector<uint32_t>& v, uint32_t seed) {
    for (size_t i = 0; i < v.size(); i++) v[i] = seed + (uint32_t)i * 2654435761u;
}

// rows x row floats to the device and back (the producer adds one), allocations counted
static long round_trip(HostStage& s, size_t rows, size_t row, bool threads, uint32_t seed) {
    std::vector<uint32_t> src(rows * row), dev(rows * row, 0xdeadbeef), out(rows * row, 0xdeadbeef);
    fill(src, seed);
    const std::vector<uint32_t> keep = src;
    uint32_t* d = dev.data();
    CHECK(s.ready(4 * src.size(), false));
    const long before = g_news;
    CHECK(s.to_device(d, src.data(), 4 * src.size(), nullptr, threads) == hipSuccess);
    for (uint32_t& x : src) x = 0;  // (it may be reused at once)
    const auto add1 = [&](size_t r0, size_t n, void* where) {
        const uint32_t* p = d + r0 * row;
        uint32_t* w = static_cast<uint32_t*>(where);
        const size_t k = n * row;
        hip_stub::enqueue([=]() {
            for (size_t i = 0; i < k; i++) w[i] = p[i] + 1;
        });
    };
    CHECK(s.to_host(out.data(), rows, 4 * row, nullptr, add1, threads) == hipSuccess);
    const long news = g_news - before;
    for (size_t i = 0; i < keep.size(); i++) CHECK(out[i] == keep[i] + 1);
    return news;
}

// (rows, row): inside a piece, inside a slot, a slot less a row, exactly and a row more, under and
// over the helpers' 1 MiB, the ring and a row more, several rings with an odd rest, 4-byte sizes
static const size_t SIZES[][2] = {{1, 1},      {3, 5},      {1, 4096},    {33, 4096},   {511, 256},  {512, 256},  {513, 256},
                                  {1023, 256}, {1025, 256}, {937, 1120},  {1024, 1024}, {1025, 1024}, {2307, 1024}, {53, 20480},
                                  {9, 131072}, {999, 1117}};

int main(int argc, char** argv) {
    const char* what = argc > 1 ? argv[1] : "";
    HostStage s;
    const size_t few = HostStage::SMALL, more = HostStage::SMALL + 4;
    if (!strcmp(what, "made_when_needed")) {
        CHECK(!s.ready(4, false) && !s.ready(more, false) && hip_stub::g_host_allocs == 0);
        CHECK(s.ready(few, true) && s.ready(4, false) && s.ready(few, true) && hip_stub::g_host_allocs == 1);
        CHECK(!s.ready(more, false) && hip_stub::g_live_events == 0);
        for (const auto& z : SIZES)
            if (4 * z[0] * z[1] <= few) round_trip(s, z[0], z[1], true, 9);
        CHECK(s.ready(more, true) && s.ready(more, false) && s.ready(4, true) && hip_stub::g_host_allocs == 2);
        for (const auto& z : SIZES) round_trip(s, z[0], z[1], true, 9);
        s.release();
        CHECK(hip_stub::g_host_frees == 2 && hip_stub::g_live_events == 0);
        // the ring first: nothing else is needed
        HostStage r;
        CHECK(r.ready(more, true) && r.ready(4, true) && hip_stub::g_host_allocs == 3);
        for (const auto& z : SIZES) round_trip(r, z[0], z[1], true, 9);
        r.release();
        // no pinned memory, or no k-th event: no ring, nothing left behind, no second try
        for (int k = 0; k <= HostStage::SLOTS; k++) {
            HostStage f;
            hip_stub::g_fail_host_malloc = k == 0;
            hip_stub::g_fail_event_at = k;
            hip_stub::g_events = 0;
            const int before = hip_stub::g_host_allocs;
            CHECK(!f.ready(more, true));
            if (k == 0) CHECK(!f.ready(few, true));
            hip_stub::g_fail_host_malloc = hip_stub::g_fail_event_at = 0;
            CHECK(!f.ready(more, true) && !f.ready(more, false));
            if (k == 0) CHECK(!f.ready(few, true) && !f.ready(few, false));
            CHECK(hip_stub::g_host_allocs == before + (k != 0) && hip_stub::g_host_allocs == hip_stub::g_host_frees);
            CHECK(hip_stub::g_live_events == 0);
            if (k != 0) {  // (few rows still have their buffer)
                CHECK(f.ready(few, true));
                round_trip(f, 3, 5, true, 9);
            }
            f.release();
        }
        CHECK(hip_stub::g_host_allocs == hip_stub::g_host_frees);
        return 0;
    }
    if (!strcmp(what, "after_an_error")) {  // few rows in, no rows out, then more
        CHECK(s.ready(few, true));
        std::vector<uint32_t> a(few / 4), da(few / 4), b(more / 4), db(more / 4);
        fill(a, 1);
        fill(b, 2);
        CHECK(s.to_device(da.data(), a.data(), few, nullptr, true) == hipSuccess);
        CHECK(s.ready(more, true));
        CHECK(s.to_device(db.data(), b.data(), more, nullptr, true) == hipSuccess);
        hipStreamSynchronize(nullptr);
        CHECK(da == a && db == b);
    }
    CHECK(s.ready(more, true));
    if (!strcmp(what, "round_trip")) {
        for (int pass = 0; pass < 3; pass++)
            for (const auto& z : SIZES) round_trip(s, z[0], z[1], pass != 1, 17 * pass + 1);
    } else if (!strcmp(what, "no_host_allocation")) {
        for (const auto& z : SIZES) CHECK(round_trip(s, z[0], z[1], false, 5) == 0);
    } else if (!strcmp(what, "after_an_error")) {
        // rows in, and the call fails before its rows out: the ring's copies still wait on the stream
        for (size_t n : {(size_t)100, (size_t)5 << 20}) {
            std::vector<uint32_t> a(n / 4), b(n / 4), da(n / 4), db(n / 4);
            fill(a, 1);
            fill(b, 2);
            CHECK(s.to_device(da.data(), a.data(), n, nullptr, true) == hipSuccess);
            CHECK(s.to_device(db.data(), b.data(), n, nullptr, true) == hipSuccess);
            hipStreamSynchronize(nullptr);
            CHECK(da == a && db == b);
        }
        // an event that cannot be recorded, at each of the first transfers of a call
        for (int k = 1; k <= 12; k++) {
            std::vector<uint32_t> src((size_t)5 << 18), dev(src.size()), out(src.size());
            fill(src, k);
            hip_stub::g_fail_record_in = k;
            const hipError_t e = s.to_device(dev.data(), src.data(), 4 * src.size(), nullptr, true);
            const auto none = [](size_t, size_t, void*) {};
            const hipError_t f = e == hipSuccess ? s.to_host(out.data(), 1280, 4096, nullptr, none, true) : e;
            CHECK(f == hipErrorInvalidValue);
            hip_stub::g_fail_record_in = 0;
            round_trip(s, 1025, 1024, true, k);
        }
        // a row that no slot holds
        uint32_t x = 0;
        const auto none = [](size_t, size_t, void*) { CHECK(!"produced"); };
        CHECK(s.to_host(&x, 1, HostStage::SLOT + 4, nullptr, none, true) == hipErrorInvalidValue);
        round_trip(s, 513, 256, true, 3);
    } else {
        CHECK(!"a case");
    }
    hipStreamSynchronize(nullptr);
    s.release();
    CHECK(hip_stub::g_host_allocs == hip_stub::g_host_frees && hip_stub::g_live_events == 0);
    return 0;
}

// Freed device blocks (pp_malloc, pp_free) on the host stand-in: see test_native_cpu.py for the cases.
#include <chrono>
#include <stdio.h>
#include <string>
#include <thread>

#include "hip_on_host.h"

#include "pp_copy.hip"
#include "pp_host.hip"

namespace pp_beam {
hipError_t init_noalloc_scratch(int) { return hipSuccess; }
}

static const size_t MIB = (size_t)1 << 20;

static void* get(size_t bytes) {
    void* p = nullptr;
    CHECK(pp_malloc(&p, bytes) == PP_OK && p);
    return p;
}

static void pause_ms(int ms) { std::this_thread::sleep_for(std::chrono::milliseconds(ms)); }

// a block is handed out again only after the device was waited for
static void reuse_waits() {
    void* a = get(MIB);
    void* during = nullptr;
    on_device_sync = [&] {
        on_device_sync = nullptr;
        during = get(MIB);          // another caller, while the free waits
    };
    CHECK(pp_free(a) == PP_OK);
    CHECK(device_syncs == 1 && during != a);
    CHECK(get(MIB) == a);
}

// two frees of one pointer at the same time: one of them is refused, and the block is kept once
static void double_free() {
    void* a = get(MIB);
    std::atomic<int> inside{0}, ok{0};
    on_device_sync = [&] {
        ++inside;
        for (int k = 0; k < 200 && inside < 2; ++k) pause_ms(1);
    };
    std::thread t[2];
    for (auto& x : t) x = std::thread([&] { ok += pp_free(a) == PP_OK; });
    for (auto& x : t) x.join();
    on_device_sync = nullptr;
    CHECK(ok == 1);
    void* b = get(MIB);
    CHECK(get(MIB) != b);           // no two owners
}

// a capture that begins while a free waits for the device: one of the two waits for the other
static void free_and_capture() {
    pp_stream s;
    CHECK(pp_stream_create(&s) == PP_OK);
    void* a = get(MIB);
    std::thread c;
    on_device_sync = [&] {
        on_device_sync = nullptr;
        c = std::thread([&] { CHECK(pp_graph_begin(s) == PP_OK); });
        pause_ms(100);
    };
    CHECK(pp_free(a) == PP_OK);
    c.join();
    CHECK(!sync_during_capture);
    // and while the capture runs frees do not wait for the device
    const int before = device_syncs;
    void* b = get(MIB);
    CHECK(pp_free(b) == PP_OK && device_syncs == before);
    pp_graph g = nullptr;
    CHECK(pp_graph_end(s, &g) == PP_OK);
    CHECK(!sync_during_capture);
}

// a stream destroyed while it records ends its capture: blocks are kept again
static void destroyed_stream() {
    pp_stream s;
    CHECK(pp_stream_create(&s) == PP_OK);
    CHECK(pp_graph_begin(s) == PP_OK);
    CHECK(pp_graph_begin(s) != PP_OK);      // a second begin is refused and counts once
    CHECK(pp_stream_destroy(s) == PP_OK);
    void* a = get(MIB);
    CHECK(pp_free(a) == PP_OK);
    CHECK(get(MIB) == a && frees == 0);
}

// allocations of the other modules take kept blocks' memory when there is no other
static void other_allocations() {
    budget = 64 * MIB;
    void* p[4];
    for (auto& q : p) q = get(16 * MIB);
    for (auto& q : p) CHECK(pp_free(q) == PP_OK);
    size_t free_bytes = 0, total = 0;
    CHECK(pp_mem_info(&free_bytes, &total) == PP_OK && free_bytes == budget);
    double* d = nullptr;
    CHECK(pp_pool::raw_alloc(&d, 40 * MIB) == hipSuccess && d);
    CHECK(hipGetLastError() == hipSuccess);     // the first attempt left no error behind
    int32_t* big = nullptr;
    CHECK(pp_pool::raw_alloc(&big, 40 * MIB) == hipErrorOutOfMemory && !big);
    CHECK(hipFree(d) == hipSuccess);
}

// at most 1 GiB is kept, the oldest blocks go first, and all of it goes back on request
static void bound_and_release() {
    void* p[8];
    for (auto& q : p) q = get(200 * MIB);
    for (auto& q : p) CHECK(pp_free(q) == PP_OK);
    CHECK(used == 4 * 208 * MIB);       // the size class of 200 MiB is 208 MiB; a fifth would pass 1 GiB
    for (int k = 0; k < 8; ++k) CHECK(blocks.count(p[k]) == (k < 4 ? 0u : 1u));
    CHECK(pp_release_staging() == PP_OK && used == 0);
}

// a kept block is not handed out on another device
static void devices_apart() {
    void* a = get(MIB);
    CHECK(pp_free(a) == PP_OK);
    CHECK(pp_init(1) == PP_OK);
    void* b = get(MIB);
    CHECK(b != a);
    CHECK(pp_init(0) == PP_OK && pp_free(b) == PP_OK && device == 0);
    CHECK(get(MIB) == a);
}

int main(int argc, char** argv) {
    CHECK(argc == 2 && pp_init(0) == PP_OK);
    const std::string w = argv[1];
    if (w == "reuse_waits") reuse_waits();
    else if (w == "double_free") double_free();
    else if (w == "free_and_capture") free_and_capture();
    else if (w == "destroyed_stream") destroyed_stream();
    else if (w == "other_allocations") other_allocations();
    else if (w == "bound_and_release") bound_and_release();
    else if (w == "devices_apart") devices_apart();
    else CHECK(!"unknown case");
    return 0;
}

// Blocking copies (pp_copy.hip) on the host stand-in: see test_native_cpu.py for the cases.
#include <chrono>
#include <stdio.h>
#include <string>

#include "hip_on_host.h"

#include "pp_copy.hip"

using pp_copy::Region;
static const size_t KIB = 1024, MIB = 1024 * KIB;

struct Pair {
    std::vector<char> a, b;
    explicit Pair(size_t n) : a(n), b(n, 0) {
        for (size_t k = 0; k < n; ++k) a[k] = (char)(k * 2654435761u >> 13);
    }
};

static const size_t kSizes[] = {1, 16 * KIB - 1, 16 * KIB, 100 * KIB + 3, MIB - 1, MIB, 4 * MIB + 5, 33 * MIB + 7};

// every byte arrives, both ways, in one and two regions
static void bytes() {
    for (size_t n : kSizes)
        for (int to_host = 0; to_host < 2; ++to_host) {
            Pair p(n), q(n / 3 + 1);
            const Region two[2] = {{to_host ? p.b.data() : p.a.data(), to_host ? p.a.data() : p.b.data(), n},
                                   {to_host ? q.b.data() : q.a.data(), to_host ? q.a.data() : q.b.data(), q.a.size()}};
            CHECK(pp_copy::transfer(two, 2, to_host, 0, nullptr) == hipSuccess);
            CHECK(p.a == p.b && q.a == q.b);
        }
    pp_copy::release();
    CHECK(pinned.empty());
}

// events that are not ready yet leave no error behind for the next launch's check
static void no_error_left() {
    std::atomic<int> asked{0};
    event_ready = [&](hipEvent_t) { return ++asked > 3; };
    for (size_t n : kSizes) {
        Pair p(n);
        asked = 0;
        const Region r = {p.b.data(), p.a.data(), n};
        CHECK(pp_copy::transfer(&r, 1, true, 0, nullptr) == hipSuccess);
        CHECK(p.a == p.b && hipGetLastError() == hipSuccess);
    }
}

// while the stream still computes, one thread waits and none polls
static void one_waiter() {
    std::atomic<bool> done{false};
    std::atomic<int> waiting{0}, most{0};
    event_ready = [&](hipEvent_t) { return done.load(); };
    on_event_sync = [&](hipEvent_t) {
        if (done) return;
        const int w = ++waiting;
        if (w > most) most = w;
        std::this_thread::sleep_for(std::chrono::milliseconds(200));
        const int asked = event_queries;        // by now the destination is populated and the short polls are over
        std::this_thread::sleep_for(std::chrono::milliseconds(300));
        CHECK(event_queries == asked);
        done = true;
        --waiting;
    };
    Pair p(16 * MIB);
    const Region r = {p.b.data(), p.a.data(), p.a.size()};
    CHECK(pp_copy::transfer(&r, 1, true, 0, nullptr) == hipSuccess);
    CHECK(p.a == p.b && most == 1);
}

// the caller's current device stays, and events belong to the stream's device
static void devices_kept() {
    hipStream_t s;
    CHECK(hipStreamCreateWithFlags(&s, 0) == hipSuccess);       // on device 0
    for (size_t n : kSizes)
        for (int to_host = 0; to_host < 2; ++to_host) {
            Pair p(n);
            CHECK(hipSetDevice(1) == hipSuccess);
            const Region r = {to_host ? p.b.data() : p.a.data(), to_host ? p.a.data() : p.b.data(), n};
            CHECK(pp_copy::transfer(&r, 1, to_host, 0, s) == hipSuccess);
            CHECK(p.a == p.b && device == 1);
        }
}

// before the library has chosen a device, copies go to the runtime as they are
static void no_device_yet() {
    for (size_t n : kSizes)
        for (int to_host = 0; to_host < 2; ++to_host) {
            Pair p(n);
            const Region r = {to_host ? p.b.data() : p.a.data(), to_host ? p.a.data() : p.b.data(), n};
            CHECK(pp_copy::transfer(&r, 1, to_host, -1, nullptr) == hipSuccess);
            CHECK(p.a == p.b);
        }
}

// small transfers are one copy a region and one wait for the stream: no events, no threads
static void small_in_one_piece() {
    for (size_t n : {16 * KIB, 100 * KIB + 3, MIB - 5})
        for (int to_host = 0; to_host < 2; ++to_host) {
            Pair p(n - 4), q(4);
            copies = 0;
            const Region two[2] = {{to_host ? q.b.data() : q.a.data(), to_host ? q.a.data() : q.b.data(), 4},
                                   {to_host ? p.b.data() : p.a.data(), to_host ? p.a.data() : p.b.data(), n - 4}};
            CHECK(pp_copy::transfer(two, 2, to_host, 0, nullptr) == hipSuccess);
            CHECK(p.a == p.b && q.a == q.b && copies == 2 && events_made == 0 && event_queries == 0);
        }
}

// a transfer that one thread does faster starts no others
static void threads_by_size() {
    const struct {
        size_t bytes, threads;
    } want[] = {{MIB, 1}, {2 * MIB + 1, 1}, {5 * MIB - 1, 1}, {5 * MIB, 2}, {8 * MIB, 3}, {16 * MIB, 6}, {64 * MIB, 6}};
    for (const auto& w : want) {
        Pair p(w.bytes);
        copiers.clear();
        const Region r = {p.b.data(), p.a.data(), w.bytes};
        CHECK(pp_copy::transfer(&r, 1, true, 0, nullptr) == hipSuccess);
        CHECK(p.a == p.b && copiers.size() == w.threads);
    }
}

int main(int argc, char** argv) {
    CHECK(argc == 2);
    const std::string w = argv[1];
    if (w == "bytes") bytes();
    else if (w == "no_error_left") no_error_left();
    else if (w == "one_waiter") one_waiter();
    else if (w == "devices_kept") devices_kept();
    else if (w == "no_device_yet") no_device_yet();
    else if (w == "small_in_one_piece") small_in_one_piece();
    else if (w == "threads_by_size") threads_by_size();
    else CHECK(!"unknown case");
    return 0;
}

// Large blocking copies between ordinary host memory and the device, pipelined through pinned buffers by several
// threads (host code only).
//
// The runtime moves pageable memory in pieces through one staging buffer and one thread: 6 to 11 GB/s, of which
// most is page faults of a fresh destination (results are new arrays).  Here a few threads share a transfer; each
// owns two pinned slots and every T-th chunk, so DMA, host copies and page faults overlap, and while the stream is
// still computing the threads already fault the destination's pages in; then the caller's thread alone waits for it.
#include <hip/hip_runtime.h>
#include <string.h>
#include <sys/mman.h>
#include <unistd.h>

#include <atomic>
#include <condition_variable>
#include <mutex>
#include <new>
#include <system_error>
#include <thread>
#include <vector>

#include "pp_internal.h"

#ifndef MADV_POPULATE_WRITE
#define MADV_POPULATE_WRITE 23
#endif

namespace pp_copy {
namespace {

// Where the lines lie, runtime / here in us:
//   to the host, fresh array   32 KB 13 / 9   128 KB 30 / 13   512 KB 93 / 37   1 MB 234 / 81   4 MB 970 / 650
//                              8 MB 1940 / 820   16 MB 3890 / 1000   32 MB 7520 / 2020
//   to the host, reused array  32 KB 9 / 9    128 KB 14 / 13   512 KB 29 / 28   1 MB 64 / 63   4 MB 234 / 187
//                              8 MB 478 / 343   16 MB 942 / 610   32 MB 1860 / 980
//   from the host              32 KB 9-21 / 9   128 KB 13-58 / 11   512 KB 23 / 22   1 MB 50 / 100   16 MB 460 / 570
//                              32 MB 1070 / 920   128 MB 4600 / 3400
// (from 1 MB the runtime pins the caller's pages and copies in place, which a fresh destination has to fault first.
// Below it a piece and a wait for the stream are all there is: in two pieces with an event each, made and destroyed,
// 128 KB took 33 us either way and 512 KB 46.)
// Threads, 1 / 2 / 3 / 6 of them, us: reused array 1 MB 63 / 134 / 149 / 264, 4 MB 187 / 218 / 241 / 335, 8 MB 376 / 349 /
// 343 / 427, 16 MB 653 / 552 / 525 / 610; fresh array 1 MB 81 / 166 / 198 / 267, 4 MB 653 / 643 / 611 / 514, 8 MB 1553 /
// 958 / 816 / 720, 16 MB 3324 / 2082 / 1573 / 996.
constexpr size_t kSmallBytes = (size_t)16 << 10;    // below: the runtime's own path
constexpr size_t kManyBytes = (size_t)1 << 20;      // below: one piece a region, no threads
constexpr size_t kUploadBytes = (size_t)32 << 20;   // uploads from kManyBytes to here: the runtime's own path
constexpr size_t kAloneBytes = (size_t)5 << 20;     // below: one thread
constexpr size_t kThreadBytes = (size_t)3 << 20;    // from there another one for each of these
constexpr int kMaxThreads = 6;
constexpr size_t kSlotBytes = (size_t)2 << 20;
constexpr size_t kSetBytes = 2 * kMaxThreads * kSlotBytes;
static_assert(kManyBytes <= kSlotBytes, "one_piece");
constexpr int kMaxSets = 2;     // at most 48 MiB pinned; a third concurrent transfer takes the runtime's own path

std::mutex g_mu;
void* g_sets[kMaxSets] = {};
bool g_busy[kMaxSets] = {};

// A pinned set, or -1: all busy, or no pinned memory to be had.
int acquire() {
    std::lock_guard<std::mutex> lk(g_mu);
    for (int k = 0; k < kMaxSets; ++k) {
        if (g_busy[k]) continue;
        if (!g_sets[k] && hipHostMalloc(&g_sets[k], kSetBytes, hipHostMallocPortable) != hipSuccess) {
            g_sets[k] = nullptr;
            (void)hipGetLastError();
            return -1;
        }
        g_busy[k] = true;
        return k;
    }
    return -1;
}

void give_back(int k) {
    std::lock_guard<std::mutex> lk(g_mu);
    g_busy[k] = false;
}

struct Chunk {
    char* host;
    char* dev;
    size_t bytes;
};

// Whole pages of [p, p + bytes) faulted in for writing (contents unchanged); failure only means later faults.
void populate(char* p, size_t bytes) {
    const uintptr_t page = (uintptr_t)sysconf(_SC_PAGESIZE);
    const uintptr_t a = ((uintptr_t)p + page - 1) & ~(page - 1), b = ((uintptr_t)p + bytes) & ~(page - 1);
    if (b > a) (void)madvise(reinterpret_cast<void*>(a), b - a, MADV_POPULATE_WRITE);
}

struct Job {
    const std::vector<Chunk>& chunks;
    bool to_host;
    int threads, device;
    hipStream_t stream;
    char* pinned;
    hipEvent_t* events;             // 2 per thread
    std::atomic<int> error{0};      // first hipError_t
    std::mutex mu;                  // caller_waits: until the caller's thread has its first chunk, the others sleep
    std::condition_variable awake;
    bool caller_waits = true;

    void wake() {
        {
            std::lock_guard<std::mutex> lk(mu);
            caller_waits = false;
        }
        awake.notify_all();
    }

    void note(hipError_t e) {
        int none = 0;
        if (e != hipSuccess) error.compare_exchange_strong(none, (int)e);
    }

    // false also where the query fails: the wait for the event reports that
    static bool not_ready(hipEvent_t ev) {
        if (hipEventQuery(ev) != hipErrorNotReady) return false;
        (void)hipGetLastError();        // the answer, not an error of this thread's next launch
        return true;
    }

    bool start(int t, size_t c, int slot) {     // DMA of chunk c from or into thread t's slot
        char* pin = pinned + (size_t)(2 * t + slot) * kSlotBytes;
        const Chunk& q = chunks[c];
        hipError_t e = to_host ? hipMemcpyAsync(pin, q.dev, q.bytes, hipMemcpyDeviceToHost, stream)
                               : hipMemcpyAsync(q.dev, pin, q.bytes, hipMemcpyHostToDevice, stream);
        if (e == hipSuccess) e = hipEventRecord(events[2 * t + slot], stream);
        note(e);
        return e == hipSuccess;
    }

    // t = 0: the caller's thread
    void run(int t) {
        copy(t);
        if (t == 0) wake();     // also where it gave up
    }

    void copy(int t) {
        // a thread starts on device 0; the caller's has been set
        if (t != 0 && hipSetDevice(device) != hipSuccess) {
            note(hipErrorInvalidDevice);
            return;
        }
        const size_t n = chunks.size();
        if (to_host) {
            for (int k = 0; k < 2; ++k)
                if ((size_t)(t + k * threads) < n && !start(t, t + k * threads, k)) return;
            size_t filled = t;
            for (size_t c = t, turn = 0; c < n; c += threads, ++turn) {
                const int slot = (int)(turn & 1);
                hipEvent_t ev = events[2 * t + slot];
                int polls = 0;      // of about 0.5 us
                while (error.load() == 0 && not_ready(ev)) {
                    if (filled < n) {
                        populate(chunks[filled].host, chunks[filled].bytes);
                        filled += threads;
                    } else if (++polls < 400) {
                        std::this_thread::yield();
                    } else {
                        break;
                    }
                }
                if (t != 0 && turn == 0) {
                    std::unique_lock<std::mutex> lk(mu);
                    if (polls == 400) awake.wait(lk, [this] { return !caller_waits; });
                }
                if (error.load()) return;
                const hipError_t e = hipEventSynchronize(ev);
                note(e);
                if (t == 0 && turn == 0) wake();
                if (e != hipSuccess) return;
                memcpy(chunks[c].host, pinned + (size_t)(2 * t + slot) * kSlotBytes, chunks[c].bytes);
                if (c + 2 * threads < n && !start(t, c + 2 * threads, slot)) return;
            }
        } else {
            for (size_t c = t, turn = 0; c < n; c += threads, ++turn) {
                const int slot = (int)(turn & 1);
                if (turn >= 2) {
                    const hipError_t e = hipEventSynchronize(events[2 * t + slot]);
                    note(e);
                    if (e != hipSuccess) return;
                }
                memcpy(pinned + (size_t)(2 * t + slot) * kSlotBytes, chunks[c].host, chunks[c].bytes);
                if (error.load() || !start(t, c, slot)) return;
            }
        }
    }
};

hipError_t plain(const Region* r, int n, bool to_host, hipStream_t s) {
    for (int k = 0; k < n; ++k) {
        if (!r[k].bytes) continue;
        const hipError_t e = to_host ? hipMemcpyAsync(r[k].host, r[k].dev, r[k].bytes, hipMemcpyDeviceToHost, s)
                                     : hipMemcpyAsync(r[k].dev, r[k].host, r[k].bytes, hipMemcpyHostToDevice, s);
        if (e != hipSuccess) return e;
    }
    return hipStreamSynchronize(s);
}

// Regions of less than one slot in all: through it as they are.
hipError_t one_piece(const Region* r, int n, bool to_host, char* pin, hipStream_t s) {
    hipError_t e = hipSuccess;
    size_t o = 0;
    for (int k = 0; k < n && e == hipSuccess; o += r[k].bytes, ++k) {
        if (!r[k].bytes) continue;
        if (!to_host) memcpy(pin + o, r[k].host, r[k].bytes);
        e = to_host ? hipMemcpyAsync(pin + o, r[k].dev, r[k].bytes, hipMemcpyDeviceToHost, s)
                    : hipMemcpyAsync(r[k].dev, pin + o, r[k].bytes, hipMemcpyHostToDevice, s);
        if (to_host) populate(static_cast<char*>(r[k].host), r[k].bytes);
    }
    const hipError_t se = hipStreamSynchronize(s);      // also after a failure: the slot serves others next
    if (e == hipSuccess) e = se;
    o = 0;
    for (int k = 0; k < n && to_host && e == hipSuccess; o += r[k].bytes, ++k)
        if (r[k].bytes) memcpy(r[k].host, pin + o, r[k].bytes);
    return e;
}

// The library's device is current while this lives: events belong to the device that is current when they are made,
// and have to belong to the stream's.
struct OnDevice {
    int before = 0;
    hipError_t error;
    explicit OnDevice(int device) : device_(device) {
        error = hipGetDevice(&before);
        if (error == hipSuccess && before != device_) error = hipSetDevice(device_);
    }
    ~OnDevice() {
        if (error == hipSuccess && before != device_) (void)hipSetDevice(before);
    }
    OnDevice(const OnDevice&) = delete;
    OnDevice& operator=(const OnDevice&) = delete;

private:
    int device_;
};

}  // namespace

hipError_t transfer(const Region* r, int n, bool to_host, int device, hipStream_t s) {
    size_t total = 0;
    bool ordinary = true;
    for (int k = 0; k < n; ++k) {
        total += r[k].bytes;
        ordinary = ordinary && (!r[k].bytes || (r[k].host && r[k].dev));
    }
    if (device < 0 || !ordinary || total < kSmallBytes || (!to_host && total >= kManyBytes && total < kUploadBytes))
        return plain(r, n, to_host, s);
    for (int k = 0; k < n; ++k) {       // pinned (or device) memory is copied in place by the runtime
        hipPointerAttribute_t at;
        if (!r[k].bytes) continue;
        if (hipPointerGetAttributes(&at, r[k].host) != hipSuccess) (void)hipGetLastError();
        else if (at.type != hipMemoryTypeUnregistered) return plain(r, n, to_host, s);
    }
    const OnDevice guard(device);
    if (guard.error != hipSuccess) return guard.error;
    const int set = acquire();
    if (set < 0) return plain(r, n, to_host, s);
    if (total < kManyBytes) {
        const hipError_t e = one_piece(r, n, to_host, static_cast<char*>(g_sets[set]), s);
        give_back(set);
        return e;
    }
    const size_t many = total < kAloneBytes ? 1 : 1 + total / kThreadBytes;
    const int threads = many > (size_t)kMaxThreads ? kMaxThreads : (int)many;
    size_t piece = (total / (2 * threads) + 4095) & ~(size_t)4095;
    if (piece > kSlotBytes) piece = kSlotBytes;
    hipEvent_t events[2 * kMaxThreads] = {};
    hipError_t rc = hipSuccess;
    bool started = false;
    try {
        std::vector<Chunk> chunks;
        chunks.reserve(total / piece + n + 1);
        for (int k = 0; k < n; ++k)
            for (size_t o = 0; o < r[k].bytes; o += piece)
                chunks.push_back({static_cast<char*>(r[k].host) + o, static_cast<char*>(r[k].dev) + o,
                                  r[k].bytes - o < piece ? r[k].bytes - o : piece});
        for (int k = 0; k < 2 * threads && rc == hipSuccess; ++k)
            rc = hipEventCreateWithFlags(&events[k], hipEventDisableTiming);
        if (rc == hipSuccess) {
            started = true;
            Job job{chunks, to_host, threads, device, s, static_cast<char*>(g_sets[set]), events};
            std::thread pool[kMaxThreads];
            int up = 1;
            for (; up < threads; ++up) {
                try {
                    pool[up] = std::thread([&job, up] { job.run(up); });
                } catch (const std::exception&) {
                    break;
                }
            }
            job.run(0);
            for (int t = up; t < threads; ++t) job.copy(t);     // shares of threads that could not be started
            for (int t = 1; t < up; ++t) pool[t].join();
            rc = (hipError_t)job.error.load();
        }
    } catch (const std::bad_alloc&) {
        rc = hipErrorOutOfMemory;
    }
    // no copy is in flight once the stream is idle: only then may the set serve another transfer
    const hipError_t se = started ? hipStreamSynchronize(s) : hipSuccess;
    if (rc == hipSuccess) rc = se;
    for (hipEvent_t e : events)
        if (e) (void)hipEventDestroy(e);
    give_back(set);
    return rc;
}

void release() {
    std::lock_guard<std::mutex> lk(g_mu);
    for (int k = 0; k < kMaxSets; ++k)
        if (g_sets[k] && !g_busy[k]) {
            (void)hipHostFree(g_sets[k]);
            g_sets[k] = nullptr;
        }
}

}  // namespace pp_copy

// The HIP runtime calls of the library's host code on ordinary memory, for tests without a device: "device" blocks are
// malloc blocks within a budget, copies are immediate, streams and events are handles whose state the test sets.
#pragma once
#include <hip/hip_runtime.h>
#include <stdlib.h>
#include <string.h>

#include <atomic>
#include <condition_variable>
#include <functional>
#include <map>
#include <mutex>
#include <set>
#include <thread>
#include <vector>

namespace host_hip {
inline std::recursive_mutex mu;
inline std::map<void*, size_t> blocks;          // live device blocks
inline std::map<void*, size_t> pinned;          // live pinned blocks
inline std::vector<size_t> mallocs;             // sizes asked of hipMalloc, in order
inline size_t budget = (size_t)1 << 44, used = 0;
inline std::atomic<int> device_syncs{0}, event_syncs{0}, event_queries{0}, events_made{0}, copies{0}, frees{0}, bad_frees{0};
inline std::set<hipStream_t> capturing;
inline std::set<std::thread::id> copiers;        // threads that enqueued copies
inline std::function<void()> on_device_sync;    // called inside hipDeviceSynchronize
inline std::function<bool(hipEvent_t)> event_ready;     // null: every event is complete
inline std::function<void(hipEvent_t)> on_event_sync;
inline bool sync_during_capture = false;        // hipDeviceSynchronize met a capture
inline thread_local int device = 0;
inline thread_local hipError_t last_error = hipSuccess;
inline int devices = 2;
inline std::map<hipEvent_t, int> event_device;
inline std::map<hipStream_t, int> stream_device;

inline hipError_t give(hipError_t e) {
    if (e != hipSuccess) last_error = e;
    return e;
}
// Blocks of the host's own memory, never touched for large sizes.
inline void* block(size_t bytes) { return malloc(bytes); }
}  // namespace host_hip

extern "C" {
using namespace host_hip;
hipError_t hipMalloc(void** p, size_t bytes) {
    std::lock_guard<std::recursive_mutex> lk(mu);
    mallocs.push_back(bytes);
    *p = nullptr;
    if (used + bytes > budget) return give(hipErrorOutOfMemory);
    *p = block(bytes);
    blocks[*p] = bytes;
    used += bytes;
    return hipSuccess;
}
hipError_t hipFree(void* p) {
    std::lock_guard<std::recursive_mutex> lk(mu);
    if (!p) return hipSuccess;
    auto it = blocks.find(p);
    if (it == blocks.end()) {
        ++bad_frees;
        return give(hipErrorInvalidValue);
    }
    ++frees;
    used -= it->second;
    blocks.erase(it);
    free(p);
    return hipSuccess;
}
hipError_t hipHostMalloc(void** p, size_t bytes, unsigned) {
    std::lock_guard<std::recursive_mutex> lk(mu);
    *p = block(bytes);
    pinned[*p] = bytes;
    return hipSuccess;
}
hipError_t hipHostFree(void* p) {
    std::lock_guard<std::recursive_mutex> lk(mu);
    if (!pinned.erase(p)) return give(hipErrorInvalidValue);
    free(p);
    return hipSuccess;
}
hipError_t hipHostGetDevicePointer(void** d, void* h, unsigned) {
    *d = h;
    return hipSuccess;
}
hipError_t hipMemGetInfo(size_t* f, size_t* t) {
    *f = budget - used;
    *t = budget;
    return hipSuccess;
}
hipError_t hipGetDeviceCount(int* n) {
    *n = devices;
    return hipSuccess;
}
hipError_t hipGetDevice(int* d) {
    *d = device;
    return hipSuccess;
}
hipError_t hipSetDevice(int d) {
    if (d < 0 || d >= devices) return give(hipErrorInvalidDevice);
    device = d;
    return hipSuccess;
}
hipError_t hipDeviceSynchronize() {
    if (on_device_sync) on_device_sync();
    std::lock_guard<std::recursive_mutex> lk(mu);
    ++device_syncs;
    if (!capturing.empty()) {
        sync_during_capture = true;
        return give(hipErrorStreamCaptureUnsupported);
    }
    return hipSuccess;
}
hipError_t hipStreamCreateWithFlags(hipStream_t* s, unsigned) {
    *s = reinterpret_cast<hipStream_t>(malloc(1));
    std::lock_guard<std::recursive_mutex> lk(mu);
    stream_device[*s] = device;
    return hipSuccess;
}
hipError_t hipStreamDestroy(hipStream_t s) {
    std::lock_guard<std::recursive_mutex> lk(mu);
    capturing.erase(s);
    return hipSuccess;
}
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipStreamBeginCapture(hipStream_t s, hipStreamCaptureMode) {
    std::lock_guard<std::recursive_mutex> lk(mu);
    if (!capturing.insert(s).second) return give(hipErrorIllegalState);
    return hipSuccess;
}
hipError_t hipStreamIsCapturing(hipStream_t s, hipStreamCaptureStatus* st) {
    std::lock_guard<std::recursive_mutex> lk(mu);
    *st = capturing.count(s) ? hipStreamCaptureStatusActive : hipStreamCaptureStatusNone;
    return hipSuccess;
}
hipError_t hipStreamEndCapture(hipStream_t s, hipGraph_t* g) {
    std::lock_guard<std::recursive_mutex> lk(mu);
    *g = nullptr;
    return capturing.erase(s) ? hipSuccess : give(hipErrorIllegalState);
}
hipError_t hipGraphInstantiate(hipGraphExec_t* e, hipGraph_t, hipGraphNode_t*, char*, size_t) {
    *e = nullptr;
    return hipSuccess;
}
hipError_t hipGraphDestroy(hipGraph_t) { return hipSuccess; }
hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) {
    ++events_made;
    *e = reinterpret_cast<hipEvent_t>(malloc(1));
    std::lock_guard<std::recursive_mutex> lk(mu);
    event_device[*e] = device;
    return hipSuccess;
}
hipError_t hipEventDestroy(hipEvent_t e) {
    std::lock_guard<std::recursive_mutex> lk(mu);
    event_device.erase(e);
    free(e);
    return hipSuccess;
}
hipError_t hipEventRecord(hipEvent_t e, hipStream_t s) {
    std::lock_guard<std::recursive_mutex> lk(mu);
    auto it = stream_device.find(s);        // an event and its stream belong to one device
    if (it != stream_device.end() && event_device[e] != it->second) return give(hipErrorInvalidHandle);
    return hipSuccess;
}
hipError_t hipEventQuery(hipEvent_t e) {
    ++event_queries;
    return !event_ready || event_ready(e) ? hipSuccess : give(hipErrorNotReady);
}
hipError_t hipEventSynchronize(hipEvent_t e) {
    ++event_syncs;
    if (on_event_sync) on_event_sync(e);
    return hipSuccess;
}
hipError_t hipMemcpyAsync(void* d, const void* s, size_t bytes, hipMemcpyKind, hipStream_t) {
    ++copies;
    {
        std::lock_guard<std::recursive_mutex> lk(mu);
        copiers.insert(std::this_thread::get_id());
    }
    memcpy(d, s, bytes);
    return hipSuccess;
}
hipError_t hipPointerGetAttributes(hipPointerAttribute_t* at, const void* p) {
    std::lock_guard<std::recursive_mutex> lk(mu);
    memset(at, 0, sizeof(*at));
    at->type = hipMemoryTypeUnregistered;
    auto it = pinned.upper_bound(const_cast<void*>(p));
    if (it != pinned.begin() && (--it, (const char*)p < (const char*)it->first + it->second)) at->type = hipMemoryTypeHost;
    return hipSuccess;
}
hipError_t hipGetLastError() {
    const hipError_t e = last_error;
    last_error = hipSuccess;
    return e;
}
const char* hipGetErrorString(hipError_t e) { return e == hipSuccess ? "no error" : "error"; }
}

#define CHECK(c)                                                    \
    do {                                                            \
        if (!(c)) {                                                 \
            fprintf(stderr, "%s:%d: %s\n", __FILE__, __LINE__, #c); \
            exit(1);                                                \
        }                                                           \
    } while (0)

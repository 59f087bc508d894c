// The part of the HIP runtime that loken_amd/csrc/stream_scratch.hip calls, for a build by the host compiler:
// memory is malloc'ed and counted, streams record or not as a test says. Test infrastructure.
#pragma once

#include <stddef.h>
#include <stdlib.h>

#include <map>
#include <mutex>
#include <string>
#include <vector>

enum hipError_t { hipSuccess = 0, hipErrorOutOfMemory = 2, hipErrorInvalidValue = 1, hipErrorStreamCaptureUnsupported = 900 };
enum hipStreamCaptureStatus { hipStreamCaptureStatusNone, hipStreamCaptureStatusActive, hipStreamCaptureStatusInvalidated };
enum hipStreamCaptureMode { hipStreamCaptureModeGlobal, hipStreamCaptureModeThreadLocal, hipStreamCaptureModeRelaxed };

struct ihipStream_t { unsigned long long capture = 0; };   // the id of the capture it records, 0: none
struct ihipEvent_t { ihipStream_t* recorded_on = nullptr; };
typedef ihipStream_t* hipStream_t;
typedef ihipEvent_t* hipEvent_t;
#define hipStreamPerThread ((hipStream_t)2)
#define hipEventDisableTiming 2

namespace fake {
inline std::mutex mu;
inline std::map<void*, std::pair<int, size_t>> live;   // address -> device, bytes
inline int frees = 0, allocations = 0, captures = 0;   // `captures`: recordings under way anywhere, in the global mode
inline bool out_of_memory = false, sync_fails = false, no_events = false;
inline std::vector<std::string> log;                   // waits and records, in order
inline thread_local int device = 0;
inline thread_local hipStreamCaptureMode mode = hipStreamCaptureModeGlobal;
inline bool refused() { return captures > 0 && mode != hipStreamCaptureModeRelaxed; }
inline size_t held() {
    std::lock_guard<std::mutex> lock(mu);
    size_t n = 0;
    for (auto& kv : live) n += kv.second.second;
    return n;
}
}  // namespace fake

inline hipError_t hipGetDevice(int* d) { *d = fake::device; return hipSuccess; }
inline hipError_t hipSetDevice(int d) { fake::device = d; return hipSuccess; }
inline hipError_t hipGetLastError() { return hipSuccess; }
inline hipError_t hipMalloc(void** p, size_t bytes) {
    std::lock_guard<std::mutex> lock(fake::mu);
    if (fake::refused()) return hipErrorStreamCaptureUnsupported;
    if (fake::out_of_memory) return hipErrorOutOfMemory;
    *p = (void*)(((size_t)++fake::allocations) << 40);   // addresses only: nothing is read through them
    fake::live[*p] = {fake::device, bytes};
    return hipSuccess;
}
inline hipError_t hipFree(void* p) {
    std::lock_guard<std::mutex> lock(fake::mu);
    if (fake::refused()) return hipErrorStreamCaptureUnsupported;
    if (!p) return hipSuccess;
    auto it = fake::live.find(p);
    if (it == fake::live.end() || it->second.first != fake::device) abort();   // freed twice, or on another device
    fake::live.erase(it);
    ++fake::frees;
    return hipSuccess;
}
inline hipError_t hipStreamGetCaptureInfo(hipStream_t s, hipStreamCaptureStatus* status, unsigned long long* id) {
    const bool real = s && s != hipStreamPerThread;
    *status = real && s->capture ? hipStreamCaptureStatusActive : hipStreamCaptureStatusNone;
    if (id) *id = real ? s->capture : 0;
    return hipSuccess;
}
inline hipError_t hipThreadExchangeStreamCaptureMode(hipStreamCaptureMode* m) {
    std::swap(*m, fake::mode);
    return hipSuccess;
}
inline void note(const char* what, const void* stream) {
    std::lock_guard<std::mutex> lock(fake::mu);
    fake::log.push_back(std::string(what) + " " + std::to_string((size_t)stream));
}
inline hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) {
    if (fake::no_events) return hipErrorOutOfMemory;
    *e = new ihipEvent_t;
    return hipSuccess;
}
inline hipError_t hipEventDestroy(hipEvent_t e) { delete e; return hipSuccess; }
inline hipError_t hipEventRecord(hipEvent_t e, hipStream_t s) { e->recorded_on = s; note("record", s); return hipSuccess; }
inline hipError_t hipStreamWaitEvent(hipStream_t s, hipEvent_t e, unsigned) {
    if (!e->recorded_on) abort();
    note("wait", s);
    return hipSuccess;
}
inline hipError_t hipStreamSynchronize(hipStream_t s) { note("synchronize", s); return hipSuccess; }
inline hipError_t hipDeviceSynchronize() { return fake::sync_fails || fake::refused() ? hipErrorStreamCaptureUnsupported : hipSuccess; }

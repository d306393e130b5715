/* A stand-in for the few runtime calls of mpcd_transfer.h, on the CPU: a copy
 * is done only when its stream or an event behind it is waited for, as late
 * as the real one may be, so a chunk used again too early shows as wrong
 * bytes. */
#pragma once

#include <cstddef>
#include <cstdlib>
#include <cstring>
#include <deque>
#include <functional>
#include <mutex>

enum hipError_t { hipSuccess = 0, hipErrorInvalidValue = 1 };
enum hipMemcpyKind { hipMemcpyHostToDevice = 1, hipMemcpyDeviceToHost = 2 };
enum hipMemoryType { hipMemoryTypeUnregistered = 0, hipMemoryTypeHost = 1, hipMemoryTypeDevice = 2 };
enum { hipHostMallocPortable = 1, hipEventDisableTiming = 2 };

struct FakeStream {
    std::mutex mu;
    std::deque<std::function<void()>> todo;
    long long done = 0, queued = 0;
    void run_to(long long k) {
        std::lock_guard<std::mutex> lk(mu);
        for (; done < k; ++done) {
            todo.front()();
            todo.pop_front();
        }
    }
};
struct FakeEvent {
    FakeStream* st = nullptr;
    long long at = 0;
};
typedef FakeStream* hipStream_t;
typedef FakeEvent* hipEvent_t;
struct hipPointerAttribute_t {
    hipMemoryType type;
};

/* the arrays the test calls registered, and whether an unregistered one is an
 * error (as it was in older runtimes) */
struct FakeRegistered {
    const char* lo = nullptr;
    const char* hi = nullptr;
    hipMemoryType type = hipMemoryTypeHost;
    bool strict = false;
};
inline FakeRegistered& fake_registered() {
    static FakeRegistered r;
    return r;
}

inline const char* hipGetErrorString(hipError_t) { return "fake error"; }
inline hipError_t hipGetLastError() { return hipSuccess; }
inline hipError_t hipGetDevice(int* d) { return *d = 0, hipSuccess; }
inline hipError_t hipSetDevice(int) { return hipSuccess; }
template <class T>
hipError_t hipMalloc(T** p, size_t n) {
    return *p = (T*)std::malloc(n), hipSuccess;
}
inline hipError_t hipFree(void* p) { return std::free(p), hipSuccess; }
template <class T>
hipError_t hipHostMalloc(T** p, size_t n, unsigned) {
    return *p = (T*)std::malloc(n), hipSuccess;
}
inline hipError_t hipHostFree(void* p) { return std::free(p), hipSuccess; }
inline hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) { return *e = new FakeEvent, hipSuccess; }
inline hipError_t hipEventDestroy(hipEvent_t e) { return delete e, hipSuccess; }
inline hipError_t hipEventRecord(hipEvent_t e, hipStream_t s) {
    std::lock_guard<std::mutex> lk(s->mu);
    e->st = s;
    e->at = s->queued;
    return hipSuccess;
}
inline hipError_t hipEventSynchronize(hipEvent_t e) {
    if (e->st) e->st->run_to(e->at);
    return hipSuccess;
}
inline hipError_t hipStreamSynchronize(hipStream_t s) {
    long long k;
    {
        std::lock_guard<std::mutex> lk(s->mu);
        k = s->queued;
    }
    s->run_to(k);
    return hipSuccess;
}
inline hipError_t hipMemcpyAsync(void* d, const void* s, size_t n, hipMemcpyKind, hipStream_t st) {
    std::lock_guard<std::mutex> lk(st->mu);
    st->todo.push_back([=] { std::memcpy(d, s, n); });
    ++st->queued;
    return hipSuccess;
}
inline hipError_t hipPointerGetAttributes(hipPointerAttribute_t* a, const void* p) {
    const FakeRegistered& r = fake_registered();
    const bool in = (const char*)p >= r.lo && (const char*)p < r.hi;
    if (!in && r.strict) return hipErrorInvalidValue;
    a->type = in ? r.type : hipMemoryTypeUnregistered;
    return hipSuccess;
}

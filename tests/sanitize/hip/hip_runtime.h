// A host-only stand-in for the few HIP calls of hostcopy.h: one in-order queue whose copies run
// as late as they may, when an event or the stream is waited for.
#pragma once

#include <cstddef>
#include <cstdlib>
#include <cstring>
#include <deque>
#include <functional>
#include <mutex>

using hipError_t = int;
constexpr hipError_t hipSuccess = 0;
enum hipMemcpyKind { hipMemcpyHostToDevice, hipMemcpyDeviceToHost };
constexpr unsigned hipEventDisableTiming = 2, hipHostMallocDefault = 0;

struct FakeStream {
    static FakeStream*& last() {
        static FakeStream* s = nullptr;
        return s;
    }
    FakeStream() { last() = this; }
    std::mutex mu;
    std::deque<std::function<void()>> queue;
    long done = 0, put = 0;
    int fail_after = -1;  // copies that succeed before one is refused (-1: all)
    void run_to(long upto) {
        while (done < upto) {
            queue.front()();
            queue.pop_front();
            ++done;
        }
    }
};
struct FakeEvent {
    FakeStream* st = nullptr;
    long at = 0;
};
using hipStream_t = FakeStream*;
using hipEvent_t = FakeEvent*;

inline const char* hipGetErrorString(hipError_t) { return "refused"; }
inline hipError_t hipMemcpyAsync(void* d, const void* s, size_t n, hipMemcpyKind, hipStream_t st) {
    std::lock_guard<std::mutex> g(st->mu);
    if (st->fail_after == 0) return 1;
    if (st->fail_after > 0) --st->fail_after;
    st->queue.push_back([=] { std::memcpy(d, s, n); });
    ++st->put;
    return hipSuccess;
}
inline hipError_t hipStreamSynchronize(hipStream_t st) {
    std::lock_guard<std::mutex> g(st->mu);
    st->run_to(st->put);
    return hipSuccess;
}
inline hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) {
    *e = new FakeEvent();
    return hipSuccess;
}
inline hipError_t hipEventDestroy(hipEvent_t e) {
    delete e;
    return hipSuccess;
}
inline hipError_t hipEventRecord(hipEvent_t e, hipStream_t st) {
    std::lock_guard<std::mutex> g(st->mu);
    e->st = st;
    e->at = st->put;
    return hipSuccess;
}
inline hipError_t hipEventSynchronize(hipEvent_t e) {
    if (!e->st) return hipSuccess;
    std::lock_guard<std::mutex> g(e->st->mu);
    e->st->run_to(e->at);
    return hipSuccess;
}
inline hipError_t hipHostMalloc(void** p, size_t n, unsigned) {
    *p = std::malloc(n);
    return *p ? hipSuccess : 2;
}
inline hipError_t hipHostFree(void* p) {
    (void)hipStreamSynchronize(FakeStream::last());  // the real one waits for the device
    std::free(p);
    return hipSuccess;
}
inline hipError_t hipGetDevice(int* d) {
    *d = 0;
    return hipSuccess;
}
inline hipError_t hipSetDevice(int) { return hipSuccess; }

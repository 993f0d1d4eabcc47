// The HIP calls that csrc/copy_back.hpp makes, over host memory: a stream is
// a queue of copies, which run when an event behind them is asked for.
#pragma once
#include <atomic>
#include <cstddef>
#include <cstdlib>
#include <cstring>
#include <deque>
#include <functional>

enum hipError_t { hipSuccess = 0, hipErrorOutOfMemory = 2, hipErrorNotReady = 600, hipErrorUnknown = 999 };
enum { hipMemcpyDeviceToHost = 2, hipEventDisableTiming = 2 };

struct FakeStream {
    std::deque<std::function<void()>> ops;
    long long queued = 0, done = 0;
    static std::atomic<long long> &copies() {
        static std::atomic<long long> n{0};
        return n;
    }
    void run_to(long long n) {
        while (done < n) {
            ops.front()();
            ops.pop_front();
            ++done;
            ++copies();
        }
    }
};
struct FakeEvent {
    FakeStream *st = nullptr;
    long long at = 0;
};
typedef FakeStream *hipStream_t;
typedef FakeEvent *hipEvent_t;

struct FakeHip {
    int mallocs = 0, events = 0;
    int fail_malloc = 0, fail_event_from = -1;
    long long fail_copy = -1;  // the event behind that many copies fails
};
inline FakeHip &fake() {
    static FakeHip f;
    return f;
}
inline const char *hipGetErrorString(hipError_t) { return "fake error"; }
inline hipError_t hipGetLastError() { return hipSuccess; }
inline hipError_t hipHostMalloc(void **p, size_t n) {
    ++fake().mallocs;
    if (fake().fail_malloc) return hipErrorOutOfMemory;
    *p = std::malloc(n);
    return hipSuccess;
}
inline hipError_t hipHostFree(void *p) {
    std::free(p);
    return hipSuccess;
}
inline hipError_t hipEventCreateWithFlags(hipEvent_t *e, unsigned) {
    if (fake().fail_event_from >= 0 && fake().events >= fake().fail_event_from) return hipErrorOutOfMemory;
    ++fake().events;
    *e = new FakeEvent;
    return hipSuccess;
}
inline hipError_t hipEventDestroy(hipEvent_t e) {
    delete e;
    return hipSuccess;
}
inline hipError_t hipMemcpyAsync(void *d, const void *s, size_t n, int, hipStream_t st) {
    st->ops.push_back([=] { std::memcpy(d, s, n); });
    ++st->queued;
    return hipSuccess;
}
inline hipError_t hipEventRecord(hipEvent_t e, hipStream_t st) {
    e->st = st;
    e->at = st->queued;
    return hipSuccess;
}
inline hipError_t hipEventQuery(hipEvent_t e) {
    static int n = 0;
    if (++n % 3 == 0 && e->st->done < e->at) e->st->run_to(e->st->done + 1);  // the device goes on by itself
    if (e->st->done < e->at) return hipErrorNotReady;
    return e->at == fake().fail_copy ? hipErrorUnknown : hipSuccess;
}
inline hipError_t hipEventSynchronize(hipEvent_t e) {
    e->st->run_to(e->at);
    return e->at == fake().fail_copy ? hipErrorUnknown : hipSuccess;
}
inline hipError_t hipStreamSynchronize(hipStream_t st) {
    st->run_to(st->queued);
    return hipSuccess;
}

// Streams, events and copies of the HIP runtime on the host, as far as
// rbhip_readback.h uses them.  A stream is a queue whose entries run in order;
// a copy into an idle stream runs at once, everything else when somebody waits
// for it (so work that is not waited for is late).  hipStreamPerThread names
// the calling thread's own stream.
#pragma once
#include <chrono>
#include <cstdlib>
#include <cstring>
#include <deque>
#include <functional>
#include <map>
#include <mutex>
#include <thread>

struct FakeStream {
    std::deque<std::function<void()>> queue;
    long queued = 0, done = 0;
};
struct FakeEvent {
    FakeStream* stream = nullptr;
    long at = 0;
};
typedef FakeStream* hipStream_t;
typedef FakeEvent* hipEvent_t;
enum hipError_t { hipSuccess = 0, hipErrorOutOfMemory = 2 };
enum hipMemcpyKind { hipMemcpyDeviceToHost = 2 };
#define hipStreamPerThread reinterpret_cast<hipStream_t>(2)
constexpr unsigned hipEventDisableTiming = 2, hipHostMallocPortable = 1;

inline std::recursive_mutex& fake_lock() {
    static std::recursive_mutex m;
    return m;
}
inline FakeStream* fake_stream(hipStream_t s) {
    static std::map<std::thread::id, FakeStream> own;
    return s == hipStreamPerThread ? &own[std::this_thread::get_id()] : s;
}
inline void fake_run(FakeStream* s, long to) {
    while (s->done < to) {
        std::function<void()> f = std::move(s->queue.front());
        s->queue.pop_front();
        f();
        s->done++;
    }
}
inline void fake_queue(hipStream_t h, std::function<void()> f) {
    std::lock_guard<std::recursive_mutex> lock(fake_lock());
    FakeStream* s = fake_stream(h);
    s->queue.push_back(std::move(f));
    s->queued++;
}
inline hipError_t hipGetLastError() { return hipSuccess; }
inline hipError_t hipSetDevice(int) { return hipSuccess; }
inline hipError_t hipHostMalloc(void** p, size_t n, unsigned) {
    *p = std::malloc(n);
    return *p ? hipSuccess : hipErrorOutOfMemory;
}
inline hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) {
    *e = new FakeEvent;
    return hipSuccess;
}
inline hipError_t hipEventDestroy(hipEvent_t e) {
    delete e;
    return hipSuccess;
}
inline hipError_t hipEventRecord(hipEvent_t e, hipStream_t h) {
    std::lock_guard<std::recursive_mutex> lock(fake_lock());
    e->stream = fake_stream(h);
    e->at = e->stream->queued;
    return hipSuccess;
}
inline hipError_t hipStreamWaitEvent(hipStream_t h, hipEvent_t e, unsigned) {
    FakeStream* on = e->stream;
    const long at = e->at;
    fake_queue(h, [on, at] { if (on) fake_run(on, at); });
    return hipSuccess;
}
inline hipError_t hipMemcpyAsync(void* to, const void* from, size_t n, hipMemcpyKind, hipStream_t h) {
    std::lock_guard<std::recursive_mutex> lock(fake_lock());
    fake_queue(h, [=] { std::memcpy(to, from, n); });
    FakeStream* s = fake_stream(h);
    if (s->queued == s->done + 1) fake_run(s, s->queued);
    return hipSuccess;
}
// (the work that is waited for ends a while after the wait began)
inline void fake_wait(FakeStream* s, long to) {
    std::this_thread::sleep_for(std::chrono::milliseconds(s->done < to ? 50 : 0));
    std::lock_guard<std::recursive_mutex> lock(fake_lock());
    fake_run(s, to);
}
inline hipError_t hipEventSynchronize(hipEvent_t e) {
    fake_wait(e->stream, e->at);
    return hipSuccess;
}
inline hipError_t hipStreamSynchronize(hipStream_t h) {
    FakeStream* s;
    {
        std::lock_guard<std::recursive_mutex> lock(fake_lock());
        s = fake_stream(h);
    }
    fake_wait(s, s->queued);
    return hipSuccess;
}

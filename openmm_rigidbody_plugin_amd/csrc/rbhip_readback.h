// Device memory to the caller's (pageable) host memory, through pinned chunks.
//
// A direct copy into pageable memory runs at 10-17 GB/s here: one thread
// copies out of the runtime's staging buffer and takes the page faults of
// fresh memory.  Device copies into pinned memory reach 56 GB/s, so a large
// read-back is split into chunks that several threads empty into the caller's
// memory, each with two chunks in flight on the owner's stream.
#pragma once

#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstring>
#include <mutex>
#include <thread>
#include <vector>

namespace rbhip {

// Pinned chunks shared by every context of the process: at most kMaxChunks
// (64 MiB), allocated when first needed, taken for one call and put back at
// its end, kept until the process ends.  A caller that finds none left copies
// directly.
class PinnedChunks {
public:
    static constexpr size_t kBytes = size_t(2) << 20;
    static constexpr int kMaxChunks = 32;
    static PinnedChunks& get() {
        static PinnedChunks* p = new PinnedChunks;   // (never destroyed: the runtime may be gone by then)
        return *p;
    }
    // up to `want` chunks
    std::vector<void*> take(int want) {
        std::lock_guard<std::mutex> lock(mtx_);
        std::vector<void*> out;
        while ((int)out.size() < want) {
            if (idle_.empty()) {
                void* p = nullptr;
                if (made_ == kMaxChunks || hipHostMalloc(&p, kBytes, hipHostMallocPortable) != hipSuccess) {
                    (void)hipGetLastError();
                    break;
                }
                made_++;
                idle_.push_back(p);
            }
            out.push_back(idle_.back());
            idle_.pop_back();
        }
        return out;
    }
    void put(const std::vector<void*>& chunks) {
        std::lock_guard<std::mutex> lock(mtx_);
        idle_.insert(idle_.end(), chunks.begin(), chunks.end());
    }

private:
    std::mutex mtx_;
    std::vector<void*> idle_;
    int made_ = 0;
};

// chunks held for the length of a scope; work that writes them is waited for
// (wait, or on the way out of a scope left early) before they are put back
struct PinnedLease {
    std::vector<void*> chunks;
    hipStream_t pending;   // work queued here may still write the chunks
    explicit PinnedLease(int want, hipStream_t writer = nullptr)
        : chunks(PinnedChunks::get().take(want)), pending(writer) {}
    ~PinnedLease() {
        if (pending) (void)hipStreamSynchronize(pending);
        PinnedChunks::get().put(chunks);
    }
    hipError_t wait() {
        hipStream_t s = pending;
        pending = nullptr;
        return hipStreamSynchronize(s);
    }
    PinnedLease(const PinnedLease&) = delete;
    PinnedLease& operator=(const PinnedLease&) = delete;
};

// copies `bytes` at device address src to dst after the work queued on
// `stream`, and waits for it.  Threads: one per 2 chunks, at most 4 (1M
// waters' positions, 72 MB into fresh memory: 6.9 ms direct, 2.6 with 3
// threads, 2.1-2.2 with 4, 6, 8 or 12; chunks of 1 MiB: 2.6).  One chunk needs
// no other thread (0.3 to 2 MB: 22 to 115 us, as a direct copy's).  The other
// threads' copies wait for an event that the caller records: a handle such as
// hipStreamPerThread names another stream in each of them.
inline hipError_t read_back(void* dst, const void* src, size_t bytes, int device, hipStream_t stream) {
    constexpr size_t chunk = PinnedChunks::kBytes;
    const size_t count = (bytes + chunk - 1) / chunk;
    const int want = (int)std::min<size_t>(4, (count + 1) / 2);
    PinnedLease lease(count == 1 ? 1 : 2 * want);
    char* to = static_cast<char*>(dst);
    const char* from = static_cast<const char*>(src);
    if (count <= 1 || lease.chunks.size() < 2) {
        const bool pinned = count <= 1 && !lease.chunks.empty();
        hipError_t e = hipMemcpyAsync(pinned ? lease.chunks[0] : dst, src, bytes, hipMemcpyDeviceToHost, stream);
        if (e == hipSuccess) e = hipStreamSynchronize(stream);
        if (e == hipSuccess && pinned) std::memcpy(dst, lease.chunks[0], bytes);
        return e;
    }
    // thread t empties chunks t, t + threads, ... through its two buffers
    const int threads = (int)lease.chunks.size() / 2;
    std::vector<hipError_t> status(threads, hipSuccess);
    struct Event {
        hipEvent_t ev = nullptr;
        ~Event() {
            if (ev) (void)hipEventDestroy(ev);
        }
    } ready;   // what was queued on the caller's stream
    hipError_t r = hipEventCreateWithFlags(&ready.ev, hipEventDisableTiming);
    if (r == hipSuccess) r = hipEventRecord(ready.ev, stream);
    if (r != hipSuccess) return r;
    auto worker = [&](int t) {
        hipError_t& e = status[t];
        e = hipSetDevice(device);
        if (e == hipSuccess) e = hipStreamWaitEvent(stream, ready.ev, 0);
        hipEvent_t done[2] = {nullptr, nullptr};
        for (int b = 0; b < 2 && e == hipSuccess; b++) e = hipEventCreateWithFlags(&done[b], hipEventDisableTiming);
        auto issue = [&](size_t c, int b) {
            e = hipMemcpyAsync(lease.chunks[2 * t + b], from + c * chunk, std::min(chunk, bytes - c * chunk),
                               hipMemcpyDeviceToHost, stream);
            if (e == hipSuccess) e = hipEventRecord(done[b], stream);
        };
        bool queued = false;
        for (int b = 0; b < 2 && e == hipSuccess; b++)
            if ((size_t)t + (size_t)b * threads < count) {
                issue((size_t)t + (size_t)b * threads, b);
                queued = true;
            }
        int b = 0;
        for (size_t c = t; c < count && e == hipSuccess; c += threads, b ^= 1) {
            e = hipEventSynchronize(done[b]);
            if (e != hipSuccess) break;
            std::memcpy(to + c * chunk, lease.chunks[2 * t + b], std::min(chunk, bytes - c * chunk));
            if (c + 2 * (size_t)threads < count) issue(c + 2 * (size_t)threads, b);
        }
        // (no copy into a chunk may be in flight when it is put back)
        if (e != hipSuccess && queued) (void)hipStreamSynchronize(stream);
        for (hipEvent_t ev : done)
            if (ev) (void)hipEventDestroy(ev);
    };
    std::vector<std::thread> team;
    int started = 1;
    try {
        for (; started < threads; started++) team.emplace_back(worker, started);
    } catch (...) {
        // no more threads: this one takes the rest's chunks in turn
    }
    worker(0);
    for (int t = started; t < threads; t++) worker(t);
    for (std::thread& th : team) th.join();
    for (hipError_t e : status)
        if (e != hipSuccess) return e;
    return hipSuccess;
}

}  // namespace rbhip

// host_copy.h -- copies between pageable host memory and the device.
//
// A copy from or to pageable memory runs at the speed of one thread that
// touches (and, for fresh memory, faults in) the caller's pages.  These copies
// go through a pinned ring in chunks: the DMA of one chunk runs beside the
// memcpy of others on a few worker threads.
// Measured, us: 33 MB of a 1080p accumulator into fresh memory 2250 -> 900, 15
// MB 1030 -> 454, 1.2 MB 111 -> 76; 24 MB of a scene up 1599 -> 998.  Copies up
// of at most 4 MB stay with the runtime's own staging: waking a worker costs
// more than it saves (1.6 MB of rays and 0.8 MB of hits 146 us with it, 232
// with quarter chunks on the workers).  Memory that the caller has pinned is
// copied by one DMA without the ring.
#pragma once

#include <hip/hip_runtime.h>

#include <condition_variable>
#include <cstddef>
#include <mutex>
#include <thread>

namespace prt {

// Counts down to zero; one thread waits for that.
class Latch {
public:
    void reset(int n) { left_ = n; }  // only while nobody waits or counts
    void done();
    void wait();

private:
    std::mutex mu_;
    std::condition_variable cv_;
    int left_ = 0;
};

// A few threads for memcpy-like jobs, started by the first of them; they never
// call HIP.
// Nothing here allocates per job or throws.
class Workers {
public:
    ~Workers();
    // Runs fn(arg) on a worker (here, if there is none).
    void start(void (*fn)(void*), void* arg);
    // fn(arg, 0) .. fn(arg, n - 1), this thread helping; returns when all are done.
    void each(int n, void (*fn)(void*, int), void* arg);

private:
    static constexpr int kThreads = 4;
    static constexpr int kJobs = 64;
    struct Job {
        void (*fn)(void*);
        void* arg;
    };
    void open();
    void run();
    std::mutex mu_;
    std::condition_variable wake_;
    Job jobs_[kJobs];
    int head_ = 0, count_ = 0;
    std::thread threads_[kThreads];
    int nthreads_ = 0;
    bool started_ = false, quit_ = false;
};

class HostCopy {
public:
    ~HostCopy();
    // Lays out the ring; false: the system gives no pinned memory, and copies go
    // through the runtime's own staging.  The first copy does it if nobody has.
    bool prepare();
    // Both wait until the copy is done.  Work already on the stream comes first.
    hipError_t to_host(void* dst, const void* src, size_t bytes, hipStream_t s);
    hipError_t to_device(void* dst, const void* src, size_t bytes, hipStream_t s);
    Workers& workers() { return workers_; }
    // The ring, kRingBytes of pinned memory, once prepare has laid it out.  Between
    // two copies it is the caller's.
    void* ring() { return ring_; }
    static constexpr int kSlots = 6;
    static constexpr size_t kChunk = size_t(2) << 20;
    static constexpr size_t kRingBytes = kSlots * kChunk;

private:
    static constexpr size_t kAskBytes = size_t(64) << 10;  // a smaller copy gains less than the question costs
    struct Slot {
        void* to;
        const void* from;
        size_t bytes;
        Latch copied;
    };
    static hipError_t plain(void* dst, const void* src, size_t bytes, hipMemcpyKind kind, hipStream_t s);
    void hand(int slot, void* to, const void* from, size_t bytes);
    Workers workers_;
    Slot slots_[kSlots];
    char* ring_ = nullptr;          // kRingBytes, pinned
    hipEvent_t ev_[kSlots] = {};    // last DMA of each slot
    bool refused_ = false;          // no ring: the system gave no pinned memory
};

}  // namespace prt

// host_copy.hip -- see host_copy.h.
#include "host_copy.h"

#include <algorithm>
#include <atomic>
#include <cstring>

namespace prt {

void Latch::done()
{
    std::lock_guard<std::mutex> lock(mu_);
    if (--left_ == 0) cv_.notify_all();
}

void Latch::wait()
{
    std::unique_lock<std::mutex> lock(mu_);
    cv_.wait(lock, [this] { return left_ <= 0; });
}

Workers::~Workers()
{
    {
        std::lock_guard<std::mutex> lock(mu_);
        quit_ = true;
    }
    wake_.notify_all();
    for (int i = 0; i < nthreads_; ++i) threads_[i].join();
}

void Workers::run()
{
    std::unique_lock<std::mutex> lock(mu_);
    for (;;) {
        wake_.wait(lock, [this] { return quit_ || count_ > 0; });
        if (count_ == 0) return;  // quit
        const Job job = jobs_[head_];
        head_ = (head_ + 1) % kJobs;
        --count_;
        lock.unlock();
        job.fn(job.arg);
        lock.lock();
    }
}

void Workers::open()
{
    if (started_) return;
    started_ = true;
    try {
        for (; nthreads_ < kThreads; ++nthreads_) threads_[nthreads_] = std::thread([this] { run(); });
    } catch (...) {
        // as many threads as the system gives
    }
}

void Workers::start(void (*fn)(void*), void* arg)
{
    open();
    {
        std::unique_lock<std::mutex> lock(mu_);
        if (nthreads_ > 0 && count_ < kJobs) {
            jobs_[(head_ + count_) % kJobs] = Job{fn, arg};
            ++count_;
            lock.unlock();
            wake_.notify_one();
            return;
        }
    }
    fn(arg);
}

void Workers::each(int n, void (*fn)(void*, int), void* arg)
{
    struct Shared {
        std::atomic<int> next{0};
        int n;
        void (*fn)(void*, int);
        void* arg;
        Latch latch;
        void take()
        {
            for (int i; (i = next.fetch_add(1)) < n;) fn(arg, i);
        }
    } shared;
    shared.n = n;
    shared.fn = fn;
    shared.arg = arg;
    const int helpers = std::max(0, std::min(n - 1, kThreads));
    shared.latch.reset(helpers);
    for (int i = 0; i < helpers; ++i)
        start(
            [](void* p) {
                Shared* s = static_cast<Shared*>(p);
                s->take();
                s->latch.done();
            },
            &shared);
    shared.take();
    if (helpers) shared.latch.wait();
}

HostCopy::~HostCopy()
{
    for (hipEvent_t e : ev_)
        if (e) (void)hipEventDestroy(e);
    if (ring_) (void)hipHostFree(ring_);
}

bool HostCopy::prepare()
{
    if (refused_) return false;
    if (!ring_ &&
        hipHostMalloc(reinterpret_cast<void**>(&ring_), kRingBytes, hipHostMallocDefault) != hipSuccess) {
        ring_ = nullptr;
        refused_ = true;
    }
    for (hipEvent_t& v : ev_)
        if (!refused_ && !v && hipEventCreateWithFlags(&v, hipEventDisableTiming) != hipSuccess) {
            v = nullptr;
            refused_ = true;
        }
    if (refused_) (void)hipGetLastError();
    return !refused_;
}

// One copy by the runtime, which stages pageable memory itself.
hipError_t HostCopy::plain(void* dst, const void* src, size_t bytes, hipMemcpyKind kind, hipStream_t s)
{
    const hipError_t e = hipMemcpyAsync(dst, src, bytes, kind, s);
    const hipError_t w = hipStreamSynchronize(s);
    return e == hipSuccess ? w : e;
}

// Starts the memcpy of a slot; its latch tells when it is done.
void HostCopy::hand(int slot, void* to, const void* from, size_t bytes)
{
    Slot& s = slots_[slot];
    s.to = to;
    s.from = from;
    s.bytes = bytes;
    s.copied.reset(1);
    workers_.start(
        [](void* p) {
            Slot* w = static_cast<Slot*>(p);
            std::memcpy(w->to, w->from, w->bytes);
            w->copied.done();
        },
        &s);
}

// The caller's memory is pinned (or the device's): the DMA engine takes it
// where it is.  Asked for copies of at least kAskBytes only.
static bool takes_dma(const void* p)
{
    hipPointerAttribute_t a{};
    if (hipPointerGetAttributes(&a, p) != hipSuccess) {
        (void)hipGetLastError();  // memory that HIP does not know is an error to it
        return false;
    }
    return a.type != hipMemoryTypeUnregistered;
}

hipError_t HostCopy::to_host(void* dst, const void* src, size_t bytes, hipStream_t s)
{
    if (bytes == 0) return hipStreamSynchronize(s);
    if ((bytes >= kAskBytes && takes_dma(dst)) || !prepare()) return plain(dst, src, bytes, hipMemcpyDeviceToHost, s);
    hipError_t e = hipSuccess;
    char* out = static_cast<char*>(dst);
    const char* in = static_cast<const char*>(src);
    if (bytes <= kChunk) {
        // waking a worker takes longer than this thread's memcpy of one chunk;
        // the second half's DMA runs beside the first half's memcpy
        const size_t half = bytes <= kChunk / 4 ? bytes : (bytes / 2 + 4095) & ~(size_t)4095;
        e = hipMemcpyAsync(ring_, in, half, hipMemcpyDeviceToHost, s);
        if (e == hipSuccess && half < bytes) {
            e = hipEventRecord(ev_[0], s);
            if (e == hipSuccess) e = hipMemcpyAsync(ring_ + half, in + half, bytes - half, hipMemcpyDeviceToHost, s);
            if (e == hipSuccess) e = hipEventSynchronize(ev_[0]);
            if (e == hipSuccess) std::memcpy(out, ring_, half);
        }
        const hipError_t w = hipStreamSynchronize(s);
        if (e == hipSuccess) e = w;
        if (e == hipSuccess) {
            const size_t at = half < bytes ? half : 0;
            std::memcpy(out + at, ring_ + at, bytes - at);
        }
        return e;
    }
    // chunk c goes by DMA into slot c mod kSlots, then a worker copies it out.
    // A slot's next DMA is issued a few chunks after its memcpy was handed
    // out, so this thread hardly waits for one.
    const int chunks = (int)((bytes + kChunk - 1) / kChunk);
    auto length = [&](int c) { return std::min(kChunk, bytes - (size_t)c * kChunk); };
    constexpr int kBehind = kSlots / 2;
    int issued = 0, handed = 0;
    for (int c = 0; c < chunks && e == hipSuccess; ++c) {
        while (issued < chunks && issued < std::max(kSlots, c + kSlots - kBehind) && e == hipSuccess) {
            const int slot = issued % kSlots;
            if (issued >= kSlots) slots_[slot].copied.wait();
            e = hipMemcpyAsync(ring_ + (size_t)slot * kChunk, in + (size_t)issued * kChunk, length(issued),
                               hipMemcpyDeviceToHost, s);
            if (e == hipSuccess) e = hipEventRecord(ev_[slot], s);
            ++issued;
        }
        if (e == hipSuccess) e = hipEventSynchronize(ev_[c % kSlots]);
        if (e != hipSuccess) break;
        hand(c % kSlots, out + (size_t)c * kChunk, ring_ + (size_t)(c % kSlots) * kChunk, length(c));
        handed = c + 1;
    }
    for (int c = std::max(0, handed - kSlots); c < handed; ++c) slots_[c % kSlots].copied.wait();
    if (e != hipSuccess) (void)hipStreamSynchronize(s);  // no DMA may still write the ring
    return e;
}

hipError_t HostCopy::to_device(void* dst, const void* src, size_t bytes, hipStream_t s)
{
    if (bytes == 0) return hipSuccess;
    // too little to gain from a second thread: the runtime's own staging
    if (bytes <= 2 * kChunk || takes_dma(src) || !prepare()) return plain(dst, src, bytes, hipMemcpyHostToDevice, s);
    hipError_t e = hipSuccess;
    char* out = static_cast<char*>(dst);
    const char* in = static_cast<const char*>(src);
    // chunk c: a worker fills slot c mod kSlots, then the DMA; the slot is
    // filled again once that DMA, issued a few chunks ago, is done
    const int chunks = (int)((bytes + kChunk - 1) / kChunk);
    auto length = [&](int c) { return std::min(kChunk, bytes - (size_t)c * kChunk); };
    constexpr int kBehind = kSlots / 2;
    int handed = 0;
    auto fill = [&]() {
        hand(handed % kSlots, ring_ + (size_t)(handed % kSlots) * kChunk, in + (size_t)handed * kChunk, length(handed));
        ++handed;
    };
    while (handed < chunks && handed < kSlots) fill();
    for (int c = 0; c < chunks && e == hipSuccess; ++c) {
        const int slot = c % kSlots;
        slots_[slot].copied.wait();
        e = hipMemcpyAsync(out + (size_t)c * kChunk, ring_ + (size_t)slot * kChunk, length(c), hipMemcpyHostToDevice, s);
        if (e == hipSuccess) e = hipEventRecord(ev_[slot], s);
        if (e == hipSuccess && c >= kBehind && handed < chunks) {
            e = hipEventSynchronize(ev_[(c - kBehind) % kSlots]);
            if (e == hipSuccess) fill();
        }
    }
    for (int c = std::max(0, handed - kSlots); c < handed; ++c) slots_[c % kSlots].copied.wait();
    const hipError_t w = hipStreamSynchronize(s);
    return e == hipSuccess ? w : e;
}

}  // namespace prt

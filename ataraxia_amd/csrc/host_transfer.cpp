// host_transfer.cpp -- see host_transfer.h.
#include "host_transfer.h"

#include <stdlib.h>
#include <string.h>
#include <sys/mman.h>

#include <algorithm>
#include <atomic>
#include <thread>

namespace atx {

namespace {

// The parts of one copy, shared by the threads that copy them.  Part k lies at
// src + (k % slots) * part; done[] holds the number after the last part copied
// out of each slot.
struct Parts {
    static constexpr uint32_t kMaxSlots = 4;
    char* dst;
    const char* src;
    size_t bytes, part;
    uint32_t count, slots;
    std::atomic<uint32_t> ready{0};   // parts that may be copied
    std::atomic<uint32_t> next{0};    // parts taken
    std::atomic<uint32_t> done[kMaxSlots] = {};
    std::atomic<bool> stop{false};

    void copy(uint32_t k)
    {
        const size_t off = (size_t)k * part;
        memcpy(dst + off, src + (size_t)(slots ? k % slots : k) * part, std::min(part, bytes - off));
        if (slots) done[k % slots].store(k + 1u, std::memory_order_release);
    }
    // Takes part after part; ends when all are taken or at `stop`.
    void run()
    {
        for (;;) {
            const uint32_t k = next.fetch_add(1, std::memory_order_relaxed);
            if (k >= count) return;
            for (uint32_t spin = 0; ready.load(std::memory_order_acquire) <= k; ++spin) {
                if (stop.load(std::memory_order_relaxed)) return;
                pause(spin);
            }
            copy(k);
        }
    }
    // Copies a part if one is ready that no thread has taken.
    bool run_one()
    {
        uint32_t k = next.load(std::memory_order_relaxed);
        while (k < ready.load(std::memory_order_acquire))
            if (next.compare_exchange_weak(k, k + 1u, std::memory_order_relaxed)) {
                copy(k);
                return true;
            }
        return false;
    }
    static void pause(uint32_t spin)
    {
        if (spin % 64 == 63) std::this_thread::yield();
        else __builtin_ia32_pause();
    }
};

// Up to n threads that run(); fewer when the system gives no more.
class Helpers {
public:
    Helpers(Parts& p, uint32_t n)
    {
        try {
            for (; n_ < n && n_ < 3; ++n_)
                t_[n_] = std::thread([&p] { p.run(); });
        } catch (...) {
        }
    }
    ~Helpers()
    {
        for (uint32_t k = 0; k < n_; ++k)
            t_[k].join();
    }

private:
    std::thread t_[3];
    uint32_t n_ = 0;
};

// Whether the runtime knows the memory at p.
bool known_to_runtime(const void* p)
{
    hipPointerAttribute_t a{};
    if (hipPointerGetAttributes(&a, p) != hipSuccess) {
        (void)hipGetLastError();
        return false;
    }
    return a.type != hipMemoryTypeUnregistered;
}

}  // namespace

HostStage::~HostStage()
{
    for (hipEvent_t e : ev_)
        if (e) (void)hipEventDestroy(e);
    if (block_) (void)hipHostFree(block_);
}

// The events, on the stream's device: they are recorded there, whichever device
// the calling thread has current.
hipError_t HostStage::make_events(hipStream_t stream)
{
    if (ev_[kSlots - 1]) return hipSuccess;
    int here = 0;
    hipDevice_t there = 0;
    hipError_t r = hipGetDevice(&here);
    if (r == hipSuccess) r = hipStreamGetDevice(stream, &there);
    if (r == hipSuccess && there != here) r = hipSetDevice(there);
    for (hipEvent_t& e : ev_)
        if (r == hipSuccess && !e) r = hipEventCreateWithFlags(&e, hipEventDisableTiming);
    if (there != here) (void)hipSetDevice(here);
    return r;
}

hipError_t HostStage::reserve(size_t bytes, hipStream_t stream)
{
    const hipError_t made = make_events(stream);
    if (made != hipSuccess) return made;
    if (bytes <= n_) return hipSuccess;
    if (block_) (void)hipHostFree(block_);
    block_ = nullptr;
    n_ = 0;
    const hipError_t r = hipHostMalloc((void**)&block_, bytes, hipHostMallocDefault);
    if (r == hipSuccess) n_ = bytes;
    else block_ = nullptr;
    return r;
}

hipError_t HostStage::copy_parts(char* dst, const char* src, size_t bytes, hipStream_t stream)
{
    Parts p;
    p.dst = dst;
    p.src = block_;
    p.bytes = bytes;
    p.part = std::min(bytes, kPartBytes);
    p.count = (uint32_t)((bytes + p.part - 1) / p.part);
    p.slots = kSlots;
    Helpers helpers(p, std::min(kCopyThreads, p.count) - 1u);
    hipError_t e = hipSuccess;
    uint32_t queued = 0, arrived = 0, spin = 0;
    while (arrived < p.count) {
        // the next part's slot is free once the part before it there is copied on
        while (queued < p.count && (queued < kSlots || p.done[queued % kSlots].load(std::memory_order_acquire) ==
                                                            queued - kSlots + 1u)) {
            const size_t off = (size_t)queued * p.part;
            e = hipMemcpyAsync(block_ + (queued % kSlots) * p.part, src + off, std::min(p.part, bytes - off),
                               hipMemcpyDeviceToHost, stream);
            if (e == hipSuccess) e = hipEventRecord(ev_[queued % kSlots], stream);
            if (e != hipSuccess) break;
            ++queued;
        }
        if (e == hipSuccess && arrived < queued) {
            e = hipEventSynchronize(ev_[arrived % kSlots]);
            if (e == hipSuccess) p.ready.store(++arrived, std::memory_order_release);
        } else if (e == hipSuccess && !p.run_one()) {
            Parts::pause(spin++);
        }
        if (e != hipSuccess) {
            p.stop.store(true, std::memory_order_relaxed);
            (void)hipStreamSynchronize(stream);   // nothing writes the block any more
            return e;
        }
    }
    p.run();
    return hipSuccess;
}

hipError_t HostStage::copy_out(void* dst, const void* src, size_t bytes, hipStream_t stream)
{
    if (bytes == 0) return hipSuccess;
    std::lock_guard<std::mutex> lk(mu_);
    bool staged = !known_to_runtime(dst);
    if (staged && reserve(std::min(bytes, kSlots * kPartBytes), stream) != hipSuccess) {
        (void)hipGetLastError();
        staged = false;
    }
    if (staged)
        return copy_parts(static_cast<char*>(dst), static_cast<const char*>(src), bytes, stream);
    const hipError_t e = hipMemcpyAsync(dst, src, bytes, hipMemcpyDeviceToHost, stream);
    return e != hipSuccess ? e : hipStreamSynchronize(stream);
}

void HostFree::operator()(void* p) const { free(p); }

HostMem host_alloc(size_t bytes)
{
    const size_t huge = size_t(2) << 20;
    if (bytes < 2 * huge) return HostMem(malloc(bytes ? bytes : 1));
    HostMem m(aligned_alloc(huge, (bytes + huge - 1) / huge * huge));
    if (m) (void)madvise(m.get(), bytes, MADV_HUGEPAGE);
    return m;
}

void copy_threaded(void* dst, const void* src, size_t bytes)
{
    Parts p;
    p.dst = static_cast<char*>(dst);
    p.src = static_cast<const char*>(src);
    p.bytes = bytes;
    p.part = size_t(1) << 20;
    p.count = (uint32_t)((bytes + p.part - 1) / p.part);
    p.slots = 0;
    p.ready.store(p.count);
    Helpers helpers(p, p.count > 1 ? std::min(4u, p.count) - 1u : 0u);
    p.run();
}

}  // namespace atx

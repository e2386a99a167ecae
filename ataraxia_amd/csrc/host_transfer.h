// host_transfer.h -- device results into the caller's (pageable) memory.
#pragma once

#include <hip/hip_runtime.h>
#include <stddef.h>
#include <stdint.h>

#include <memory>
#include <mutex>

namespace atx {

// Copies device memory to pageable host memory through a pinned block that
// its owner (a renderer, a batch, a server) keeps: the device copies part
// after part into the block at the link's rate (8.3 MB: 157 us) while up to
// kCopyThreads threads, the caller among them, copy the finished parts on.
// The runtime's own pageable copy takes its parts one after another, each
// waited for, and one thread touches the destination's fresh pages: 8 MB into
// new memory 2000 us, with huge pages 790, into pages already there 480; four
// threads on huge pages take 225 us.  Copies by several threads take turns.
class HostStage {
public:
    HostStage() = default;
    ~HostStage();
    HostStage(const HostStage&) = delete;
    HostStage& operator=(const HostStage&) = delete;
    // Waits for the copy (and for what is on `stream` before it).  Memory
    // the runtime knows (pinned, managed, device) is copied to directly, and so
    // is any when no pinned block can be had.
    hipError_t copy_out(void* dst, const void* src, size_t bytes, hipStream_t stream);

private:
    static constexpr uint32_t kCopyThreads = 4;
    // Four parts of 1 MiB in flight: the first touch of a pinned block costs
    // the host about 60 us per MiB, so the block is no larger than the pipeline
    // needs.  A copy of one part is copied on by the caller alone.
    static constexpr uint32_t kSlots = 4;
    static constexpr size_t kPartBytes = size_t(1) << 20;
    hipError_t make_events(hipStream_t stream);
    hipError_t reserve(size_t bytes, hipStream_t stream);
    hipError_t copy_parts(char* dst, const char* src, size_t bytes, hipStream_t stream);
    std::mutex mu_;
    char* block_ = nullptr;
    size_t n_ = 0;
    hipEvent_t ev_[kSlots] = {};
};

// Host memory for results that wait for their caller, not cleared; on huge
// pages from 4 MiB on (an eighth of the time to touch them first).
struct HostFree {
    void operator()(void* p) const;
};
using HostMem = std::unique_ptr<void, HostFree>;
HostMem host_alloc(size_t bytes);   // empty when there is none

// memcpy by up to four threads (large blocks, fresh destination pages).
void copy_threaded(void* dst, const void* src, size_t bytes);

}  // namespace atx

// Device results to caller memory, through pinned staging where that is pageable.
//
// A copy to pageable memory goes through the runtime's own staging buffer one
// MiB at a time, the transfer and the CPU copy (which also faults in the
// caller's fresh pages) taking turns: about 90 us per MiB, of which the transfer
// is 20.  Here every piece is transferred to pinned memory at once and copied
// out by up to kThreads threads as it arrives: a 1080p float image 2.33 -> 1.26 ms,
// 720p 0.86 -> 0.57 ms, 400 x 300 145 -> 120 us (with one thread 1.40 and 0.95 ms;
// pieces of 4 MiB 1.60 ms at 1080p, of 0.5 and 0.25 MiB slower by 0.4 and 1 ms).
#pragma once
#include <hip/hip_runtime.h>

#include <cstddef>

namespace lfh {

class Readback {
public:
    Readback() = default;
    Readback(const Readback&) = delete;
    Readback& operator=(const Readback&) = delete;
    ~Readback() { release(); }
    // Copies `bytes` of device memory to dst and, when d_flag is given, the int
    // there to *flag, after the work queued on s; both are there on return.
    hipError_t read(void* dst, const void* src, size_t bytes, const int* d_flag, int* flag, int device,
                    hipStream_t s);
    void release();

private:
    static constexpr size_t kPiece = (size_t)1 << 20;
    static constexpr int kPieces = 32;   // pinned memory held: at most 32 MiB and the flag
    static constexpr int kThreads = 4;
    hipError_t ensure(size_t bytes);
    char* pin_ = nullptr;
    size_t cap_ = 0;                     // bytes of pin_ for pieces; the flag follows
    hipEvent_t ev_[kPieces] = {};
};

}  // namespace lfh

// Workspace of the C entry points that split a reduction without a caller
// workspace (attn_fwd_split_static, launch / attn_fwd for grids too small for
// the GPU, conv3d_fwd / launch_conv3d likewise). Internal to the library.
//
// The partial results live in a file-scope device array. It is part of the
// library's code object, so every GPU on which any kernel of the library is
// loaded holds its own copy (kScratchBytes) until the process ends, whether or
// not a call ever uses it. The kernels write every workspace entry the merge
// reads within the same call, so nothing is cleared between calls.
//
// A call takes as many consecutive pieces of the array (kScratchPiece) as it
// needs. Calls that use the same piece are ordered on the GPU, whatever streams
// they are issued on: each records an event on its stream after its kernels,
// and the next one first makes its stream wait for that event (the host lock
// keeps wait, launches and record of one call together). Calls on different
// streams are given different pieces while these last, and run side by side
// (conv3d 512 -> 512 of 512 voxels on four streams: 28 us a call as one chain,
// 13 side by side, 22 on one stream). A call made under stream capture takes
// the first pieces and neither waits nor records (an event recorded outside the
// graph cannot order its replays): a graph that contains one is ordered only by
// the stream it is launched on, and must not run concurrently with other
// streams' calls that use the array on that device.
#pragma once

#include <stddef.h>
#include <hip/hip_runtime_api.h>
#include <mutex>

namespace gfx906_amd {

constexpr size_t kScratchBytes = size_t(96) << 20;
constexpr size_t kScratchPiece = size_t(6) << 20;

struct DevScratch;

// One call's use of the scratch of its stream's device: acquire() before its
// launches, release() after them; the lock is held in between. A call that ends
// on an error releases it too (a launch before the failed one may be queued):
// the destructor does.
class ScratchUse {
 public:
    enum Status {
        kReady,        // ptr is usable
        kUnavailable,  // under capture: not allowed, or no call outside capture has set it up
        kFailed,       // error: `error`
    };
    ScratchUse();
    ~ScratchUse() { (void)release(); }
    ScratchUse(const ScratchUse&) = delete;
    ScratchUse& operator=(const ScratchUse&) = delete;
    // bytes > 0; more than kScratchBytes fails.
    Status acquire(hipStream_t stream, size_t bytes, bool allow_capture);
    hipError_t release();  // no-op unless acquired

    void* ptr = nullptr;
    const char* error = nullptr;

 private:
    std::unique_lock<std::mutex> lock_;
    DevScratch* dev_ = nullptr;
    hipStream_t stream_ = nullptr;
    const void* key_ = nullptr;  // what tells streams apart (a preference only)
    int first_ = 0, count_ = 0;  // pieces
    bool capturing_ = false;
};

}  // namespace gfx906_amd

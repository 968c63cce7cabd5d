// Static device scratch shared by the calls that split a reduction without a
// caller workspace (see scratch.h).
#include <hip/hip_runtime.h>

#include "scratch.h"

namespace gfx906_amd {

// Host code must not pass `scratch` itself to a kernel (on the host it names a
// stand-in, not device memory): it uses the device address that
// hipGetSymbolAddress returns, looked up once per device.
static __device__ __align__(256) char scratch[kScratchBytes];

constexpr int kMaxDevices = 64;
constexpr int kPieces = kScratchBytes / kScratchPiece;
static_assert(kPieces * kScratchPiece == kScratchBytes, "whole pieces");

// A piece of a device's scratch as the last call outside capture left it.
struct ScratchPiece {
    hipEvent_t done;     // recorded by the last call whose first piece this was
    int guard;           // the piece whose `done` covers the last call that used this one
    const void* stream;  // that call's stream, a preference only
    unsigned long long used;  // number of that call (0: none)
};
struct DevScratch {
    void* ptr;  // device address of `scratch`
    unsigned long long calls;
    ScratchPiece piece[kPieces];
};

namespace {

std::mutex g_scratch_mu;
DevScratch g_scratch[kMaxDevices];

// Looks up `scratch` on device dev and creates its ordering events, once.
// Caller holds g_scratch_mu.
hipError_t scratch_setup(int dev) {
    DevScratch& d = g_scratch[dev];
    if (d.ptr) return hipSuccess;
    int cur = 0;
    hipError_t e = hipGetDevice(&cur);
    if (e == hipSuccess && dev != cur) e = hipSetDevice(dev);
    if (e != hipSuccess) return e;
    void* p = nullptr;
    e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
    if (e == hipSuccess && !p) e = hipErrorInvalidSymbol;
    // The events only order kernels of this device on two of its streams
    // (hipStreamWaitEvent); nothing on the host or on another device inspects
    // them, so their records need no system-scope fence: the kernels' own release
    // at their end makes the scratch visible to the device's later kernels.
    // Without the fence a call that splits costs about 2 us less of GPU time
    // (measured on MI355X: B1 H1 S1024 D64 through launch() 16.3 -> 14.5 us).
    int made = 0;
    while (e == hipSuccess && made < kPieces) {
        e = hipEventCreateWithFlags(&d.piece[made].done,
                                    hipEventDisableTiming | hipEventDisableSystemFence);
        made += e == hipSuccess;
    }
    if (dev != cur) {
        const hipError_t r = hipSetDevice(cur);
        if (e == hipSuccess) e = r;
    }
    if (e != hipSuccess) {
        while (made > 0) (void)hipEventDestroy(d.piece[--made].done);
        return e;
    }
    d.ptr = p;
    return hipSuccess;
}

// First of the n pieces for a call on `stream`: pieces that the stream's last
// calls used (no other call to wait for), else the ones unused for longest.
int pick_pieces(const DevScratch& d, int n, const void* stream) {
    int best = 0;
    unsigned long long best_used = ~0ull;
    for (int p = 0; p + n <= kPieces; ++p) {
        bool own = true;
        unsigned long long used = 0;
        for (int k = p; k < p + n; ++k) {
            own = own && d.piece[k].used && d.piece[k].stream == stream;
            if (d.piece[k].used > used) used = d.piece[k].used;
        }
        if (own) return p;
        if (used < best_used) {
            best_used = used;
            best = p;
        }
    }
    return best;
}

}  // namespace

ScratchUse::ScratchUse() : lock_(g_scratch_mu, std::defer_lock) {}

ScratchUse::Status ScratchUse::acquire(hipStream_t stream, size_t bytes,
                                       bool allow_capture) {
    auto failed = [&](hipError_t e) {
        error = hipGetErrorString(e);
        return kFailed;
    };
    // Device of `stream` (the current device for the null stream).
    int dev = 0;
    hipError_t e = hipGetDevice(&dev);
    if (e == hipSuccess && stream) e = hipStreamGetDevice(stream, &dev);
    if (e != hipSuccess) return failed(e);
    if (dev < 0 || dev >= kMaxDevices) {
        error = "device index beyond the scratch table";
        return kFailed;
    }
    hipStreamCaptureStatus st = hipStreamCaptureStatusNone;
    if ((e = hipStreamIsCapturing(stream, &st)) != hipSuccess) return failed(e);
    capturing_ = st != hipStreamCaptureStatusNone;
    if (capturing_ && !allow_capture) return kUnavailable;
    lock_.lock();
    DevScratch& d = g_scratch[dev];
    if (!d.ptr) {
        if (capturing_) return kUnavailable;
        if ((e = scratch_setup(dev)) != hipSuccess) return failed(e);
    }
    if (bytes > kScratchBytes) {
        error = "more than the scratch holds";
        return kFailed;
    }
    dev_ = &d;
    stream_ = stream;
    count_ = (int)((bytes + kScratchPiece - 1) / kScratchPiece);
    first_ = 0;
    ptr = d.ptr;
    if (capturing_) return kReady;
    static thread_local char this_thread;
    key_ = stream == hipStreamPerThread ? (const void*)&this_thread : (const void*)stream;
    first_ = pick_pieces(d, count_, key_);
    ptr = (char*)d.ptr + first_ * kScratchPiece;
    // Also where the last call's stream has this one's handle: handles do not
    // name streams (a new stream can get a destroyed one's). The runtime, which
    // knows the stream, drops the wait where it really is the same.
    for (int k = first_; k < first_ + count_; ++k) {
        const ScratchPiece& sp = d.piece[k];
        if (!sp.used || (k > first_ && sp.guard == d.piece[k - 1].guard && d.piece[k - 1].used))
            continue;
        if ((e = hipStreamWaitEvent(stream, d.piece[sp.guard].done, 0)) != hipSuccess) {
            dev_ = nullptr;
            return failed(e);
        }
    }
    return kReady;
}

hipError_t ScratchUse::release() {
    DevScratch* const d = dev_;
    dev_ = nullptr;
    if (!d || capturing_) return hipSuccess;
    // One record covers all pieces. It may replace one that other pieces still
    // name as their guard; this call waited for that one, so the new one covers
    // it too.
    const hipError_t e = hipEventRecord(d->piece[first_].done, stream_);
    if (e != hipSuccess) {  // (no event to order the next call by)
        (void)hipStreamSynchronize(stream_);
        return e;
    }
    ++d->calls;
    for (int k = first_; k < first_ + count_; ++k) {
        d->piece[k].guard = first_;
        d->piece[k].stream = key_;
        d->piece[k].used = d->calls;
    }
    return hipSuccess;
}

}  // namespace gfx906_amd

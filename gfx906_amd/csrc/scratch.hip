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
struct DevScratch {
    void* ptr;           // device address of `scratch`
    hipEvent_t done;     // recorded after the last call outside capture that used it
    bool recorded;
};

namespace {

std::mutex g_scratch_mu;
DevScratch g_scratch[kMaxDevices];

// Looks up `scratch` on device dev and creates its ordering event, once.
// Caller holds g_scratch_mu.
hipError_t scratch_setup(int dev) {
    DevScratch& d = g_scratch[dev];
    if (d.ptr) return hipSuccess;
    int cur = 0;
    hipError_t e = hipGetDevice(&cur);
    if (e == hipSuccess && dev != cur) e = hipSetDevice(dev);
    if (e != hipSuccess) return e;
    void* p = nullptr;
    hipEvent_t ev = nullptr;
    e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
    if (e == hipSuccess && !p) e = hipErrorInvalidSymbol;
    // The event only orders kernels of this device on two of its streams
    // (hipStreamWaitEvent); nothing on the host or on another device inspects
    // it, so its record needs no system-scope fence: the kernels' own release
    // at their end makes the scratch visible to the device's later kernels.
    // Without the fence a call that splits costs about 2 us less of GPU time
    // (measured on MI355X: B1 H1 S1024 D64 through launch() 16.3 -> 14.5 us).
    if (e == hipSuccess)
        e = hipEventCreateWithFlags(&ev, hipEventDisableTiming | hipEventDisableSystemFence);
    if (dev != cur) {
        const hipError_t r = hipSetDevice(cur);
        if (e == hipSuccess) e = r;
    }
    if (e != hipSuccess) {
        if (ev) (void)hipEventDestroy(ev);
        return e;
    }
    d.ptr = p;
    d.done = ev;
    d.recorded = false;
    return hipSuccess;
}

}  // namespace

ScratchUse::ScratchUse() : lock_(g_scratch_mu, std::defer_lock) {}

ScratchUse::Status ScratchUse::acquire(hipStream_t stream, bool allow_capture) {
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
    // Also where the last call's stream has this one's handle: handles do not
    // name streams (hipStreamPerThread is one value for every thread's own
    // stream, and a new stream can get a destroyed one's). The runtime, which
    // knows the stream, drops the wait where it really is the same.
    if (!capturing_ && d.recorded && (e = hipStreamWaitEvent(stream, d.done, 0)) != hipSuccess)
        return failed(e);
    dev_ = &d;
    stream_ = stream;
    ptr = d.ptr;
    return kReady;
}

hipError_t ScratchUse::release() {
    DevScratch* const d = dev_;
    dev_ = nullptr;
    if (!d || capturing_) return hipSuccess;
    const hipError_t e = hipEventRecord(d->done, stream_);
    if (e == hipSuccess)
        d->recorded = true;
    else  // (no event to order the next call by)
        (void)hipStreamSynchronize(stream_);
    return e;
}

}  // namespace gfx906_amd

// ScratchUse (gfx906_amd/csrc/scratch.hip) on a HIP runtime that only keeps
// account: streams and events are numbers, and every wait and record is a line
// of output. argv[1] names the sequence of calls. Built and run by
// test_scratch_order.py with the host compiler; needs no GPU.
#include <cstdio>
#include <cstring>
#include <thread>

#include "scratch.h"

using gfx906_amd::kScratchBytes;
using gfx906_amd::kScratchPiece;
using gfx906_amd::ScratchUse;

static int n_events = 0, record_fails = 0;
static bool capturing = false;

extern "C" {
hipError_t hipGetDevice(int* dev) { return *dev = 0, hipSuccess; }
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipStreamGetDevice(hipStream_t, hipDevice_t* dev) { return *dev = 0, hipSuccess; }
hipError_t hipStreamIsCapturing(hipStream_t, hipStreamCaptureStatus* st) {
    *st = capturing ? hipStreamCaptureStatusActive : hipStreamCaptureStatusNone;
    return hipSuccess;
}
hipError_t hipGetSymbolAddress(void** p, const void*) {
    return *p = reinterpret_cast<void*>(uintptr_t(1) << 40), hipSuccess;
}
hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) {
    *e = reinterpret_cast<hipEvent_t>(uintptr_t(++n_events));
    return hipSuccess;
}
hipError_t hipEventDestroy(hipEvent_t) { return hipSuccess; }
hipError_t hipStreamWaitEvent(hipStream_t s, hipEvent_t e, unsigned) {
    std::printf("wait s%d e%d\n", int((uintptr_t)s), int((uintptr_t)e));
    return hipSuccess;
}
hipError_t hipEventRecord(hipEvent_t e, hipStream_t s) {
    if (record_fails > 0) return --record_fails, hipErrorUnknown;
    std::printf("record s%d e%d\n", int((uintptr_t)s), int((uintptr_t)e));
    return hipSuccess;
}
hipError_t hipStreamSynchronize(hipStream_t s) {
    std::printf("synchronize s%d\n", int((uintptr_t)s));
    return hipSuccess;
}
const char* hipGetErrorString(hipError_t) { return "error"; }
}

static hipStream_t stream(int n) { return reinterpret_cast<hipStream_t>(uintptr_t(n)); }

// One call on stream n with `pieces` pieces of the scratch.
static void call(int n, int pieces = 1) {
    ScratchUse use;
    if (use.acquire(stream(n), pieces * kScratchPiece - 1, true) != ScratchUse::kReady)
        std::printf("not ready\n");
    std::printf("call s%d %d+%d\n", n,
                int(((uintptr_t)use.ptr - (uintptr_t(1) << 40)) / kScratchPiece), pieces);
    if (use.release() != hipSuccess) std::printf("not released\n");
}

int main(int argc, char** argv) {
    const char* what = argc > 1 ? argv[1] : "";
    if (!std::strcmp(what, "same handle")) {
        call(7);
        call(7);  // (7 destroyed, and a new stream given its handle)
        call(7);
    } else if (!std::strcmp(what, "threads")) {
        call(2), call(2);  // hipStreamPerThread's value
        std::thread([] { call(2), call(2); }).join();
    } else if (!std::strcmp(what, "full")) {
        call(7, 10);
        call(8, 10);   // no ten other pieces are left
        call(9, 6);
        call(7, 10);
        call(9, 1);
        call(8, 16);
        call(7, 1);
    } else if (!std::strcmp(what, "guards")) {
        call(7, 8);
        call(8, 8);
        call(7, 1);    // records what pieces 1-7 are guarded by
        call(9, 16);
        ScratchUse use;
        std::printf("%d\n", use.acquire(stream(7), kScratchBytes + 1, true) == ScratchUse::kFailed);
    } else if (!std::strcmp(what, "two streams")) {
        call(7);
        call(8);
        call(7);
    } else if (!std::strcmp(what, "failed call")) {
        {
            ScratchUse use;  // its second launch fails: no release()
            use.acquire(stream(7), kScratchBytes, true);
            std::printf("launch s7\n");
        }
        call(8);
    } else if (!std::strcmp(what, "failed record")) {
        record_fails = 1;
        call(7);
        call(8);
    } else if (!std::strcmp(what, "capture")) {
        call(7);
        capturing = true;
        call(8);
        capturing = false;
        call(9);
    } else {
        return 1;
    }
    return 0;
}

"""The static scratch shared by host threads, each on its own default stream.

hipStreamPerThread is one handle for as many streams as there are threads. Two
threads issue conv3d_fwd and attn_fwd calls that split, all through the static
scratch, at the same time; every result equals its serial one bit for bit.
"""

import ctypes
import threading

import pytest
import torch

import gfx906_amd
from gfx906_amd import kitchen
from oracle import conv3d as oc

pytestmark = pytest.mark.gpu
PER_THREAD = ctypes.c_void_p(2)  # hipStreamPerThread
CL = torch.channels_last_3d


def hip_runtime():
    """The HIP runtime that this process has loaded."""
    with open("/proc/self/maps") as f:
        return ctypes.CDLL(next(p for p in (line.split()[-1] for line in f) if "libamdhip64" in p))


def make_attn(lib, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    q, k, v = (torch.randn(1, 4, 2048, 128, generator=g, device="cuda").half() for _ in range(3))
    assert lib.attn_split_workspace_bytes(1, 4, 2048, 2048, 128) > 0

    def run(stream):
        o = torch.empty_like(q)
        torch.cuda.synchronize()

        def issue():
            rc = lib.attn_fwd(q.data_ptr(), k.data_ptr(), v.data_ptr(), o.data_ptr(), 1, 4, 2048,
                              2048, 128, ctypes.c_float(0.088), stream)
            assert rc == 0, lib.attn_last_error()
        return o, issue
    return run


def make_conv(lib, seed):
    x, w, b, res = oc.make_case((1, 256, 3, 18, 18), (256, 3, 3, 3), (1, 1, 1), True, True, seed)
    dev = [torch.from_numpy(a).cuda().contiguous(
        memory_format=CL if a.ndim == 5 else torch.contiguous_format) for a in (x, w, b, res)]
    call = kitchen.plan(*dev, [1, 1, 1])
    n, d, h, ww, c, k, t, r, s, sd, sh, sw, z, p, q = call.dims

    def run(stream):
        o = torch.empty_like(call.out)
        torch.cuda.synchronize()
        ptr = [a.data_ptr() for a in (call.x, call.weight, call.bias, call.residual, o)]
        args = ([ctypes.c_void_p(a) for a in ptr] + [ctypes.c_int(a) for a in call.dims]
                + [ctypes.c_long(n * z * p * q)]
                + [ctypes.c_long(a) for a in (*call.xs, *call.os, *call.rs)] + [stream])

        def issue():
            assert lib.conv3d_fwd(*args) == 0
        return o, issue
    return run


def test_two_threads_on_their_own_streams():
    print("case scratch: two threads on hipStreamPerThread", flush=True)
    lib = ctypes.CDLL(str(gfx906_amd.KERNEL_LIB))
    lib.attn_last_error.restype = ctypes.c_char_p
    lib.attn_split_workspace_bytes.restype = ctypes.c_size_t
    lib.attn_fwd.argtypes = [ctypes.c_void_p] * 4 + [ctypes.c_int] * 5 + [ctypes.c_float,
                                                                          ctypes.c_void_p]
    jobs = [make_attn(lib, 1), make_conv(lib, 2), make_conv(lib, 3), make_attn(lib, 4)]
    serial = []
    for job in jobs:
        o, issue = job(ctypes.c_void_p(0))
        issue()
        torch.cuda.synchronize()
        serial.append(o)
    rounds = [[(n, *jobs[n](PER_THREAD)) for _ in range(10) for n in mine]
              for mine in ((0, 1), (2, 3))]  # (all buffers before the first call)
    errors, hip = [], hip_runtime()

    def work(mine):
        try:
            for _, _, issue in mine:
                issue()
            assert hip.hipStreamSynchronize(PER_THREAD) == 0  # (it ends with its thread)
        except BaseException as e:  # noqa: BLE001
            errors.append(e)

    threads = [threading.Thread(target=work, args=(mine,)) for mine in rounds]
    for t in threads:
        t.start()
    for t in threads:
        t.join(60)
    torch.cuda.synchronize()
    assert not errors, errors
    for mine in rounds:
        for n, o, _ in mine:
            assert torch.equal(o, serial[n]), n

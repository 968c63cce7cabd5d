"""conv3d with its reduction split over several workgroups.

A problem with few output tiles splits its reduction into ranges whose fp32
sums a second kernel adds up. The tests force range counts around the edges
(one unit per range, counts that do not divide the units, a batch of the
reduce kernel and one more) on small layers, through the op (workspace from
torch) and the C entry (static scratch, bit-equal), and check the planner's
own choice on a layer small enough to be split. The bar is the fp16 half-ulp
of the exact result plus 1e-3, as for the unsplit kernel. Each case prints its
parameters first.
"""

import ctypes

import numpy as np
import pytest
import torch

import gfx906_amd
from gfx906_amd import kitchen
from oracle import conv3d as oc

DEV = "cuda"
CL = torch.channels_last_3d


def lib():
    h = ctypes.CDLL(str(gfx906_amd.KERNEL_LIB))
    h.conv3d_workspace_bytes.restype = ctypes.c_size_t
    h.conv3d_workspace_bytes.argtypes = [ctypes.c_long, ctypes.c_int, ctypes.c_long]
    h.conv3d_last_error.restype = ctypes.c_char_p
    return h


def to_dev(a):
    return None if a is None else torch.from_numpy(a).to(DEV).contiguous(
        memory_format=CL if a.ndim == 5 else torch.contiguous_format)


def run_capi(call):
    n, d, h, w, c, k, t, r, s, sd, sh, sw, z, p, q = call.dims
    out = torch.empty_like(call.out)
    ptr = [x.data_ptr() if x is not None else 0
           for x in (call.x, call.weight, call.bias, call.residual, out)]
    args = ([ctypes.c_void_p(x) for x in ptr] + [ctypes.c_int(v) for v in call.dims]
            + [ctypes.c_long(n * z * p * q)]
            + [ctypes.c_long(v) for v in (*call.xs, *call.os, *call.rs)]
            + [ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)])
    handle = lib()
    assert handle.conv3d_fwd(*args) == 0, handle.conv3d_last_error()
    return out


def check(got, exact, what):
    g = got.detach().float().cpu().double()
    e = torch.from_numpy(np.ascontiguousarray(exact))
    _, ex = torch.frexp(e.abs())
    bar = torch.ldexp(torch.ones_like(e), (ex - 12).clamp(min=-25)) + 1e-3
    d = (g - e).abs()
    print(f"{what}: max-abs {d.max().item():.3e}", flush=True)
    assert bool((d <= bar).all()), (what, d.max().item())


CASES = [  # x, (k, window), stride, bias, residual; C = 8: a unit spans taps, 27 units of 8 left over
    ((1, 64, 3, 10, 12), (64, 3, 3, 3), (1, 1, 1), True, True),
    ((1, 8, 4, 9, 11), (24, 3, 3, 3), (1, 1, 1), False, True),
    ((2, 40, 3, 9, 9), (136, 3, 3, 3), (2, 2, 2), True, False),
    ((1, 512, 1, 6, 6), (8, 1, 1, 1), (1, 1, 1), True, False),
]


@pytest.mark.gpu
@pytest.mark.parametrize("nsplit", [1, 2, 3, 4, 5, 8, 64])
@pytest.mark.parametrize("i", range(len(CASES)))
@pytest.mark.parametrize("cfg", ["4x32", "3x64", "2x64", "4x32x256", "3x64x256", "2x64x256",
                                 "3x32x256", "4x64x128", "2x64x64"])
def test_forced_split_counts(monkeypatch, cfg, i, nsplit):
    xs, ws, stride, has_b, has_r = CASES[i]
    print(f"case conv split: {cfg} {xs} {ws} n{nsplit}", flush=True)
    x, w, b, res = oc.make_case(xs, ws, stride, has_b, has_r, seed=500 + i)
    call = kitchen.plan(to_dev(x), to_dev(w), to_dev(b), to_dev(res), list(stride))
    monkeypatch.setenv("GFX906_AMD_CONV_CFG", cfg)
    monkeypatch.setenv("GFX906_AMD_CONV_NSPLIT", str(nsplit))
    got = call.run(gfx906_amd.extension()).clone()
    capi = run_capi(call)
    torch.cuda.synchronize()
    check(got, oc.conv3d_gemm(x, w, b, res, stride), f"{cfg} case{i} n{nsplit}")
    assert torch.equal(got, capi)


@pytest.mark.gpu
@pytest.mark.parametrize("nsplit", [1, 2, 3])
@pytest.mark.parametrize("c,k", [(8, 24), (16, 200), (32, 64), (40, 136), (56, 512)])
def test_small_channel_counts(monkeypatch, c, k, nsplit):
    """C < 64: the configuration is chosen anew for the planned ranges."""
    print(f"case conv split: C{c} K{k} n{nsplit}", flush=True)
    x, w, b, res = oc.make_case((1, c, 4, 12, 21), (k, 3, 3, 3), (1, 1, 1), True, True, seed=600 + c)
    call = kitchen.plan(to_dev(x), to_dev(w), to_dev(b), to_dev(res), [1, 1, 1])
    monkeypatch.setenv("GFX906_AMD_CONV_NSPLIT", str(nsplit))
    got = call.run(gfx906_amd.extension()).clone()
    capi = run_capi(call)
    torch.cuda.synchronize()
    check(got, oc.conv3d_gemm(x, w, b, res, (1, 1, 1)), f"C{c} n{nsplit}")
    assert torch.equal(got, capi)


@pytest.mark.gpu
def test_small_layer_is_split_and_accurate_in_a_graph(monkeypatch):
    x, w, b, res = oc.make_case((1, 256, 3, 18, 18), (256, 3, 3, 3), (1, 1, 1), True, True, 510)
    print("case conv split: planner's own choice, eager and captured", flush=True)
    assert lib().conv3d_workspace_bytes(256, 256, 256 * 27) > 0
    ext = gfx906_amd.extension()
    call = kitchen.plan(to_dev(x), to_dev(w), to_dev(b), to_dev(res), [1, 1, 1])
    eager = call.run(ext).clone()
    capi = run_capi(call)
    check(eager, oc.conv3d_gemm(x, w, b, res, (1, 1, 1)), "planned split")
    assert torch.equal(eager, capi)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        call.run(ext)
        unsplit = run_capi(call)  # the C entry takes no scratch under capture
    with monkeypatch.context() as m:
        m.setenv("GFX906_AMD_CONV_NSPLIT", "1")
        plain = run_capi(call)
    assert not torch.equal(plain, eager)
    for _ in range(3):
        call.out.zero_()
        unsplit.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(call.out, eager)
        assert torch.equal(unsplit, plain)
        check(unsplit, oc.conv3d_gemm(x, w, b, res, (1, 1, 1)), "captured C entry")


def test_plan_sizes(monkeypatch):
    # (needs no GPU: the planner assumes 256 CUs without one)
    ws = lib().conv3d_workspace_bytes
    assert ws(23064, 512, 13824) == 0          # 242 tiles fill the GPU
    assert ws(2048, 512, 13824) % (2048 * 512 * 4) == 0 and ws(2048, 512, 13824) > 0
    assert ws(2048, 512, 256) == 0             # a short reduction
    assert ws(0, 512, 256) == 0 and ws(16, -8, 256) == 0
    for n, units in ((2, 27), (5, 27), (64, 27)):
        monkeypatch.setenv("GFX906_AMD_CONV_NSPLIT", str(n))
        per = -(-units // min(n, units))
        assert ws(100, 64, 64 * 27) == -(-units // per) * 100 * 64 * 4
    monkeypatch.setenv("GFX906_AMD_CONV_NSPLIT", "8")
    assert ws(1 << 20, 512, 13824) == 0        # 17 GB of partial sums: not split


@pytest.mark.parametrize("M,K,KG", [(1 << 40, 64, 1000), ((1 << 31) - 256, 64, 1728),
                                    (1 << 32, 64, 1728), (256, 64, 1 << 40), (256, 64, 1 << 62),
                                    (256, (1 << 31) - 8, 64), (256, 1 << 20, 1024),
                                    ((1 << 31) - 512, 1 << 20, 8)])
def test_sizes_past_the_limits_need_no_workspace(M, K, KG):
    # (needs no GPU; such calls are refused by conv3d_fwd_split itself)
    assert lib().conv3d_workspace_bytes(M, K, KG) == 0


@pytest.mark.gpu
def test_too_many_voxels_raise():
    print("case conv split: M past 2^31", flush=True)
    x, w, b, res = oc.make_case((1, 8, 1, 4, 4), (8, 1, 1, 1), (1, 1, 1), False, False, seed=1)
    call = kitchen.plan(to_dev(x), to_dev(w), None, None, [1, 1, 1])
    dims = list(call.dims)
    dims[0] = 1 << 28  # M = 2^32: refused before any launch
    with pytest.raises(RuntimeError, match="M must be"):
        gfx906_amd.extension().conv3d(call.x, call.weight, None, None, call.out, dims, call.xs,
                                      call.os, call.rs)

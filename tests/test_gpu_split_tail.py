"""Grids a little past a whole number of rounds: only the last units split.

The work units (query tiles of all heads) that fill the GPU run unsplit; the
rest split their keys, and the merge covers their rows alone. Cases put the
first split row at a head's start, inside a head and in a ragged last query
tile, with one split unit and with many, for D = 40, 64, 128 and 512, fp16 and
bf16, contiguous and [B, S, H, D] layouts. The output is held to the bars
against SDPA MATH in fp32, rows of unsplit units must equal the unsplit
kernel's bit for bit, and every entry point must give the same bits (without a
workspace, and under capture for the C entries: unsplit). Each case prints its
parameters first.
"""


import pytest
import torch

import gfx906_amd
from oracle.attention import MAX_ABS_TOL, MEAN_ABS_TOL, error_stats, make_inputs, sdpa_math_fp32

DEV = "cuda"
CASES = [  # B, H, Sq, Skv, D, dtype; slots: 256 units (512 for D <= 64)
    (1, 257, 8, 1030, 128, "fp16"),     # one split unit, its rows a head's
    (2, 129, 33, 1500, 128, "bf16"),    # two split units
    (1, 37, 1750, 2000, 128, "fp16"),   # 259 units: the last, ragged tiles of one head
    (1, 5, 13300, 1100, 128, "fp16"),   # 260 units, the first split row inside a head
    (1, 17, 7700, 1400, 64, "fp16"),    # 527 units
    (3, 172, 100, 1100, 40, "bf16"),    # 516 units, padded head dim
    (1, 52, 640, 600, 512, "fp16"),     # 260 units of 128 rows
    (2, 1, 16500, 1111, 512, "bf16"),   # 258 units, ragged
]


def handle():
    return gfx906_amd.capi()


def units(B, H, Sq, D):
    bm = 128 if D == 512 else 256
    return B * H * -(-Sq // bm), 512 if D <= 64 else 256, bm


def first_split_row(B, H, Sq, D):
    n, slots, bm = units(B, H, Sq, D)
    whole, nqt = n // slots * slots, -(-Sq // bm)
    return whole // nqt * Sq + whole % nqt * bm


@pytest.mark.parametrize("case", CASES)
def test_plan_splits_the_tail_only(case):
    # (needs no GPU: plans assume 256 CUs)
    B, H, Sq, Skv, D, _ = case
    need = handle().attn_split_workspace_bytes(B, H, Sq, Skv, D)
    rows = B * H * Sq - first_split_row(B, H, Sq, D)
    assert need > 16 and (need - 16) % (rows * (D + 2) * 4) == 0
    assert (need - 16) // (rows * (D + 2) * 4) >= 2


def test_full_grids_and_short_keys_stay_unsplit():
    f = handle().attn_split_workspace_bytes
    assert f(1, 16, 16384, 16384, 128) == 0   # 1024 units
    assert f(2, 24, 8192, 512, 64) == 0       # 1536 units of two per CU
    assert f(1, 257, 8, 640, 64) == 0         # the K/V-resident kernel's
    assert f(1, 257, 8, 200, 128) == 0        # four key tiles: nothing to split
    assert f(1, 511, 8, 2000, 128) == 0       # a nearly full last round
    assert 0 < f(1, 16, 4250, 4250, 128) <= 96 << 20


def call(q, k, v, scale, how, dtype):
    B, H, Sq, D = q.shape
    Skv = k.shape[2]
    o = torch.full_like(q, float("nan"))
    args = [q.data_ptr(), k.data_ptr(), v.data_ptr(), o.data_ptr(), B, H, Sq, Skv, D, scale,
            torch.cuda.current_stream().cuda_stream, 1 if dtype == "bf16" else 0,
            None, None, None, None]
    h = handle()
    if how == "static":
        rc = h.attn_fwd_split_static(*args)
    elif how == "no workspace":
        rc = h.attn_fwd_split(*args, None, 0)
    else:
        rc = h.attn_fwd_ex(*args)
    assert rc == 0, h.attn_last_error()
    return o


@pytest.mark.gpu
@pytest.mark.parametrize("case", CASES)
def test_tail_split(case):
    B, H, Sq, Skv, D, dtype = case
    print(f"case tail: B{B} H{H} Sq{Sq} Skv{Skv} D{D} {dtype}", flush=True)
    q, k, v = make_inputs(B, H, Sq, Skv, D, 1.0, 1.0, 700 + D)
    if dtype == "bf16":
        q, k, v = (t.to(torch.bfloat16) for t in (q, k, v))
    q, k, v = (t.to(DEV) for t in (q, k, v))
    scale = D ** -0.5
    out = gfx906_amd.attn(q, k, v, scale)
    plain = call(q, k, v, scale, "unsplit", dtype)
    assert torch.equal(call(q, k, v, scale, "static", dtype), out)
    assert torch.equal(call(q, k, v, scale, "no workspace", dtype), plain)
    r0 = first_split_row(B, H, Sq, D)
    flat, flat0 = out.reshape(-1, D), plain.reshape(-1, D)
    assert torch.equal(flat[:r0], flat0[:r0]) and not torch.equal(flat[r0:], flat0[r0:])
    # [B, S, H, D] views in and out: the same bits
    t = [x.transpose(1, 2).contiguous().transpose(1, 2) for x in (q, k, v)]
    o = torch.empty((B, Sq, H, D), dtype=q.dtype, device=DEV)
    gfx906_amd.attn(*t, scale, out=o.transpose(1, 2))
    assert torch.equal(o.transpose(1, 2), out)
    mult = 8 if dtype == "bf16" else 1
    heads = sorted({0, (r0 // Sq) % (B * H), (r0 // Sq + 1) % (B * H), B * H - 1})
    fold = [x.reshape(1, B * H, -1, D)[:, heads].cpu() for x in (q, k, v)]
    # (the last rows of each head: split ones of the tail's heads among them)
    rows = slice(max(0, Sq - 600), Sq)
    ref = sdpa_math_fp32(fold[0][:, :, rows].contiguous(), fold[1], fold[2], scale)
    got = out.reshape(1, B * H, Sq, D)[:, heads][:, :, rows].float().cpu()
    mx, mn = error_stats(got, ref)
    print(f"  max-abs {mx:.3e} mean-abs {mn:.3e}", flush=True)
    assert mx <= MAX_ABS_TOL * mult and mn <= MEAN_ABS_TOL * mult


@pytest.mark.gpu
def test_captured_c_entry_runs_the_tail_unsplit():
    B, H, Sq, Skv, D, dtype = CASES[0]
    print(f"case tail in a graph: B{B} H{H} Sq{Sq} Skv{Skv} D{D}", flush=True)
    q, k, v = (t.to(DEV) for t in make_inputs(B, H, Sq, Skv, D, 1.0, 1.0, 9))
    scale = D ** -0.5
    eager, plain = gfx906_amd.attn(q, k, v, scale), call(q, k, v, scale, "unsplit", dtype)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        op = gfx906_amd.attn(q, k, v, scale)
        static = call(q, k, v, scale, "static", dtype)
    for _ in range(3):
        op.zero_()
        static.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(op, eager) and torch.equal(static, plain)
        gfx906_amd.attn(q, k, v, -scale)  # eager work between replays

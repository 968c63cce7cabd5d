"""Head dims up to 48 on the ring kernel: QK^T and PV over 32 or 48 dims only.

Every such head dim, tile max on and off, split and unsplit, ragged counts,
fp16 and bf16, held to the bars against SDPA MATH in fp32 (rounding-aware),
and a split tail of a grid past 512 units. Each case prints its parameters
first.
"""

import pytest
import torch

import gfx906_amd
from oracle.attention import make_inputs, sdpa_math_fp32, within_rounded_tolerance

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.mark.parametrize("nsplit", ["1", "3"])
@pytest.mark.parametrize("tile_max", ["0", "1"])
@pytest.mark.parametrize("D", [8, 16, 24, 32, 40, 48, 56])
def test_narrow_heads(monkeypatch, D, tile_max, nsplit):
    monkeypatch.setenv("GFX906_AMD_ATTN_KVRES", "0")
    monkeypatch.setenv("GFX906_AMD_ATTN_TILEMAX", tile_max)
    monkeypatch.setenv("GFX906_AMD_ATTN_NSPLIT", nsplit)
    for n, (B, H, Sq, Skv) in enumerate([(1, 1, 1, 1), (2, 3, 257, 130), (1, 2, 300, 1100)]):
        for bf16 in (False, True):
            print(f"case narrow: B{B} H{H} Sq{Sq} Skv{Skv} D{D} bf16 {bf16} tile max {tile_max} "
                  f"n{nsplit}", flush=True)
            q, k, v = make_inputs(B, H, Sq, Skv, D, 1.5, 1.0, 60 + n)
            if bf16:
                q, k, v = (t.to(torch.bfloat16) for t in (q, k, v))
            out = gfx906_amd.attn(q.to(DEV), k.to(DEV), v.to(DEV), D ** -0.5)
            ok, mx, mn = within_rounded_tolerance(out.float().cpu(), sdpa_math_fp32(q, k, v, D ** -0.5),
                                                  *(("bf16", 8.0) if bf16 else ("fp16", 1.0)))
            assert ok, (mx, mn)


@pytest.mark.parametrize("D", [16, 48])
def test_narrow_split_tail(D):
    B, H, Sq, Skv = 3, 172, 100, 1100  # 516 units, the last 4 split
    print(f"case narrow tail: D{D}", flush=True)
    assert gfx906_amd.capi().attn_split_workspace_bytes(B, H, Sq, Skv, D) > 0
    q, k, v = make_inputs(B, H, Sq, Skv, D, 1.0, 1.0, 61)
    out = gfx906_amd.attn(q.to(DEV), k.to(DEV), v.to(DEV), D ** -0.5).float().cpu()
    for b, hs in ((0, slice(0, 4)), (2, slice(164, 172))):
        ref = sdpa_math_fp32(*(t[b:b + 1, hs].contiguous() for t in (q, k, v)), D ** -0.5)
        ok, mx, mn = within_rounded_tolerance(out[b:b + 1, hs], ref, "fp16")
        assert ok, (b, mx, mn)

"""Scores of -inf and scores below every fp16 one.

A key whose score is -inf weighs nothing, whatever the head dim (padded ones
among them), and wherever such keys lie: in the first tile, in a whole key
range, between finite ones. A row of nothing else is NaN (0 for D = 128), in
every kernel and split alike. Finite scores of any size that fp32 holds count.
Outputs are held to the bars against SDPA MATH in fp32 over the keys that
count. Each case prints its parameters first.
"""

import math

import pytest
import torch

import gfx906_amd
from oracle.attention import make_inputs, sdpa_math_fp32, within_rounded_tolerance

pytestmark = pytest.mark.gpu
DEV = "cuda"
# Kernel and split forced through the environment. res: the K/V-resident kernel.
FORMS = {
    "default": {},
    "rows": {"ROWS": "1"},
    "rows x 3": {"ROWS": "3", "NSPLIT": "3"},
    "ring, tile max": {"ROWS": "0", "NSPLIT": "1", "KVRES": "0", "TILEMAX": "1"},
    "ring, block max": {"ROWS": "0", "NSPLIT": "1", "KVRES": "0", "TILEMAX": "0"},
    "ring x 3": {"ROWS": "0", "NSPLIT": "3", "KVRES": "0", "TILEMAX": "1"},
    "ring x 3, block max": {"ROWS": "0", "NSPLIT": "3", "KVRES": "0", "TILEMAX": "0"},
    "res": {"ROWS": "0", "NSPLIT": "1", "KVRES": "1"},
}


def force(monkeypatch, form):
    for name, value in FORMS[form].items():
        monkeypatch.setenv("GFX906_AMD_ATTN_" + name, value)


def near(out, ref, bf16, what):
    fmt, mult = ("bf16", 8.0) if bf16 else ("fp16", 1.0)
    ok, mx, mn = within_rounded_tolerance(out.float().cpu(), ref, fmt, mult)
    assert ok, (what, mx, mn)


def masked_inputs(H, Sq, Skv, D, spans, seed, bf16=False, amp=1.0):
    """q > 0, keys -inf outside `spans`; keep marks the keys that count."""
    q, k, v = make_inputs(1, H, Sq, Skv, D, amp, 1.0, seed)
    if bf16:
        q, k, v = (t.to(torch.bfloat16) for t in (q, k, v))
    q = q.abs() + 0.01
    keep = torch.zeros(Skv, dtype=torch.bool)
    for a, b in spans:
        keep[a:b] = True
    k[:, :, ~keep] = float("-inf")
    return q, k, v, keep


def check(q, k, v, keep, scale, bf16, what, run=gfx906_amd.attn):
    ref = sdpa_math_fp32(q, k[:, :, keep], v[:, :, keep], scale)
    near(run(q.to(DEV), k.to(DEV), v.to(DEV), scale), ref, bf16, what)


@pytest.mark.parametrize("form", list(FORMS))
@pytest.mark.parametrize("D", [8, 16, 24, 32, 40, 48, 56])
def test_padded_head_dims(monkeypatch, D, form):
    force(monkeypatch, form)
    print(f"case masked: padded D{D} {form}", flush=True)
    for bf16 in (False, True):
        q, k, v, keep = masked_inputs(2, 70, 600, D, ((0, 70), (300, 310), (599, 600)), D, bf16)
        check(q, k, v, keep, 0.1, bf16, form)


# Finite keys past the first tiles only, in the middle range of three, in the last.
SPANS = [((300, 310),), ((590, 600),), ((70, 90), (599, 600))]


@pytest.mark.parametrize("form", list(FORMS))
@pytest.mark.parametrize("D", [40, 64, 128])
def test_first_tiles_and_whole_ranges(monkeypatch, D, form):
    force(monkeypatch, form)
    print(f"case masked: first tiles D{D} {form}", flush=True)
    for n, spans in enumerate(SPANS):
        for bf16 in (False, True):
            q, k, v, keep = masked_inputs(2, 70, 600, D, spans, D + n, bf16)
            check(q, k, v, keep, 0.1, bf16, (form, spans))
    out = gfx906_amd.attn(q.to(DEV), torch.full_like(k, float("-inf")).to(DEV), v.to(DEV), 0.1)
    assert bool((out == 0).all() if D == 128 else out.isnan().all())


@pytest.mark.parametrize("form", ["ring x 3", "ring x 3, block max", "rows x 3", "default"])
@pytest.mark.parametrize("D", [40, 64, 128])
def test_large_scales(monkeypatch, D, form):
    force(monkeypatch, form)
    print(f"case masked: scale 60 D{D} {form}", flush=True)
    q, k, v, keep = masked_inputs(2, 70, 600, D, ((0, 70), (300, 310)), D, amp=0.05)
    check(q, k, v, keep, 60.0, False, form)


@pytest.mark.parametrize("form", list(FORMS))
@pytest.mark.parametrize("D", [40, 64, 128])
def test_scores_far_below_zero(monkeypatch, D, form):
    """bf16 scores of -1.5e37 and less: the largest takes all the weight. (The
    scale makes scores in log2 units exact, as any rounding of theirs is far
    above 1.)"""
    force(monkeypatch, form)
    print(f"case masked: far scores D{D} {form}", flush=True)
    far_scores(D, gfx906_amd.attn)


def far_scores(D, run):
    q = torch.zeros(1, 2, 70, D, dtype=torch.bfloat16)
    k = torch.zeros(1, 2, 600, D, dtype=torch.bfloat16)
    v = make_inputs(1, 2, 70, 600, D, 1.0, 1.0, 3)[2].to(torch.bfloat16)
    q[..., 0] = 1e18
    k[..., 0] = -2e19
    for best in (5, 333, 599):
        kb = k.clone()
        kb[:, :, best, 0] = -1.5e19
        out = run(q.to(DEV), kb.to(DEV), v.to(DEV), math.log(2.0)).cpu()
        assert torch.equal(out, v[:, :, best:best + 1].expand_as(out)), best


# D = 512 ---------------------------------------------------------------------------


def tokens(x):
    return x.transpose(2, 3).contiguous().transpose(2, 3)


def token_attn(q, k, v, scale):
    return gfx906_amd.attn(tokens(q), tokens(k), tokens(v), scale, out=tokens(torch.zeros_like(q)))


D512 = {  # kernel by layout and override, key ranges
    "rows": (gfx906_amd.attn, {"NSPLIT": "1"}),
    "rows x 3": (gfx906_amd.attn, {"NSPLIT": "3"}),
    "tokens": (token_attn, {"NSPLIT": "1"}),
    "tokens x 3": (token_attn, {"NSPLIT": "3"}),
    "16 rows": (gfx906_amd.attn, {"NSPLIT": "1", "D512W": "0"}),
    "16 rows x 3": (gfx906_amd.attn, {"NSPLIT": "3", "D512W": "0"}),
}


@pytest.mark.parametrize("form", list(D512))
def test_d512(monkeypatch, form):
    run, env = D512[form]
    for name, value in env.items():
        monkeypatch.setenv("GFX906_AMD_ATTN_" + name, value)
    print(f"case masked: D512 {form}", flush=True)
    for n, spans in enumerate(SPANS + [((0, 40), (300, 310))]):
        for bf16 in (False, True):
            q, k, v, keep = masked_inputs(2, 70, 600, 512, spans, 512 + n, bf16)
            check(q, k, v, keep, 0.02, bf16, (form, spans), run)
    out = run(q.to(DEV), torch.full_like(k, float("-inf")).to(DEV), v.to(DEV), 0.02)
    assert bool(out.isnan().all())
    far_scores(512, run)


@pytest.mark.parametrize("layout", ["rows", "tokens"])
def test_d512_split_tail(layout):
    """A range of the tail without finite scores leaves its rows as they are unsplit."""
    H, Sq, Skv = 52, 640, 600  # 260 units of 128 rows, the last four split
    print(f"case masked: D512 tail, {layout}", flush=True)
    assert gfx906_amd.capi().attn_split_workspace_bytes(1, H, Sq, Skv, 512) > 0
    q, k, v, keep = masked_inputs(H, Sq, Skv, 512, ((0, 100),), 9)
    run = gfx906_amd.attn if layout == "rows" else token_attn
    got = run(q.to(DEV), k.to(DEV), v.to(DEV), 0.02)[:, -1:].cpu()
    ref = sdpa_math_fp32(q[:, -1:], k[:, -1:, keep], v[:, -1:, keep], 0.02)
    near(got, ref, False, layout)


@pytest.mark.parametrize("D", [40, 64, 128, 512])
def test_no_keys_are_zeros(D):
    """Skv = 0 is not a row of -inf scores: zeros."""
    print(f"case masked: no keys D{D}", flush=True)
    q, k, v = make_inputs(1, 2, 70, 8, D, 1.0, 1.0, 1)
    out = gfx906_amd.attn(q.to(DEV), k[:, :, :0].to(DEV), v[:, :, :0].to(DEV), 0.1)
    assert bool((out == 0).all())

"""Scores of -inf.

A key whose score is -inf weighs nothing, whatever the head dim (padded ones
among them). Outputs are held to the bars against SDPA MATH in fp32 over the
keys that count. Each case prints its parameters first.
"""

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

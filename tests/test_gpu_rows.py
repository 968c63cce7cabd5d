"""attn_fwd_rows: few query rows per workgroup, the keys shared out to its waves.

Query counts around a workgroup's 32 or 64 rows, key counts around a wave's
step, a round of the eight waves' steps and a split range (waves and ranges
without keys among them), for D = 8, 40, 64 and 128, with each row count and
split forced, and the ring kernel forced on the same shapes. Held to the bars
against SDPA MATH in fp32 (rounding-aware where the output format has no room
under them). Strided views, sharp rows, a negative scale, NaN and infinite
keys, and the default dispatch have cases of their own. Where a forced count
cannot run (its partial results would not fit the workspace of the ring
kernel's plan) the case is left out, and the results have to differ from the
ring kernel's somewhere: the kernel that is named is the one that runs. Each
prints its parameters first.
"""

import pytest
import torch

import gfx906_amd
from oracle.attention import MAX_ABS_TOL, make_inputs, sdpa_math_fp32, within_rounded_tolerance

pytestmark = pytest.mark.gpu
DEV = "cuda"
SHAPES = [  # B, H, Sq, Skv
    (1, 1, 1, 1), (1, 2, 15, 31), (1, 1, 31, 63), (2, 1, 32, 64), (1, 1, 33, 65), (1, 3, 64, 200),
    (1, 1, 65, 255), (1, 1, 100, 257), (1, 2, 63, 511), (2, 2, 7, 513), (1, 1, 129, 1100),
]


def near(out, ref, bf16, what):
    fmt, mult = ("bf16", 8.0) if bf16 else ("fp16", 1.0)
    ok, mx, mn = within_rounded_tolerance(out.float().cpu(), ref, fmt, mult)
    assert ok, (what, mx, mn)


def forms(Ds, rows):
    """(D, rows) pairs; D = 128 has no form of 64 rows."""
    return pytest.mark.parametrize("D,rows", [(D, r) for D in Ds for r in rows
                                              if not (D == 128 and "x64" in r)])


def force(monkeypatch, rows):
    monkeypatch.setenv("GFX906_AMD_ATTN_ROWS", rows)
    if "x" in rows or int(rows) > 1:  # a workspace for the ranges
        monkeypatch.setenv("GFX906_AMD_ATTN_NSPLIT", rows.split("x")[0])


def ranges(rows, B, H, Sq, Skv, D):
    """Key ranges that the few-rows kernel runs when `rows` is forced, 0 if it cannot."""
    step = 32 if D == 128 else 64
    steps = -(-Skv // step)
    n = -(-steps // -(-steps // min(int(rows.split("x")[0]), steps)))
    need = gfx906_amd.capi().attn_split_workspace_bytes(B, H, Sq, Skv, D)
    return n if n == 1 or n * B * H * Sq * (D + 2) * 4 + 16 <= need else 0


def ring(monkeypatch, q, k, v, scale):
    with monkeypatch.context() as m:
        m.setenv("GFX906_AMD_ATTN_ROWS", "0")
        return gfx906_amd.attn(q, k, v, scale)


@forms([8, 40, 64, 128], ["0", "1", "2", "5", "1x64", "3x64"])
def test_forced_rows_and_ranges(monkeypatch, D, rows):
    force(monkeypatch, rows)
    most, differs = 0, False
    for n, (B, H, Sq, Skv) in enumerate(SHAPES):
        run = ranges(rows, B, H, Sq, Skv, D) if rows != "0" else 1
        most = max(most, run)
        if run == 0:
            continue
        for bf16 in (False, True):
            print(f"case rows {rows}: B{B} H{H} Sq{Sq} Skv{Skv} D{D} bf16 {bf16}", flush=True)
            q, k, v = make_inputs(B, H, Sq, Skv, D, 1.0, 1.0, 900 + n)
            if bf16:
                q, k, v = (t.to(torch.bfloat16) for t in (q, k, v))
            scale = D ** -0.5 * (-1 if n % 3 == 0 else 1)
            dev = [t.to(DEV) for t in (q, k, v)]
            out = gfx906_amd.attn(*dev, scale)
            near(out, sdpa_math_fp32(q, k, v, scale), bf16, (rows, B, H, Sq, Skv, D, bf16))
            differs |= not torch.equal(out, ring(monkeypatch, *dev, scale))
    assert differs == (rows != "0")
    assert most == max(1, int(rows.split("x")[0]))  # the forced count ran somewhere


@forms([40, 64, 128], ["1", "1x64", "4"])
def test_layouts_give_the_same_bits(monkeypatch, D, rows):
    force(monkeypatch, rows)
    assert ranges(rows, 2, 3, 77, 700, D) > 0
    print(f"case rows {rows} layouts D{D}", flush=True)
    q, k, v = (t.to(DEV) for t in make_inputs(2, 3, 77, 700, D, 2.0, 1.0, 31))
    ref = gfx906_amd.attn(q, k, v, 0.2)
    near(ref, sdpa_math_fp32(q.cpu(), k.cpu(), v.cpu(), 0.2), False, "sharp rows")
    assert not torch.equal(ref, ring(monkeypatch, q, k, v, 0.2))
    t = [x.transpose(1, 2).contiguous().transpose(1, 2) for x in (q, k, v)]
    o = torch.full((2, 80, 3, D), 7.0, dtype=q.dtype, device=DEV)
    gfx906_amd.attn(*t, 0.2, out=o[:, :77].transpose(1, 2))
    assert torch.equal(o[:, :77].transpose(1, 2), ref) and bool((o[:, 77:] == 7.0).all())
    # keys shared by the heads (stride 0)
    ke, ve = k[:, :1].expand(2, 3, 700, D), v[:, :1].expand(2, 3, 700, D)
    assert torch.equal(gfx906_amd.attn(q, ke, ve, 0.2),
                       gfx906_amd.attn(q, ke.contiguous(), ve.contiguous(), 0.2))


@forms([40, 64, 128], ["1", "1x64", "3"])
def test_special_values(monkeypatch, D, rows):
    """A NaN query reaches its own row, a NaN key or value every row; a step of
    keys far below the others adds nothing."""
    force(monkeypatch, rows)
    assert ranges(rows, 1, 2, 50, 600, D) > 0
    print(f"case rows {rows} special D{D}", flush=True)
    base = make_inputs(1, 2, 50, 600, D, 1.0, 1.0, 77)
    for which in range(3):
        q, k, v = (t.clone() for t in base)
        (q, k, v)[which][0, 1, 21, 3] = float("nan")
        got = gfx906_amd.attn(q.to(DEV), k.to(DEV), v.to(DEV), 0.1).float().cpu()
        ref = sdpa_math_fp32(q, k, v, 0.1)
        assert torch.equal(got.isnan(), ref.isnan()), which
        keep = ~ref.isnan()
        assert (got[keep] - ref[keep]).abs().max() <= MAX_ABS_TOL
    q, k, v = (t.clone() for t in base)
    q[...] = q.abs() + 0.01
    k[0, :, 1:] = k[0, :, 1:].clamp(-1, 1)
    k[0, :, 64:128] = -60000.0  # a whole step of one wave far below the others
    got = gfx906_amd.attn(q.to(DEV), k.to(DEV), v.to(DEV), 0.1).float().cpu()
    assert (got - sdpa_math_fp32(q, k, v, 0.1)).abs().max() <= MAX_ABS_TOL


@pytest.mark.parametrize("D,form", [
    (D, form) for D in (40, 64, 128)
    for form in ("default", "rows1", "rows1x64", "rows3", "ring1", "ring4", "tail")
    if (D, form) != (128, "rows1x64")])
def test_infinite_keys(monkeypatch, D, form):
    """Keys whose scores are all -inf weigh nothing, also where they are all
    that a wave's first step, a whole key range or a split tail's range sees;
    rows of nothing else are NaN (0 for D = 128)."""
    if form.startswith("rows"):
        monkeypatch.setenv("GFX906_AMD_ATTN_ROWS", form[4:])
        monkeypatch.setenv("GFX906_AMD_ATTN_NSPLIT", form[4])
    elif form.startswith("ring"):
        monkeypatch.setenv("GFX906_AMD_ATTN_ROWS", "0")
        monkeypatch.setenv("GFX906_AMD_ATTN_NSPLIT", form[4])
    # (tail: 272 or 527 query tiles, a little past the workgroup slots)
    H, Sq, Skv = (16, 4250, 1400) if D == 128 else (17, 7700, 1400)
    if form != "tail":
        H, Sq, Skv = 2, 70, 1100
    print(f"case {form} infinite keys D{D}", flush=True)
    q, k, v = make_inputs(1, H, Sq, Skv, D, 1.0, 1.0, 78)
    q = q.abs() + 0.01  # a key of -inf then scores -inf in every row
    keep = torch.zeros(Skv, dtype=torch.bool)
    keep[:70] = keep[640:660] = True
    k[:, :, ~keep] = float("-inf")
    got = gfx906_amd.attn(q.to(DEV), k.to(DEV), v.to(DEV), 0.1)[:, -1:, -100:].cpu()
    near(got, sdpa_math_fp32(q[:, -1:, -100:], k[:, -1:, keep], v[:, -1:, keep], 0.1), False, form)
    k[...] = float("-inf")
    got = gfx906_amd.attn(q.to(DEV), k.to(DEV), v.to(DEV), 0.1)
    assert bool((got == 0).all() if D == 128 else got.isnan().all())


def test_default_dispatch(monkeypatch):
    """Small grids take the kernel by default, in every entry point alike."""
    q, k, v = (t.to(DEV) for t in make_inputs(1, 4, 300, 300, 64, 1.0, 1.0, 5))
    print("case rows default dispatch", flush=True)
    lib = gfx906_amd.capi()

    def capi(fn, *extra):
        o = torch.empty_like(q)
        rc = fn(q.data_ptr(), k.data_ptr(), v.data_ptr(), o.data_ptr(), 1, 4, 300, 300, 64, 0.125,
                torch.cuda.current_stream().cuda_stream, *extra)
        assert rc == 0, lib.attn_last_error()
        return o

    out = gfx906_amd.attn(q, k, v, 0.125)
    strides = (0, None, None, None, None)
    assert torch.equal(out, capi(lib.attn_fwd)) and torch.equal(out, capi(lib.attn_fwd_ex, *strides))
    monkeypatch.setenv("GFX906_AMD_ATTN_ROWS", "1")
    assert torch.equal(out, gfx906_amd.attn(q, k, v, 0.125))
    monkeypatch.setenv("GFX906_AMD_ATTN_ROWS", "0")
    assert not torch.equal(out, gfx906_amd.attn(q, k, v, 0.125))

"""attn_fwd_tok512: token-contiguous K and V, D = 512, 32 query rows per wave.

Query counts around a wave's 32 rows, an 8-token store and a 128-row unit, key
counts around a 32-key tile, with q and o each token-contiguous (q read as
Q^T tiles for whole 8-token chunks, o stored as runs of tokens) or row-contiguous (element by element), split
and unsplit (forced counts), several heads and batches, fp16 and bf16, and a
negative scale. Held to the bars against SDPA MATH in fp32 and to within
rounding of the row-contiguous kernel; elements around o stay untouched. Each
case prints its parameters first.
"""

import ctypes

import pytest
import torch

import gfx906_amd
from oracle.attention import MAX_ABS_TOL, MEAN_ABS_TOL, error_stats, sdpa_math_fp32

DEV = "cuda"
SHAPES = [  # B, H, Sq, Skv
    (1, 1, 1, 8), (1, 1, 7, 24), (1, 2, 31, 32), (2, 1, 33, 40), (1, 1, 127, 64),
    (1, 1, 129, 200), (2, 2, 250, 96), (1, 1, 300, 1032),
    (1, 1, 8, 64), (1, 2, 24, 40), (2, 1, 40, 104), (1, 1, 136, 64), (1, 2, 264, 264),
]


def tokens(x, pad=0):
    """[B, H, S, D] seen through a [B, H, D, S + pad] buffer (rows of a multiple
    of 8 tokens), NaN outside."""
    B, H, S, D = x.shape
    row = -(-S // 8) * 8 + pad
    buf = torch.full((B, H, D, row), float("nan"), dtype=x.dtype, device=x.device)
    buf[..., :S] = x.transpose(2, 3)
    return buf, buf[..., :S].transpose(2, 3)


def st(t):
    return (ctypes.c_longlong * 4)(*t.stride())


@pytest.mark.gpu
@pytest.mark.parametrize("nsplit", [1, 3])
@pytest.mark.parametrize("q_tok,o_tok", [(True, True), (True, False), (False, True)])
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("B,H,Sq,Skv", SHAPES)
def test_tok512(monkeypatch, B, H, Sq, Skv, dtype, q_tok, o_tok, nsplit):
    print(f"case tok512: B{B} H{H} Sq{Sq} Skv{Skv} {dtype} q_tok {q_tok} o_tok {o_tok} n{nsplit}",
          flush=True)
    if nsplit:
        monkeypatch.setenv("GFX906_AMD_ATTN_NSPLIT", str(nsplit))
    g = torch.Generator().manual_seed(Sq * 1000 + Skv)
    q, k, v = ((torch.randn(B, H, s, 512, generator=g) * m).to(dtype).to(DEV)
               for s, m in ((Sq, 1.0), (Skv, 1.0), (Skv, 1.0)))
    scale = -(512 ** -0.5)
    ref = gfx906_amd.attn(q, k, v, scale)
    (_, kt), (_, vt) = tokens(k, 8), tokens(v)
    qt = tokens(q)[1] if q_tok else q
    obuf, o = tokens(torch.zeros_like(q), 8) if o_tok else (None, torch.zeros_like(q))
    lib = gfx906_amd.capi()
    need = lib.attn_split_workspace_bytes(B, H, Sq, Skv, 512)
    ws = torch.empty(max(need, 16), dtype=torch.uint8, device=DEV)
    rc = lib.attn_fwd_split(qt.data_ptr(), kt.data_ptr(), vt.data_ptr(), o.data_ptr(), B, H, Sq,
                            Skv, 512, scale, torch.cuda.current_stream().cuda_stream,
                            0 if dtype == torch.float16 else 1, st(qt), st(kt), st(vt), st(o),
                            ws.data_ptr(), need)
    assert rc == 0, lib.attn_last_error()
    torch.cuda.synchronize()
    mult = 1 if dtype == torch.float16 else 8
    assert (o.float() - ref.float()).abs().max().item() <= MAX_ABS_TOL * mult
    exact = sdpa_math_fp32(q.cpu(), k.cpu(), v.cpu(), scale)
    mx, mn = error_stats(o.float().cpu(), exact)
    assert mx <= MAX_ABS_TOL * mult and mn <= MEAN_ABS_TOL * mult, (mx, mn)
    if o_tok:
        assert bool(obuf[..., Sq:].isnan().all())


@pytest.mark.gpu
def test_tok512_whole_units_and_a_split_tail(monkeypatch):
    # 65 heads of 4 units: 256 unsplit units, the last head's split and merged
    assert 0 < gfx906_amd.capi().attn_split_workspace_bytes(1, 65, 500, 1032, 512) < 65 << 20
    test_tok512(monkeypatch, 1, 65, 500, 1032, torch.float16, True, True, None)


@pytest.mark.gpu
@pytest.mark.parametrize("wide", ["", "0"])
@pytest.mark.parametrize("nsplit", [1, 3, None])
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("B,H,Sq,Skv", [(1, 1, 8, 8), (2, 1, 56, 72), (1, 2, 64, 128),
                                        (1, 1, 136, 200), (2, 2, 264, 1032), (1, 65, 504, 1032),
                                        (1, 1, 1, 1), (2, 1, 33, 65), (1, 2, 127, 300),
                                        (2, 1, 250, 515), (1, 65, 500, 1035)])
def test_row_copies(monkeypatch, B, H, Sq, Skv, dtype, nsplit, wide):
    """attn_fwd_split_copied: the row-contiguous kernel's bits, stored by tokens
    (also with GFX906_AMD_ATTN_D512W=0, whose kernel stores rows only)."""
    print(f"case row copies: B{B} H{H} Sq{Sq} Skv{Skv} {dtype} n{nsplit} wide {wide!r}", flush=True)
    if nsplit:
        monkeypatch.setenv("GFX906_AMD_ATTN_NSPLIT", str(nsplit))
    g = torch.Generator().manual_seed(Sq + Skv)
    q, k, v = (torch.randn(B, H, s, 512, generator=g).to(dtype).to(DEV) for s in (Sq, Skv, Skv))
    ref = gfx906_amd.attn(q, k, v, 0.04)
    if wide:
        monkeypatch.setenv("GFX906_AMD_ATTN_D512W", wide)
    odd = 0 if Sq % 8 == 0 else 1  # odd counts: rows of any alignment
    (_, qt), (_, kt), (_, vt) = tokens(q, odd), tokens(k, 8), tokens(v, 3 * odd)
    obuf, o = tokens(torch.zeros_like(q), 16 - odd)
    lib = gfx906_amd.capi()
    # (the plan without the override, whose own kernel runs no split tail)
    need = max(lib.attn_split_workspace_bytes(B, H, Sq, Skv, 512), 64 << 20)
    n = lib.attn_row_copies_bytes(B, H, Sq, Skv, 512)
    assert n == B * H * (Sq + 2 * Skv) * 1024
    ws = torch.empty(need, dtype=torch.uint8, device=DEV)
    copies = torch.full((n + 64,), 7, dtype=torch.uint8, device=DEV)
    rc = lib.attn_fwd_split_copied(qt.data_ptr(), kt.data_ptr(), vt.data_ptr(), o.data_ptr(), B, H,
                                   Sq, Skv, 512, 0.04, torch.cuda.current_stream().cuda_stream,
                                   0 if dtype == torch.float16 else 1, st(qt), st(kt), st(vt), st(o),
                                   ws.data_ptr(), need, copies.data_ptr(), n)
    assert rc == 0, lib.attn_last_error()
    torch.cuda.synchronize()
    assert torch.equal(o, ref) and bool(obuf[..., Sq:].isnan().all())
    assert bool((copies[n:] == 7).all())


def test_row_copies_rejects():
    # (needs no GPU: refused before any HIP call)
    lib = gfx906_amd.capi()
    p = ctypes.c_void_p(0x10000)
    tok = (ctypes.c_longlong * 4)(512 * 64, 512 * 64, 1, 64)
    rows = (ctypes.c_longlong * 4)(512 * 64, 512 * 64, 512, 1)
    need = lib.attn_split_workspace_bytes(1, 1, 64, 64, 512)
    n = lib.attn_row_copies_bytes(1, 1, 64, 64, 512)

    def call(sq=64, skv=64, q=tok, k=tok, v=tok, o=tok, copies=p, nbytes=n, d=512):
        rc = lib.attn_fwd_split_copied(p, p, p, p, 1, 1, sq, skv, d, 0.04, None, 0, q, k, v, o, p,
                                       need, copies, nbytes)
        return rc, lib.attn_last_error()

    for kw, msg in ((dict(copies=None), b"missing"), (dict(nbytes=n - 1), b"smaller"),
                    (dict(copies=ctypes.c_void_p(0x10008)), b"misaligned"),
                    (dict(q=rows), b"token-contiguous"), (dict(o=rows), b"token-contiguous"),
                    (dict(k=rows, v=rows), b"token-contiguous"), (dict(skv=0), b"need queries"),
                    (dict(d=64), b"token-contiguous"),
                    (dict(o=(ctypes.c_longlong * 4)(64, 64, 1, 2)), b"overlap")):
        rc, err = call(**kw)
        assert rc == 1 and msg in err, (kw, err)
    assert lib.attn_row_copies_bytes(1, 1, 64, 64, 128) == 0


@pytest.mark.gpu
@pytest.mark.parametrize("Sq,Skv", [(1, 6408), (1, 100), (1, 64), (40, 1), (1, 1)])
def test_one_token(Sq, Skv):
    """The op on token-strided tensors of one query or one key (whose token
    stride says nothing), past the in-place limit, at a count that is no
    multiple of 8, and in place."""
    print(f"case tok512: one token, Sq{Sq} Skv{Skv}", flush=True)
    g = torch.Generator().manual_seed(Sq + Skv)
    q, k, v = (torch.randn(1, 2, s, 512, generator=g).half().to(DEV) for s in (Sq, Skv, Skv))
    obuf, o = tokens(torch.zeros_like(q), 8)
    got = gfx906_amd.attn(tokens(q)[1], tokens(k)[1], tokens(v)[1], 0.04, out=o)
    mx, mn = error_stats(got.float().cpu(), sdpa_math_fp32(q.cpu(), k.cpu(), v.cpu(), 0.04))
    assert mx <= MAX_ABS_TOL and mn <= MEAN_ABS_TOL, (mx, mn)
    assert bool(obuf[..., Sq:].isnan().all())

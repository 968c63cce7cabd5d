"""Performance cases of the MI355X attention forward and conv3d backend.

Each case is one call that a program using this package makes: the attention
operator (``gfx906_amd.attn``), the host hooks (``attention_hooks.dit`` for
DiT layers, ``attention_hooks.vae_attn`` for a VAE's mid block) or the conv3d
backend (``kitchen.fp16_conv3d``, ``kitchen.fp16_conv3d_out``).

``listed()`` returns the named cases and ``draw(rng)`` one more of the same
ranges. ``prepare`` makes a case's inputs on the GPU, ``run`` makes the call,
``work`` counts what it cannot do without, ``exact`` gives the result in 64
bits and ``tolerance`` the error another correct implementation may show.
"""

from __future__ import annotations

import math

import torch

import gfx906_amd
from gfx906_amd import attention_hooks, kitchen

DTYPES = {"fp16": torch.float16, "bf16": torch.bfloat16}
CL = torch.channels_last_3d


def _attn(B, H, Sq, Skv, D, dtype="fp16", qk=1.0, **name):
    """gfx906_amd.attn on contiguous [B, H, S, D]; q, k ~ qk * N(0, 1), v ~ N(0, 1)."""
    return dict(op="attn", B=B, H=H, Sq=Sq, Skv=Skv, D=D, dtype=dtype, qk=qk, **name)


def _dit(B, H, S, D, dtype="bf16", **name):
    """A DiT layer's self-attention through the container hook: q, k, v are
    [B, S, H, D] projections viewed as [B, H, S, D]; the result is [B, S, H*D]."""
    return dict(op="dit", B=B, H=H, Sq=S, Skv=S, D=D, dtype=dtype, qk=1.0, **name)


def _vae(b, h, w, dtype="fp16", **name):
    """A VAE mid block's attention: [b, 512, h, w] activations, one 512-wide head."""
    return dict(op="vae", B=b, h=h, w=w, dtype=dtype, **name)


def _conv(x, k, window, stride=(1, 1, 1), bias=True, res=False, out=False, **name):
    """VALID conv3d of channels_last_3d x (n, c, d, h, w), filter k x c x window;
    `out`: written into a tensor the caller holds (fp16_conv3d_out)."""
    n, c, d, h, w = x
    t, r, s = window
    return dict(op="conv", n=n, c=c, d=d, h=h, w=w, k=k, t=t, r=r, s=s, sd=stride[0],
                sh=stride[1], sw=stride[2], bias=bias, res=res, out=out, **name)


def listed():
    return [
        # The smallest call: one short head (a test-sized model, the first
        # attention of a tiny latent). Launches and host time count.
        _attn(1, 1, 1024, 1024, 64, name="small_d64"),
        # A DiT block on a video latent with a token count that is no multiple
        # of anything, in bf16 through the host hook: the layer the hook
        # serves dozens of times per denoising step.
        _dit(1, 16, 4250, 128, name="dit_bf16_ragged"),
        # The benchmark's headline: a long DiT sequence.
        _attn(1, 16, 16384, 16384, 128, name="long_d128"),
        # Cross-attention of a large query set to 512 keys, sharp rows.
        _attn(2, 24, 8192, 512, 64, qk=2.0, name="cross_d64_sharp"),
        # Cross-attention to a 77-token text prompt (a U-Net's 64x64 level,
        # both guidance halves in one batch).
        _attn(2, 16, 4096, 77, 64, name="text_cross_d64"),
        # Self-attention at that level with the 40-wide heads U-Nets use,
        # which are padded to the kernel's 64.
        _attn(2, 8, 4096, 4096, 40, name="unet_d40"),
        # The longest sequence of the benchmark's configurations.
        _attn(1, 8, 131072, 131072, 64, name="longest_d64"),
        # VAE mid block on a 512x512 image's 64x64 latent.
        _vae(1, 64, 64, name="vae_64x64"),
        # VAE mid block on a 1280x720 frame's 90x160 latent, bf16.
        _vae(1, 90, 160, dtype="bf16", name="vae_90x160_bf16"),
        # VAE decoder residual layer on video (the conv benchmark's layer).
        _conv((1, 512, 8, 64, 64), 512, (3, 3, 3), name="conv_decode_512"),
        # The same layer on a small latent (34x34 padded), with the block's
        # residual added in the epilogue: few output tiles.
        _conv((1, 512, 4, 34, 34), 512, (3, 3, 3), res=True, name="conv_latent_512_res"),
        # Encoder downsampling layer: 128 channels, spatial stride 2, odd
        # input size, into the caller's buffer.
        _conv((1, 128, 6, 257, 257), 128, (3, 3, 3), (1, 2, 2), out=True,
              name="conv_encode_stride2"),
    ]


def _log_int(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def _flops(case):
    return work(case)["flops"]


def draw(rng):
    """One more case of the listed ranges, without a name."""
    while True:
        kind = rng.choice(["self", "self", "cross", "few", "dit", "vae", "conv", "conv", "conv"])
        dtype = rng.choice(["fp16", "fp16", "bf16"])
        narrow = rng.choice([8, 16, 24, 32, 40, 48, 56])
        if kind == "self":  # from a short head to long sequences, any head dim class
            D = rng.choice([64, 64, 128, 128, narrow])
            S = _log_int(rng, 64, 20000)
            case = _attn(rng.choice([1, 1, 2]), _log_int(rng, 1, 24), S, S, D, dtype)
        elif kind == "cross":  # text and context cross-attention
            D = rng.choice([64, 64, 128, narrow])
            case = _attn(rng.choice([1, 2]), _log_int(rng, 4, 24), _log_int(rng, 64, 16384),
                         _log_int(rng, 1, 1024), D, dtype, qk=rng.choice([1.0, 2.0]))
        elif kind == "few":  # a few query rows against a long key range
            case = _attn(rng.choice([1, 2]), _log_int(rng, 1, 16), _log_int(rng, 1, 16),
                         _log_int(rng, 1024, 100000), rng.choice([64, 128]), dtype)
        elif kind == "dit":
            case = _dit(rng.choice([1, 1, 2]), rng.choice([8, 12, 16, 20, 24]),
                        _log_int(rng, 256, 16384), rng.choice([64, 128, 128]), dtype)
        elif kind == "vae":
            case = _vae(1, _log_int(rng, 16, 128), _log_int(rng, 16, 160), dtype)
        else:
            layer = rng.choice(["res", "res", "res", "shortcut", "in", "down"])
            c = rng.choice([64, 96, 128, 192, 256, 384, 512])
            d, h, w = rng.randint(1, 8), _log_int(rng, 16, 256), _log_int(rng, 16, 256)
            if layer == "res":  # 3x3x3 layer of a residual block, input already padded
                case = _conv((1, c, d + 2, h + 2, w + 2), c, (3, 3, 3), res=rng.random() < 0.5)
            elif layer == "shortcut":  # 1x1x1 change of channels
                case = _conv((1, c, d, h, w), rng.choice([64, 128, 256, 512]), (1, 1, 1))
            elif layer == "in":  # latent or pixel channels to the first feature width
                case = _conv((1, rng.choice([8, 16, 32]), d + 2, h + 2, w + 2), c, (3, 3, 3))
            else:  # downsampling, space or space and time
                st = rng.choice([(1, 2, 2), (2, 2, 2)])
                win = (3, 3, 3) if st[0] == 2 else rng.choice([(3, 3, 3), (1, 3, 3)])
                case = _conv((1, c, d + 2, h + 1, w + 1), c, win, st, out=rng.random() < 0.5)
        if _flops(case) <= 2.5e12:
            return case


# -- inputs ------------------------------------------------------------------------------


class _Held:
    """The container the host hands its tensors over in: peek() looks, take() gives."""

    def __init__(self, t):
        self.t = t

    def peek(self):
        return self.t

    def take(self):
        t, self.t = self.t, None
        return t


def _no_fallback(*args, **kwargs):
    raise RuntimeError("the kernel declined the call")


def _conv_out_shape(c):
    return (c["n"], c["k"], (c["d"] - c["t"]) // c["sd"] + 1, (c["h"] - c["r"]) // c["sh"] + 1,
            (c["w"] - c["s"]) // c["sw"] + 1)


def _inputs(case, seed):
    """The case's input tensors, on the GPU, from the seed alone."""
    g = torch.Generator(device="cuda").manual_seed(seed)

    def normal(shape, dtype, mult=1.0):
        return (torch.randn(shape, generator=g, device="cuda") * mult).to(dtype)

    op = case["op"]
    if op == "attn":
        dt, qk = DTYPES[case["dtype"]], case["qk"]
        lead = (case["B"], case["H"])
        q = normal((*lead, case["Sq"], case["D"]), dt, qk)
        k = normal((*lead, case["Skv"], case["D"]), dt, qk)
        return q, k, normal((*lead, case["Skv"], case["D"]), dt)
    if op == "dit":
        dt = DTYPES[case["dtype"]]
        shape = (case["B"], case["Sq"], case["H"], case["D"])
        return tuple(normal(shape, dt).transpose(1, 2) for _ in range(3))
    if op == "vae":
        dt = DTYPES[case["dtype"]]
        return tuple(normal((case["B"], 512, case["h"], case["w"]), dt) for _ in range(3))
    half = torch.float16
    c = case
    taps = c["t"] * c["r"] * c["s"]
    x = normal((c["n"], c["c"], c["d"], c["h"], c["w"]), half).contiguous(memory_format=CL)
    w = normal((c["k"], c["c"], c["t"], c["r"], c["s"]), half, (c["c"] * taps) ** -0.5)
    b = normal((c["k"],), half) if c["bias"] else None
    res = normal(_conv_out_shape(c), half).contiguous(memory_format=CL) if c["res"] else None
    return x, w.contiguous(memory_format=CL), b, res


def prepare(case, seed):
    state = {"op": case["op"], "in": _inputs(case, seed)}
    if case["op"] == "attn":
        state["scale"] = case["D"] ** -0.5
    elif case["op"] == "dit":
        state["heads"] = case["H"]
    elif case["op"] == "conv":
        state["stride"] = [case["sd"], case["sh"], case["sw"]]
        if case["out"]:
            state["out"] = torch.empty(_conv_out_shape(case), dtype=torch.float16, device="cuda",
                                       memory_format=CL)
    return state


def run(state):
    op = state["op"]
    if op == "attn":
        q, k, v = state["in"]
        return gfx906_amd.attn(q, k, v, state["scale"])
    if op == "dit":
        q, k, v = state["in"]
        return attention_hooks.dit(_Held(q), _Held(k), _Held(v), state["heads"],
                                   skip_reshape=True)
    if op == "vae":
        q, k, v = state["in"]
        return attention_hooks.vae_attn(q, k, v, _no_fallback)
    x, w, b, res = state["in"]
    if "out" in state:
        kitchen.fp16_conv3d_out(x, w, b, res, state["stride"], state["out"])
        return state["out"]
    return kitchen.fp16_conv3d(x, w, b, res, state["stride"])


# -- work, results, tolerances -----------------------------------------------------------


def work(case):
    """Operations of the two products (or of the convolution) and the bytes of
    every input read once and the output written once, 2 bytes an element."""
    c = case
    if c["op"] == "conv":
        n, k, z, p, q = _conv_out_shape(c)
        m, taps = n * z * p * q, c["t"] * c["r"] * c["s"]
        elems = (c["n"] * c["c"] * c["d"] * c["h"] * c["w"] + k * c["c"] * taps + m * k
                 + (k if c["bias"] else 0) + (m * k if c["res"] else 0))
        return {"bytes": 2 * elems, "flops": 2 * m * k * c["c"] * taps}
    if c["op"] == "vae":
        H, D = 1, 512
        Sq = Skv = c["h"] * c["w"]
    else:
        H, D, Sq, Skv = c["H"], c["D"], c["Sq"], c["Skv"]
    bh = c["B"] * H
    return {"bytes": 4 * bh * (Sq + Skv) * D, "flops": 4 * bh * Sq * Skv * D}


def _exact_attention(q, k, v, scale):
    """softmax(scale q k^T) v in float64 per head and block of query rows."""
    B, H, Sq, D = q.shape
    out = torch.empty((B, H, Sq, D), dtype=torch.float64, device=q.device)
    rows = max(1, min(Sq, (1 << 28) // k.shape[2]))
    for b in range(B):
        for h in range(H):
            kt = k[b, h].double().t().contiguous()
            vd = v[b, h].double()
            for r in range(0, Sq, rows):
                s = (q[b, h, r:r + rows].double() * scale) @ kt
                out[b, h, r:r + rows] = torch.softmax(s, dim=-1) @ vd
    return out


def _exact_conv(case, x, w, b, res):
    """The convolution in float64 as one matrix product per filter tap."""
    c = case
    n, k, z, p, q = _conv_out_shape(c)
    acc = torch.zeros((n * z * p * q, k), dtype=torch.float64, device=x.device)
    xc = x.permute(0, 2, 3, 4, 1)
    for t in range(c["t"]):
        for r in range(c["r"]):
            for s in range(c["s"]):
                part = xc[:, t:t + (z - 1) * c["sd"] + 1:c["sd"],
                          r:r + (p - 1) * c["sh"] + 1:c["sh"],
                          s:s + (q - 1) * c["sw"] + 1:c["sw"]]
                acc += part.reshape(-1, c["c"]).double() @ w[:, :, t, r, s].double().t().contiguous()
    if b is not None:
        acc += b.double()
    out = acc.view(n, z, p, q, k).permute(0, 4, 1, 2, 3)
    return out if res is None else out + res.double()


def exact(case, seed):
    op = case["op"]
    if op == "conv":
        return _exact_conv(case, *_inputs(case, seed))
    q, k, v = _inputs(case, seed)
    if op == "attn":
        return _exact_attention(q, k, v, case["D"] ** -0.5)
    if op == "dit":
        o = _exact_attention(q, k, v, case["D"] ** -0.5)
        return o.transpose(1, 2).reshape(case["B"], case["Sq"], case["H"] * case["D"])
    tokens = [x.reshape(case["B"], 512, -1).transpose(1, 2).unsqueeze(1) for x in (q, k, v)]
    o = _exact_attention(*tokens, 512 ** -0.5)
    return o.squeeze(1).transpose(1, 2).reshape(q.shape)


def tolerance(case):
    """About four times the relative error against float64 measured over the
    listed cases and drawn ones: the 16-bit rounding of the output (conv3d
    2.1e-4) and of the softmax weights (fp16 2.9e-4, bf16 2.3e-3), sums in 32
    bits."""
    if case["op"] == "conv":
        return {"rel": 8e-4}
    return {"rel": 1.2e-3 if case["dtype"] == "fp16" else 1e-2}

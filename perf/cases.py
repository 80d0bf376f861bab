"""Timed workloads of the library, through its public entry points.

A case is a dict of plain values.  `listed()` holds the workloads that the
repository's own configurations, tests and benchmark name; `draw(rng)` draws
further ones of the same kinds and ranges.  `prepare` makes what a program has
in hand before a call (weights uploaded once per process, device buffers),
`run` makes one call, `exact` gives the same result in 64-bit torch arithmetic.

Kinds:
  step              one denoiser step, raw caption to velocity (whole 28-block model)
  vae               latent -> image (whole decoder)
  gemma             prompt tokens -> hidden states (whole 26-layer encoder), host arrays
  glumb16           the Mix-FFN of one block on fp16 activations
  linear_attention16, cross_attention16
                    the two attention kernels of one block on fp16 activations
  self_attention32, cross_attention32
                    the fp32 op-level attention blocks (the calls that
                    attention_block_3d and cross_attention_block_3d make)
"""
import math
import os
import sys

import numpy as np
import torch

_PKG = os.path.join(os.getcwd(), "sana.cpp_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)
import sana_dit  # noqa: E402

C, E, F, CAPTION, LATENT, LAYERS = 1152, 5760, 2880, 2304, 32, 28
SELF_HEADS, CROSS_HEADS = 36, 16
VAE_CHANNELS = (128, 256, 512, 512, 1024, 1024)
VAE_ATTENTION = (False, False, False, True, True, True)
VAE_SCALING = 0.41407
# the 2B text encoder; a call gathers a few hundred embedding rows, so the
# table is cut to keep the upload short
GEMMA = dict(sana_dit.GEMMA2_2B, vocab=32768)


def listed():
    return [
        # a 512 px image, CFG pair, masked caption: the smallest step, bound by launches and latency
        {"name": "step_512px", "kind": "step", "images": 1, "side": 16, "caption": 300, "masked": True},
        # the headline: 1024 px, CFG pair, 300-token caption
        {"name": "step_1024px", "kind": "step", "images": 1, "side": 32, "caption": 300, "masked": False},
        # the largest image the model is used for
        {"name": "step_4096px", "kind": "step", "images": 1, "side": 128, "caption": 300, "masked": False},
        # the decode after a 1024 px loop
        {"name": "vae_1024px", "kind": "vae", "images": 1, "h": 32, "w": 32},
        # a small odd-sized preview
        {"name": "vae_odd", "kind": "vae", "images": 1, "h": 11, "w": 13},
        # instruction-prefixed prompt and negative prompt of one request
        {"name": "gemma_pair", "kind": "gemma", "a": 438, "b": 300},
        # one short prompt alone
        {"name": "gemma_short", "kind": "gemma", "a": 23, "b": 0},
        # the Mix-FFN at 2048 px (64 x 64 tokens), CFG pair
        {"name": "glumb16_64x64", "kind": "glumb16", "images": 2, "h": 64, "w": 64},
        # the linear attention at 2048 px with 16 heads of 72
        {"name": "linear_attention16_4096", "kind": "linear_attention16", "images": 2, "tokens": 4096, "heads": 16},
        # the cross attention of a small odd grid (23 x 23) on a short masked caption: one small launch
        {"name": "cross_attention16_529", "kind": "cross_attention16", "images": 2, "tokens": 529, "caption": 77,
         "masked": True},
        # fp32 op-level self attention at 1024 px
        {"name": "self_attention32_1024", "kind": "self_attention32", "images": 2, "tokens": 1024, "heads": 36},
        # fp32 op-level cross attention at 512 px, masked caption
        {"name": "cross_attention32_256", "kind": "cross_attention32", "images": 2, "tokens": 256, "caption": 300,
         "masked": True},
    ]


def _log_int(rng, lo, hi):
    """An integer of [lo, hi], spread over its logarithm."""
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["step", "vae", "gemma", "glumb16", "linear_attention16", "cross_attention16",
                       "self_attention32", "cross_attention32"])
    c = {"kind": kind}
    if kind == "step":
        c["images"] = rng.choice([1, 1, 2, 3])
        c["side"] = _log_int(rng, 8, int(math.sqrt(16384 / c["images"])))
        c["caption"] = _log_int(rng, 16, 512)
        c["masked"] = rng.random() < 0.5
    elif kind == "vae":
        c["images"] = rng.choice([1, 1, 1, 2])
        c["h"] = _log_int(rng, 6, 40)
        c["w"] = _log_int(rng, 6, 40)
    elif kind == "gemma":
        c["a"] = _log_int(rng, 4, 1024)
        c["b"] = _log_int(rng, 4, 512) if rng.random() < 0.5 else 0
    elif kind == "glumb16":
        c["images"] = rng.choice([1, 2, 4])
        c["h"] = _log_int(rng, 8, 96)
        c["w"] = _log_int(rng, 8, 96)
    else:
        c["images"] = rng.choice([1, 2, 4])
        small = kind.endswith("32")
        c["tokens"] = _log_int(rng, 64, 4096 if small else 16384)
        if kind.startswith("cross"):
            c["caption"] = _log_int(rng, 16, 512)
            c["masked"] = rng.random() < 0.5
        else:
            c["heads"] = rng.choice([16, 36])
    return c


# ---------------------------------------------------------------- shared state
_KEPT = {}


def _once(key, make):
    if key not in _KEPT:
        _KEPT[key] = make()
    return _KEPT[key]


def _dev():
    return torch.device("cuda")


def _stream():
    """The one stream that a serving program runs its calls on."""
    return _once("stream", torch.cuda.Stream).cuda_stream


def _gen(seed):
    return torch.Generator(device=_dev()).manual_seed(int(seed))


def _randn(shape, g, scale=1.0, dtype=torch.float32):
    return (torch.randn(shape, device=_dev(), generator=g) * scale).to(dtype)


def _mask(images, length, seed):
    """Additive key mask of padded captions, as the prompt encoder builds it."""
    g = torch.Generator().manual_seed(int(seed) + 77)
    m = torch.full((images, length), -10000.0)
    for b in range(images):
        real = int(torch.randint(max(1, length // 8), length + 1, (1,), generator=g))
        m[b, :real] = 0.0
    return m.to(_dev())


_F16_SUFFIX = ("to_q.weight", "to_k.weight", "to_v.weight", "to_out.0.weight", "conv_inverted.weight",
               "conv_point.weight")


def _dit_weights():
    """{name: device tensor}: N(0, 0.02), caption_norm ones; GEMM operands hold fp16 values."""
    g = _gen(1000)
    w = {}
    for name, shape in sorted(sana_dit.manifest().items()):
        if name == "caption_norm.weight":
            w[name] = torch.ones(shape, device=_dev())
            continue
        f16 = name.startswith("caption_projection.linear") and name.endswith("weight") or name.endswith(_F16_SUFFIX)
        w[name] = _randn(shape, g, 0.02, torch.float16 if f16 else torch.float32)
    return w


def _dit():
    def make():
        d = sana_dit.Dit()
        for name, t in _once("dit_weights", _dit_weights).items():
            a = t.cpu().numpy()
            d.set_weight_f16(name, a) if a.dtype == np.float16 else d.set_weight(name, a)
        d.check_weights()
        return d
    return _once("dit", make)


def _is_norm(name):
    return name.endswith("norm.weight") or name.endswith("norm_out.weight")


def _vae_weights():
    g = _gen(7000)
    w = {}
    for name, shape in sorted(sana_dit.vae_manifest(VAE_CHANNELS, VAE_ATTENTION).items()):
        z = _randn(shape, g)
        w[name] = 1 + 0.1 * z if _is_norm(name) else (z * 0.02).half().float()
    return w


def _vae():
    def make():
        v = sana_dit.Vae(VAE_CHANNELS, VAE_ATTENTION)
        for name, t in _once("vae_weights", _vae_weights).items():
            v.set_weight(name, t.cpu().numpy())
        v.check_weights()
        return v
    return _once("vae", make)


def _gemma_weights():
    """One draw per tensor shape, shared by the layers."""
    g = _gen(3000)
    w = {}
    for shape in sorted(set(sana_dit.gemma_manifest(**GEMMA).values())):
        z = _randn(shape, g)
        w[shape] = 1 + 0.1 * z if len(shape) == 1 else (z * 0.02).half().float()
    return w


def _gemma():
    def make():
        e = sana_dit.Gemma(GEMMA)
        host = {s: t.cpu().numpy() for s, t in _once("gemma_weights", _gemma_weights).items()}
        for name, shape in sana_dit.gemma_manifest(**GEMMA).items():
            e.set_weight(name, host[shape])
        e.check_weights()
        return e
    return _once("gemma", make)


# ---------------------------------------------------------------- prepare
def _inputs(case, seed):
    """The inputs of a case, from its seed alone."""
    k, g = case["kind"], _gen(seed)
    if k == "step":
        B, L, S = 2 * case["images"], case["caption"], case["side"]
        return {"caption": _randn((B, L, CAPTION), g), "latent": _randn((case["images"], LATENT, S, S), g),
                "mask": _mask(B, L, seed) if case["masked"] else None, "t": float(1 + (int(seed) * 37 + 998) % 999)}
    if k == "vae":
        return {"latent": _randn((case["images"], LATENT, case["h"], case["w"]), g)}
    if k == "gemma":
        r = np.random.default_rng(int(seed))
        return {"a": r.integers(0, GEMMA["vocab"], case["a"], dtype=np.int32),
                "b": r.integers(0, GEMMA["vocab"], case["b"], dtype=np.int32)}
    B = case["images"]
    if k == "glumb16":
        h = torch.float16
        return {"x": _randn((B * case["h"] * case["w"], C), g, 1.0, h), "w_inv": _randn((E, C), g, 0.02, h),
                "b_inv": _randn((E,), g, 0.02), "w_dw": _randn((9, E), g, 0.2), "b_dw": _randn((E,), g, 0.02),
                "w_pt": _randn((C, F), g, 0.02, h)}
    N = case["tokens"]
    if k == "linear_attention16":
        return {"qkv": _randn((B * N, 3 * C), g, 1.0, torch.float16)}
    L = case.get("caption", 0)
    mask = _mask(B, L, seed) if case.get("masked") else None
    if k == "cross_attention16":
        Lp = -(-L // 32) * 32
        vt = torch.zeros((B, C, Lp), device=_dev(), dtype=torch.float16)
        vt[:, :, :L] = _randn((B, C, L), g, 1.0, torch.float16)
        return {"q": _randn((B * N, C), g, 1.0, torch.float16), "k": _randn((B * L, C), g, 1.0, torch.float16),
                "vt": vt, "mask": mask}
    # op level: linear weights [in, out] as the C++ API holds them
    out = {"x": _randn((B * N, C), g), "mask": mask}
    if L:
        out["context"] = _randn((B * L, C), g)
    for n in "qkvo":
        out["w" + n] = _randn((C, C), g, 0.03)
        out["b" + n] = _randn((C,), g, 0.02)
    return out


def prepare(case, seed):
    k = case["kind"]
    s = dict(_inputs(case, seed), case=case)
    B = case.get("images", 1)
    empty = lambda *shape, dtype=torch.float32: torch.empty(shape, device=_dev(), dtype=dtype)  # noqa: E731
    if k == "step":
        s["model"] = _dit()
        s["out"] = empty(2 * B, LATENT, case["side"], case["side"])
    elif k == "vae":
        s["model"] = _vae()
        s["image"] = empty(B, 3, 32 * case["h"], 32 * case["w"])
    elif k == "gemma":
        s["model"] = _gemma()
    elif k == "glumb16":
        M = B * case["h"] * case["w"]
        s["hid"], s["glu"] = empty(M, E, dtype=torch.float16), empty(M, F, dtype=torch.float16)
        s["out"] = empty(M, C)
    elif k == "linear_attention16":
        H, N = case["heads"], case["tokens"]
        s["ws"] = empty(sana_dit.lib().sana_hip_linear_attention_workspace(B, N, H, C // H) // 4 + 4)
        s["out"] = empty(B * N, C, dtype=torch.float16)
    elif k == "cross_attention16":
        s["out"] = empty(B * case["tokens"], C, dtype=torch.float16)
    else:
        N, L = case["tokens"], case.get("caption", 0)
        H = case.get("heads", CROSS_HEADS)
        rows = {"q": N, "k": L or N, "v": L or N}
        for n, r in rows.items():
            s["p" + n], s["h" + n] = empty(B * r, C), empty(B, H, r, C // H)
        s["ho"], s["po"], s["out"] = empty(B, H, N, C // H), empty(B * N, C), empty(B * N, C)
        if L:
            s["scores"] = empty(B * H, N, L)
        else:
            s["state"] = empty(B * H, C // H + 1, C // H)
    _stream()
    torch.cuda.synchronize()
    return s


# ---------------------------------------------------------------- run
def _linear32(x, rows, w, b, out, st):
    sana_dit.check(sana_dit.lib().sana_op_gemm_f32(x.data_ptr(), C, 0, w.data_ptr(), C, 0, 0, b.data_ptr(), 1,
                                                   out.data_ptr(), C, 0, rows, C, C, 1, 0, st))


def _heads32(x, y, B, N, H, split, st):
    sana_dit.check(sana_dit.lib().sana_op_heads_f32(x.data_ptr(), y.data_ptr(), B, N, H, C // H, split, st))


def run(s):
    case = s["case"]
    k, B, st, lib, check = case["kind"], case.get("images", 1), _stream(), sana_dit.lib(), sana_dit.check
    if k == "step":
        S = case["side"]
        s["model"].step_device(s["caption"], case["caption"], s["mask"], s["latent"], (B, LATENT, S, S), s["t"],
                               s["out"], st)
        return s["out"]
    if k == "vae":
        s["model"].decode_device(s["latent"], tuple(s["latent"].shape), s["image"], st)
        return s["image"]
    if k == "gemma":
        if case["b"]:
            return s["model"].encode_pair(s["a"], s["b"])
        return s["model"].encode(s["a"])
    if k == "glumb16":
        h, w = case["h"], case["w"]
        M = B * h * w
        check(lib.sana_hip_gemm(s["x"].data_ptr(), C, s["w_inv"].data_ptr(), C, M, E, C, s["b_inv"].data_ptr(), 1,
                                s["hid"].data_ptr(), E, None, 0, st))
        check(lib.sana_hip_dwconv_glu(s["hid"].data_ptr(), E, s["w_dw"].data_ptr(), s["b_dw"].data_ptr(),
                                      s["glu"].data_ptr(), F, B, h, w, F, st))
        check(lib.sana_hip_gemm(s["glu"].data_ptr(), F, s["w_pt"].data_ptr(), F, M, C, F, None, 0, None, 0,
                                s["out"].data_ptr(), C, st))
        return s["out"]
    N = case["tokens"]
    if k == "linear_attention16":
        H, q = case["heads"], s["qkv"].data_ptr()
        check(lib.sana_hip_linear_attention(q, q + 2 * C, q + 4 * C, 3 * C, s["out"].data_ptr(), C, B, N, H, C // H,
                                            s["ws"].data_ptr(), st))
        return s["out"]
    m = s["mask"].data_ptr() if s["mask"] is not None else None
    if k == "cross_attention16":
        L = case["caption"]
        check(lib.sana_hip_cross_attention(s["q"].data_ptr(), C, s["k"].data_ptr(), C, s["vt"].data_ptr(),
                                           s["vt"].shape[2], m, s["out"].data_ptr(), C, B, N, L, CROSS_HEADS,
                                           C // CROSS_HEADS, st))
        return s["out"]
    # projections, head split, attention, merge, output projection (attention_block_3d / cross_attention_block_3d)
    L = case.get("caption", 0)
    H = case.get("heads", CROSS_HEADS)
    D = C // H
    for n, src, r in (("q", "x", N), ("k", "context" if L else "x", L or N), ("v", "context" if L else "x", L or N)):
        _linear32(s[src], B * r, s["w" + n], s["b" + n], s["p" + n], st)
        _heads32(s["p" + n], s["h" + n], B, r, H, 1, st)
    if L:
        check(lib.sana_op_gemm_f32(s["hq"].data_ptr(), D, N * D, s["hk"].data_ptr(), D, L * D, 1, None, 1,
                                   s["scores"].data_ptr(), L, N * L, N, L, D, B * H, 0, st))
        check(lib.sana_op_softmax_f32(s["scores"].data_ptr(), s["scores"].data_ptr(), B * H * N, L,
                                      1.0 / math.sqrt(D), m, H * N, st))
        check(lib.sana_op_gemm_f32(s["scores"].data_ptr(), L, N * L, s["hv"].data_ptr(), D, L * D, 0, None, 1,
                                   s["ho"].data_ptr(), D, N * D, N, D, L, B * H, 0, st))
    else:
        check(lib.sana_op_linear_attention_f32(s["hq"].data_ptr(), s["hk"].data_ptr(), s["hv"].data_ptr(),
                                               s["ho"].data_ptr(), B * H, N, N, D, s["state"].data_ptr(), st))
    _heads32(s["ho"], s["po"], B, N, H, 0, st)
    _linear32(s["po"], B * N, s["wo"], s["bo"], s["out"], st)
    return s["out"]


# ---------------------------------------------------------------- work
def _linear_attention_flops(rows, heads, d):
    return 2 * 2 * rows * heads * (d + 1) * d


def work(case):
    k, B = case["kind"], case.get("images", 1)
    if k == "step":
        rows, N, L = 2 * B * case["side"] ** 2, case["side"] ** 2, case["caption"]
        cr = 2 * B * L
        per = 2 * rows * (3 * C * C + C * C + C * C + C * C + E * C + F * C) + 2 * 9 * rows * E
        per += _linear_attention_flops(rows, SELF_HEADS, C // SELF_HEADS) + 2 * 2 * rows * L * C + 2 * 2 * cr * C * C
        flops = LAYERS * per + 2 * cr * (CAPTION * C + C * C) + 2 * rows * 2 * LATENT * C
        params = LAYERS * (8 * C * C + E * C + F * C) + CAPTION * C + C * C
        time_params = 256 * C + C * C + 6 * C * C + LAYERS * (11 * E + 6 * C)
        return {"flops": flops,
                "bytes": 2 * params + 4 * time_params + 4 * (cr * CAPTION + 3 * B * LATENT * N + cr * case["masked"])}
    if k == "vae":
        n, L, h, w = len(VAE_CHANNELS), len(VAE_CHANNELS), case["h"], case["w"]
        f, p = 2 * 9 * LATENT * VAE_CHANNELS[-1] * h * w, 9 * LATENT * VAE_CHANNELS[-1]
        for i in range(n - 1, -1, -1):
            c, sc = VAE_CHANNELS[i], 2 ** (L - 1 - i)
            P = h * sc * w * sc
            if i + 1 < n:
                f += 2 * 9 * VAE_CHANNELS[i + 1] * c * P
                p += 9 * VAE_CHANNELS[i + 1] * c
            for _ in range(3):
                if not VAE_ATTENTION[i]:
                    f += 2 * (2 * 9 * c * c * P)
                    p += 2 * 9 * c * c
                else:
                    e = 4 * c
                    f += 2 * P * (3 * c * c + 25 * 3 * c + 32 * 3 * c + c * 2 * c + 2 * e * c + 9 * 2 * e + c * e)
                    f += 2 * _linear_attention_flops(P, c // 32, 32)
                    p += 3 * c * c + 25 * 3 * c + 32 * 3 * c + c * 2 * c + 2 * e * c + 9 * 2 * e + c * e
        P = h * w * 4 ** (n - 1)
        f += 2 * 9 * VAE_CHANNELS[0] * 3 * P
        return {"flops": B * f, "bytes": 2 * p + 4 * B * (LATENT * h * w + 3 * P)}
    if k == "gemma":
        H, d, n = GEMMA["hidden"], GEMMA["head_dim"], GEMMA["layers"]
        dq, dkv, ffn = GEMMA["heads"] * d, GEMMA["kv_heads"] * d, GEMMA["ffn"]
        mats = H * (dq + 2 * dkv) + dq * H + 3 * H * ffn
        f = 0
        for T in (case["a"], case["b"]):
            f += n * (2 * T * mats + 2 * 2 * (T * (T + 1) // 2) * dq)
        T = case["a"] + case["b"]
        return {"flops": f, "bytes": n * 2 * mats + T * (4 + 2 * H + 4 * H)}
    if k == "glumb16":
        M = B * case["h"] * case["w"]
        return {"flops": 2 * M * (E * C + F * C + 9 * E),
                "bytes": 2 * (M * C + E * C + F * C) + 4 * (11 * E + M * C)}
    N = case["tokens"]
    if k == "linear_attention16":
        return {"flops": _linear_attention_flops(B * N, case["heads"], C // case["heads"]), "bytes": 2 * 4 * B * N * C}
    L = case.get("caption", 0)
    if k == "cross_attention16":
        return {"flops": 2 * 2 * B * N * L * C, "bytes": 2 * (2 * B * N * C + 2 * B * L * C) + 4 * B * L * case["masked"]}
    if k == "self_attention32":
        return {"flops": 2 * 4 * B * N * C * C + _linear_attention_flops(B * N, case["heads"], C // case["heads"]),
                "bytes": 4 * (2 * B * N * C + 4 * C * C + 4 * C)}
    return {"flops": 2 * (2 * B * N + 2 * B * L) * C * C + 2 * 2 * B * N * L * C,
            "bytes": 4 * (2 * B * N * C + B * L * C + 4 * C * C + 4 * C + B * L * case["masked"])}


def tolerance(case):
    """fp16 operands with fp32 sums (fp32 throughout for the *32 kinds): about
    four times the measured distance from the 64-bit result (step 2.5e-4, vae
    4.9e-4, gemma 3.6e-4, glumb16 3.7e-4, linear_attention16 2.1e-4,
    cross_attention16 2.7e-4, the fp32 kinds 1.3e-6)."""
    return {"rel": {"step": 1e-3, "vae": 2e-3, "gemma": 1.5e-3, "glumb16": 1.5e-3, "linear_attention16": 9e-4,
                    "cross_attention16": 1.1e-3, "self_attention32": 5e-6, "cross_attention32": 5e-6}[case["kind"]]}


# ---------------------------------------------------------------- exact
def _silu64(x):
    return x * torch.sigmoid(x)


def _gelu64(x):
    return 0.5 * x * (1.0 + torch.tanh(math.sqrt(2.0 / math.pi) * (x + 0.044715 * x ** 3)))


def _taps(x, w, ks):
    """Depthwise ks x ks (zero padded) on [B, H, W, ch]; w [ks * ks, ch]."""
    B, H, W, ch = x.shape
    r = ks // 2
    p = torch.zeros((B, H + 2 * r, W + 2 * r, ch), device=x.device, dtype=x.dtype)
    p[:, r:r + H, r:r + W] = x
    out = torch.zeros_like(x)
    for ky in range(ks):
        for kx in range(ks):
            out += p[:, ky:ky + H, kx:kx + W] * w[ky * ks + kx]
    return out


def _linear_attention64(q, k, v, heads):
    """q, k, v [B, N, ch] -> [B, N, ch]."""
    B, N, ch = q.shape
    hd = lambda x: x.reshape(B, N, heads, ch // heads).transpose(1, 2).contiguous()  # noqa: E731
    q, k, v = torch.relu(hd(q)), torch.relu(hd(k)), hd(v)
    num = torch.matmul(q, torch.matmul(k.transpose(2, 3).contiguous(), v))
    den = torch.matmul(q, k.sum(2).unsqueeze(-1)) + 1e-15
    return (num / den).transpose(1, 2).reshape(B, N, ch)


def _attention64(q, k, v, heads, mask):
    B, N, ch = q.shape
    D = ch // heads
    hd = lambda x: x.reshape(B, -1, heads, D).transpose(1, 2).contiguous()  # noqa: E731
    q, k, v = hd(q), hd(k), hd(v)
    s = torch.matmul(q, k.transpose(2, 3).contiguous()) / math.sqrt(D)
    if mask is not None:
        s = s + mask.double()[:, None, None, :]
    return torch.matmul(torch.softmax(s, -1), v).transpose(1, 2).reshape(B, N, ch)


def _glumb64(x, H, W, w_inv, b_inv, w_dw, b_dw, w_pt):
    """x [B, H * W, ch]; w_dw tap-major [9, 2 * half]."""
    B = x.shape[0]
    h = _silu64(x @ w_inv.T + b_inv)
    h = _taps(h.reshape(B, H, W, -1), w_dw, 3) + b_dw
    half = h.shape[-1] // 2
    return (h[..., :half] * _silu64(h[..., half:])).reshape(B, H * W, half) @ w_pt.T


def _layer_norm64(x, eps):
    m = x.mean(-1, keepdim=True)
    d = x - m
    return d / torch.sqrt((d * d).mean(-1, keepdim=True) + eps)


def _rms64(x, w, eps):
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + eps) * w


def _exact_step(case, i):
    W = _once("dit_weights", _dit_weights)
    f = lambda n: W[n].double()  # noqa: E731
    B, S = 2 * case["images"], case["side"]
    N = S * S
    h = _gelu64(i["caption"].double() @ f("caption_projection.linear_1.weight").T + f("caption_projection.linear_1.bias"))
    ctx = _rms64(h @ f("caption_projection.linear_2.weight").T + f("caption_projection.linear_2.bias"),
                 f("caption_norm.weight"), 1e-5)
    lat = i["latent"].double().reshape(case["images"], LATENT, N).transpose(1, 2)
    x = torch.cat([lat, lat]) @ f("patch_embed.proj.weight").reshape(C, LATENT).T + f("patch_embed.proj.bias")
    freq = torch.exp(torch.arange(128, device=_dev(), dtype=torch.float64) * (-math.log(10000.0) / 128))
    a = i["t"] * freq
    te = "time_embed.emb.timestep_embedder."
    e = _silu64(torch.cat([torch.cos(a), torch.sin(a)]) @ f(te + "linear_1.weight").T + f(te + "linear_1.bias"))
    emb = e @ f(te + "linear_2.weight").T + f(te + "linear_2.bias")
    tmod = (_silu64(emb) @ f("time_embed.linear.weight").T + f("time_embed.linear.bias")).reshape(6, C)
    for blk in range(LAYERS):
        p = f"transformer_blocks.{blk}."
        m = tmod + f(p + "scale_shift_table")
        y = _layer_norm64(x, 1e-6) * (1 + m[1]) + m[0]
        q, k, v = (y @ f(p + f"attn1.to_{n}.weight").T for n in "qkv")
        o = _linear_attention64(q, k, v, SELF_HEADS) @ f(p + "attn1.to_out.0.weight").T + f(p + "attn1.to_out.0.bias")
        x = x + m[2] * o
        q = x @ f(p + "attn2.to_q.weight").T + f(p + "attn2.to_q.bias")
        k = ctx @ f(p + "attn2.to_k.weight").T + f(p + "attn2.to_k.bias")
        v = ctx @ f(p + "attn2.to_v.weight").T + f(p + "attn2.to_v.bias")
        o = _attention64(q, k, v, CROSS_HEADS, i["mask"])
        x = x + o @ f(p + "attn2.to_out.0.weight").T + f(p + "attn2.to_out.0.bias")
        y = _layer_norm64(x, 1e-6) * (1 + m[4]) + m[3]
        x = x + m[5] * _glumb64(y, S, S, f(p + "ff.conv_inverted.weight").reshape(E, C), f(p + "ff.conv_inverted.bias"),
                                f(p + "ff.conv_depth.weight").reshape(E, 9).T, f(p + "ff.conv_depth.bias"),
                                f(p + "ff.conv_point.weight").reshape(C, F))
    sst = f("scale_shift_table")
    y = _layer_norm64(x, 1e-6) * (1 + emb + sst[1]) + emb + sst[0]
    out = y @ f("proj_out.weight").T + f("proj_out.bias")
    return out.transpose(1, 2).reshape(B, LATENT, S, S).contiguous()


def _conv64(x, w, b):
    """3x3 same convolution of [B, H, W, ci] with w [co, ci, 3, 3]."""
    B, H, W, ci = x.shape
    p = torch.zeros((B, H + 2, W + 2, ci), device=x.device, dtype=x.dtype)
    p[:, 1:1 + H, 1:1 + W] = x
    out = torch.zeros((B * H * W, w.shape[0]), device=x.device, dtype=x.dtype)
    for ky in range(3):
        for kx in range(3):
            out += p[:, ky:ky + H, kx:kx + W].reshape(B * H * W, ci) @ w[:, :, ky, kx].T
    if b is not None:
        out += b
    return out.reshape(B, H, W, -1)


def _exact_vae(case, i):
    Wt = _once("vae_weights", _vae_weights)
    f = lambda n: Wt[n].double()  # noqa: E731
    n = len(VAE_CHANNELS)
    x = i["latent"].double().permute(0, 2, 3, 1).contiguous() / VAE_SCALING
    x = _conv64(x, f("decoder.conv_in.weight"), f("decoder.conv_in.bias")) + x.repeat_interleave(
        VAE_CHANNELS[-1] // LATENT, dim=3)
    for lv in range(n - 1, -1, -1):
        c, p, base = VAE_CHANNELS[lv], f"decoder.up_blocks.{lv}.", 0
        if lv + 1 < n:
            B, H, W, ci = x.shape
            up = x.repeat_interleave(2, 1).repeat_interleave(2, 2)
            y = _conv64(up, f(p + "0.conv.weight"), f(p + "0.conv.bias"))
            short = x.repeat_interleave(4 * c // ci, dim=3).reshape(B, H, W, c, 2, 2)
            x = y + short.permute(0, 1, 4, 2, 5, 3).reshape(B, 2 * H, 2 * W, c)
            base = 1
        B, H, W, _ = x.shape
        for layer in range(base, base + 3):
            q = f"{p}{layer}."
            if not VAE_ATTENTION[lv]:
                h = _silu64(_conv64(x, f(q + "conv1.weight"), f(q + "conv1.bias")))
                x = x + _rms64(_conv64(h, f(q + "conv2.weight"), None), f(q + "norm.weight"), 1e-5) + f(q + "norm.bias")
                continue
            qkv = torch.cat([x @ f(q + f"attn.to_{m}.weight").T for m in "qkv"], -1)
            ms = _taps(qkv, f(q + "attn.to_qkv_multiscale.0.proj_in.weight").reshape(3 * c, 25).T, 5)
            wg = f(q + "attn.to_qkv_multiscale.0.proj_out.weight").reshape(3 * c // 32, 32, 32)
            ms = torch.matmul(ms.reshape(-1, 3 * c // 32, 32).transpose(0, 1).contiguous(),
                              wg.transpose(1, 2).contiguous()).transpose(0, 1)
            heads = []
            for src in (qkv, ms):
                s = src.reshape(B, H * W, c // 32, 3, 32)
                heads.append(_linear_attention64(*(s[..., j, :].reshape(B, H * W, c) for j in range(3)), c // 32))
            o = torch.cat(heads, -1) @ f(q + "attn.to_out.weight").T
            x = x + (_rms64(o, f(q + "attn.norm_out.weight"), 1e-5) + f(q + "attn.norm_out.bias")).reshape(B, H, W, c)
            o = _glumb64(x.reshape(B, H * W, c), H, W, f(q + "conv_out.conv_inverted.weight").reshape(-1, c),
                         f(q + "conv_out.conv_inverted.bias"), f(q + "conv_out.conv_depth.weight").reshape(-1, 9).T,
                         f(q + "conv_out.conv_depth.bias"), f(q + "conv_out.conv_point.weight").reshape(c, -1))
            x = x + (_rms64(o, f(q + "conv_out.norm.weight"), 1e-5) + f(q + "conv_out.norm.bias")).reshape(B, H, W, c)
    x = torch.relu(_rms64(x, f("decoder.norm_out.weight"), 1e-5) + f("decoder.norm_out.bias"))
    return _conv64(x, f("decoder.conv_out.weight"), f("decoder.conv_out.bias")).permute(0, 3, 1, 2).contiguous()


def _rope64(x, theta):
    T, _, d = x.shape
    inv = theta ** (-torch.arange(0, d, 2, device=x.device, dtype=torch.float64) / d)
    a = torch.arange(T, device=x.device, dtype=torch.float64)[:, None] * inv
    c, s = torch.cos(a)[:, None], torch.sin(a)[:, None]
    u, v = x[..., :d // 2], x[..., d // 2:]
    return torch.cat([u * c - v * s, v * c + u * s], -1)


def _exact_gemma(tokens):
    G, Wt = GEMMA, _once("gemma_weights", _gemma_weights)
    names = sana_dit.gemma_manifest(**G)
    f = lambda n: Wt[names[n]].double()  # noqa: E731
    T, nh, nkv, d, eps = len(tokens), G["heads"], G["kv_heads"], G["head_dim"], G["rms_eps"]
    x = Wt[names["token_embd.weight"]][torch.from_numpy(tokens).to(_dev()).long()].double() * math.sqrt(G["hidden"])
    pos = torch.arange(T, device=_dev())
    late = pos[None, :] > pos[:, None]
    for l in range(G["layers"]):
        p = f"blk.{l}."
        h = _rms64(x, f(p + "attn_norm.weight"), eps)
        q = _rope64((h @ f(p + "attn_q.weight").T).reshape(T, nh, d), G["rope_theta"]) * G["query_scale"]
        k = _rope64((h @ f(p + "attn_k.weight").T).reshape(T, nkv, d), G["rope_theta"])
        v = (h @ f(p + "attn_v.weight").T).reshape(T, nkv, d)
        k, v = k.repeat_interleave(nh // nkv, 1), v.repeat_interleave(nh // nkv, 1)
        hidden = late | (pos[None, :] <= pos[:, None] - G["sliding_window"]) if l % 2 == 0 else late
        s = torch.matmul(q.transpose(0, 1).contiguous(), k.permute(1, 2, 0).contiguous())
        s = (G["softcap"] * torch.tanh(s / G["softcap"])).masked_fill(hidden, -math.inf)
        o = torch.matmul(torch.softmax(s, -1), v.transpose(0, 1).contiguous()).transpose(0, 1).reshape(T, nh * d)
        x = x + _rms64(o @ f(p + "attn_output.weight").T, f(p + "post_attention_norm.weight"), eps)
        h = _rms64(x, f(p + "ffn_norm.weight"), eps)
        y = _gelu64(h @ f(p + "ffn_gate.weight").T) * (h @ f(p + "ffn_up.weight").T)
        x = x + _rms64(y @ f(p + "ffn_down.weight").T, f(p + "post_ffw_norm.weight"), eps)
    return _rms64(x, f("output_norm.weight"), eps).cpu().numpy()


def exact(case, seed):
    k, i, B = case["kind"], _inputs(case, seed), case.get("images", 1)
    if k == "step":
        return _exact_step(case, i)
    if k == "vae":
        return _exact_vae(case, i)
    if k == "gemma":
        return (_exact_gemma(i["a"]), _exact_gemma(i["b"])) if case["b"] else _exact_gemma(i["a"])
    d = {n: t.double() if isinstance(t, torch.Tensor) else t for n, t in i.items()}
    if k == "glumb16":
        h, w = case["h"], case["w"]
        return _glumb64(d["x"].reshape(B, h * w, C), h, w, d["w_inv"], d["b_inv"], d["w_dw"], d["b_dw"],
                        d["w_pt"]).reshape(B * h * w, C)
    N = case["tokens"]
    if k == "linear_attention16":
        q, kk, v = d["qkv"].reshape(B, N, 3, C).unbind(2)
        return _linear_attention64(q, kk, v, case["heads"]).reshape(B * N, C)
    if k == "cross_attention16":
        L = case["caption"]
        v = d["vt"][:, :, :L].transpose(1, 2)
        return _attention64(d["q"].reshape(B, N, C), d["k"].reshape(B, L, C), v, CROSS_HEADS, i["mask"]).reshape(B * N, C)
    L = case.get("caption", 0)
    src = {"q": d["x"], "k": d["context"] if L else d["x"], "v": d["context"] if L else d["x"]}
    q, kk, v = ((src[n] @ d["w" + n] + d["b" + n]).reshape(B, -1, C) for n in "qkv")
    o = _attention64(q, kk, v, CROSS_HEADS, i["mask"]) if L else _linear_attention64(q, kk, v, case["heads"])
    return o.reshape(B * N, C) @ d["wo"] + d["bo"]

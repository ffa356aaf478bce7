"""Performance cases of the quantized denoiser path: the calls a denoise step
makes through the package's public entry points, at the shapes of the SD1.5,
SDXL and FLUX configs and over the ranges around them (other image sizes,
batches, context lengths, data types).

Kinds of case:

* ``linear``  one ``Int8Linear`` call, ``[M, K] -> [M, N]``;
* ``geglu``   the UNet feed-forward ``int8_geglu_ff``, dim -> 2 x 4 dim -> dim;
* ``mlp``     ``int8_mlp``, dim -> 4 dim -> dim with a GELU between;
* ``modlin``  LayerNorm-modulate-quantize, then the layer on the codes;
* ``gated``   ``residual + gate * linear2(cat(attention, gelu(mlp)))``;
* ``qknorm``  the per-head q / k RMSNorm + rotary pass, with the copy of v;
* ``attn``    ``attention_bhld(..., "int8_turing")`` on strided views;
* ``block``   one UNet transformer block: self-attention, cross-attention over
  a text context and the GEGLU feed-forward, with their norms and residuals.

Activations are N(0, 1) with 0.5% of the channels 20 times larger, weights and
biases N(0, 0.02); attention keys carry a per-channel offset of N(0, 2) in the
UNet cases. Layers rotate by 256 where their width allows it, else not at all.
"""

import math

import torch
import torch.nn as nn
import torch.nn.functional as F

import diffucore_amd as dc

DTYPES = {"fp16": torch.float16, "bf16": torch.bfloat16, "fp32": torch.float32}


def listed():
    return [
        # the smallest: SDXL cross-attention's stacked k / v projection of a
        # 77-token text context, two samples; launches and latency count
        {"name": "ctx_kv", "kind": "linear", "M": 154, "K": 2048, "N": 2560, "dtype": "fp16", "bias": False},
        # the SD1.5 linear of the float32 config: unrotated, float32 in and out
        {"name": "sd15_ff_fp32", "kind": "linear", "M": 8192, "K": 320, "N": 1280, "dtype": "fp32", "bias": True},
        # SDXL's stacked q / k / v at the 832 x 1216 image size (52 x 76 tokens): a ragged row count
        {"name": "sdxl_qkv_832x1216", "kind": "linear", "M": 7904, "K": 640, "N": 1920, "dtype": "fp16", "bias": False},
        # FLUX 1024^2: the img and the txt stream's MLP of a double block
        {"name": "flux_mlp_img", "kind": "mlp", "M": 4096, "dim": 3072, "dtype": "bf16", "act": "tanh"},
        {"name": "flux_mlp_txt", "kind": "mlp", "M": 512, "dim": 3072, "dtype": "bf16", "act": "tanh"},
        # a FLUX single block's linear1 behind its modulated LayerNorm, and its gated linear2
        {"name": "flux_linear1", "kind": "modlin", "M": 4608, "K": 3072, "N": 21504, "dtype": "bf16"},
        {"name": "flux_linear2", "kind": "gated", "M": 4608, "K1": 3072, "K2": 12288, "N": 3072, "dtype": "bf16"},
        # a FLUX double block's q / k norm and rotary pass over the img stream
        {"name": "flux_qk_norm", "kind": "qknorm", "B": 1, "L": 4096, "H": 24, "D": 128, "dtype": "bf16"},
        # self-attention: SD1.5 512^2 (head dim 40), SDXL at 832 x 1216 (a ragged length), FLUX 1024^2
        {"name": "sd15_attn", "kind": "attn", "B": 2, "H": 8, "Lq": 4096, "Lk": 4096, "D": 40, "dtype": "fp16"},
        {"name": "sdxl_attn_832x1216", "kind": "attn", "B": 2, "H": 10, "Lq": 3952, "Lk": 3952, "D": 64, "dtype": "fp16"},
        {"name": "flux_attn", "kind": "attn", "B": 1, "H": 24, "Lq": 4608, "Lk": 4608, "D": 128, "dtype": "bf16"},
        # a whole call: one SDXL transformer block of the 1280-channel level, 32 x 32 tokens, the CFG pair
        {"name": "sdxl_block", "kind": "block", "B": 2, "L": 1024, "dim": 1280, "H": 20, "ctx": 77, "ctx_dim": 2048,
         "dtype": "fp16"},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["linear", "linear", "linear", "geglu", "mlp", "modlin", "gated", "qknorm", "attn", "attn", "attn",
                       "block"])
    half = rng.choice(["fp16", "fp16", "bf16"])
    if kind == "linear":
        K, N = rng.choice([(320, 320), (320, 960), (320, 1280), (640, 640), (640, 1920), (768, 640), (1280, 1280),
                           (1280, 3840), (2048, 1280), (2048, 2560), (3072, 3072), (3072, 9216)])
        return {"kind": kind, "M": _log(rng, 20, 9216), "K": K, "N": N,
                "dtype": rng.choice([half, half, half, "fp32"]), "bias": rng.random() < 0.5}
    if kind == "geglu":
        return {"kind": kind, "M": _log(rng, 128, 8192), "dim": rng.choice([320, 640, 1280]), "dtype": half}
    if kind == "mlp":
        act = rng.choice(["tanh", "erf"])
        return {"kind": kind, "M": _log(rng, 64, 4096), "dim": 3072 if act == "tanh" else 2048, "dtype": "bf16",
                "act": act}
    if kind == "modlin":
        return {"kind": kind, "M": _log(rng, 64, 4608), "K": 3072, "N": rng.choice([9216, 21504]), "dtype": "bf16"}
    if kind == "gated":
        return {"kind": kind, "M": _log(rng, 64, 4608), "K1": 3072, "K2": 12288, "N": 3072, "dtype": "bf16"}
    if kind == "qknorm":
        return {"kind": kind, "B": rng.choice([1, 2]), "L": _log(rng, 128, 4096), "H": 24, "D": 128, "dtype": "bf16"}
    if kind == "attn":
        H, D = rng.choice([(8, 40), (8, 80), (10, 64), (20, 64), (24, 128)])
        L = _log(rng, 200, 4608)
        B = 1 if D == 128 else rng.choice([1, 2])
        if H == 20:
            L = min(L, 2400 + L % 64)
        return {"kind": kind, "B": B, "H": H, "Lq": L, "Lk": rng.choice([L, L, L, _log(rng, 200, L + 1)]), "D": D,
                "dtype": "bf16" if D == 128 else half}
    dim, H, most = rng.choice([(640, 10, 4096), (1280, 20, 1024)])
    return {"kind": "block", "B": rng.choice([1, 2]), "L": _log(rng, 200, most), "dim": dim, "H": H, "ctx": 77,
            "ctx_dim": 2048, "dtype": half}


# ---------------------------------------------------------------- inputs

def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(seed)


def _acts(g, shape, dtype):
    """N(0, 1) with 0.5% of the channels (at least one) 20 times larger."""
    x = torch.randn(shape, generator=g, device="cuda")
    n = max(1, shape[-1] // 200)
    x[..., torch.randperm(shape[-1], generator=g, device="cuda")[:n]] *= 20.0
    return x.to(dtype)


def _group(width):
    return 256 if width % 256 == 0 else 0


def _weights(g, n, k, bias, dtype):
    """(weight, bias or None) of one float layer, N(0, 0.02)."""
    w = (torch.randn(n, k, generator=g, device="cuda") * 0.02).to(dtype)
    return w, (torch.randn(n, generator=g, device="cuda") * 0.02).to(dtype) if bias else None


def _layer(w, b):
    """The W8A8 layer a loader makes of a float one."""
    n, k = w.shape
    lin = nn.Linear(k, n, bias=b is not None, device="meta")
    lin.weight = nn.Parameter(w, requires_grad=False)
    if b is not None:
        lin.bias = nn.Parameter(b, requires_grad=False)
    return dc.Int8Linear.from_linear(lin, _group(k), "cuda")


def _layer_shapes(c):
    """{name: (out features, in features, bias)} of the case's float layers."""
    kind = c["kind"]
    if kind == "linear":
        return {"lin": (c["N"], c["K"], c["bias"])}
    if kind == "geglu":
        return {"proj": (8 * c["dim"], c["dim"], True), "out": (c["dim"], 4 * c["dim"], True)}
    if kind == "mlp":
        return {"l1": (4 * c["dim"], c["dim"], True), "l2": (c["dim"], 4 * c["dim"], True)}
    if kind == "modlin":
        return {"lin": (c["N"], c["K"], True)}
    if kind == "gated":
        return {"lin": (c["N"], c["K1"] + c["K2"], True)}
    if kind == "block":
        d = c["dim"]
        return {"qkv": (3 * d, d, False), "out1": (d, d, True), "q2": (d, d, False), "kv2": (2 * d, c["ctx_dim"], False),
                "out2": (d, d, True), "proj": (8 * d, d, True), "ff": (d, 4 * d, True)}
    return {}


def _rotary(L, D):
    """[1, L, D / 2, 2, 2] float32 rotation matrices of positions 0 .. L - 1."""
    inv = 10000.0 ** (-torch.arange(0, D, 2, dtype=torch.float64, device="cuda") / D)
    a = torch.arange(L, dtype=torch.float64, device="cuda")[:, None] * inv
    c, s = a.cos(), a.sin()
    return torch.stack((c, -s, s, c), -1).unflatten(-1, (2, 2)).float()[None]


def _inputs(c, seed):
    """The tensors of a case: activations, and the float layers' weights."""
    g = _gen(seed)
    dt = DTYPES[c["dtype"]]
    kind = c["kind"]
    s = {"w": {k: _weights(g, n, kk, b, dt) for k, (n, kk, b) in _layer_shapes(c).items()}}
    if kind == "linear":
        s["x"] = _acts(g, (c["M"], c["K"]), dt)
    elif kind in ("geglu", "mlp"):
        s["x"] = _acts(g, (c["M"], c["dim"]), dt)
    elif kind == "modlin":
        s["x"] = _acts(g, (c["M"], c["K"]), dt)
        s["sc1"] = 1 + (torch.randn(1, c["K"], generator=g, device="cuda") * 0.2).to(dt)
        s["sh"] = (torch.randn(1, c["K"], generator=g, device="cuda") * 0.2).to(dt)
    elif kind == "gated":
        s["attn"] = torch.randn(c["M"], c["K1"], generator=g, device="cuda").mul_(0.3).to(dt)
        s["mlp"] = torch.randn(c["M"], c["K2"], generator=g, device="cuda").to(dt)
        s["res"] = torch.randn(c["M"], c["N"], generator=g, device="cuda").to(dt)
        s["gate"] = (torch.randn(1, c["N"], generator=g, device="cuda") * 0.5).to(dt)
    elif kind == "qknorm":
        s["qkv"] = torch.randn(c["B"], c["L"], 3, c["H"], c["D"], generator=g, device="cuda").to(dt)
        s["wq"], s["wk"] = ((1 + 0.1 * torch.randn(c["D"], generator=g, device="cuda")).to(dt) for _ in range(2))
        s["pe"] = _rotary(c["L"], c["D"])
    elif kind == "attn":
        for n, L in (("q", c["Lq"]), ("k", c["Lk"]), ("v", c["Lk"])):
            t = torch.randn(c["B"], L, c["H"] * c["D"], generator=g, device="cuda")
            if n == "k" and c["D"] < 128:   # UNet keys; FLUX normalizes its own per head
                t += 2.0 * torch.randn(c["H"] * c["D"], generator=g, device="cuda")
            s[n] = t.to(dt)
    else:
        s["x"] = _acts(g, (c["B"], c["L"], c["dim"]), dt)
        s["ctx"] = _acts(g, (c["B"], c["ctx"], c["ctx_dim"]), dt)
        s["norms"] = [[(1 + 0.1 * torch.randn(c["dim"], generator=g, device="cuda")).to(dt),
                       (0.1 * torch.randn(c["dim"], generator=g, device="cuda")).to(dt)] for _ in range(3)]
    return s


def prepare(case, seed):
    s = _inputs(case, seed)
    s["case"] = case
    s["layers"] = {k: _layer(w, b) for k, (w, b) in s.pop("w").items()}
    if case["kind"] == "attn":
        for n in "qkv":   # (B, H, L, D) views of the projections' outputs
            s[n] = s[n].unflatten(-1, (case["H"], case["D"])).transpose(1, 2)
    return s


# ---------------------------------------------------------------- one pass

def _heads(t, h):
    return t.unflatten(-1, (h, -1)).transpose(1, 2)


def run(s):
    c, ly = s["case"], s["layers"]
    kind = c["kind"]
    if kind == "linear":
        return ly["lin"](s["x"])
    if kind == "geglu":
        return dc.int8_geglu_ff(s["x"], ly["proj"], ly["out"])
    if kind == "mlp":
        return dc.int8_mlp(s["x"], ly["l1"], ly["l2"], "tanh" if c["act"] == "tanh" else "none")
    if kind == "modlin":
        lin = ly["lin"]
        q, sc = dc.ln_mod_quantize(s["x"], s["sc1"], s["sh"], c["M"], 1e-6, lin.group)
        return lin.matmul_quantized(q, sc, s["x"].dtype)
    if kind == "gated":
        lin = ly["lin"]
        q, sc = dc.act_quantize(s["mlp"], lin.group, "gelu_tanh", prefix=s["attn"])
        return dc.matmul_quantized_gated([(lin, q, sc, s["res"], s["gate"])], s["res"].dtype)[0]
    if kind == "qknorm":
        x = s["qkv"]
        return dc.flux_qk_norm_rope(x[:, :, 0], x[:, :, 1], s["wq"], s["wk"], s["pe"], v=x[:, :, 2])
    if kind == "attn":
        return dc.attention_bhld(s["q"], s["k"], s["v"], "int8_turing")
    x, ctx, H = s["x"], s["ctx"], c["H"]
    (g1, b1), (g2, b2), (g3, b3) = s["norms"]
    d = (c["dim"],)
    q, k, v = ly["qkv"](F.layer_norm(x, d, g1, b1)).chunk(3, -1)
    x = x + ly["out1"](dc.attention_bhld(_heads(q, H), _heads(k, H), _heads(v, H), "int8_turing"))
    q = ly["q2"](F.layer_norm(x, d, g2, b2))
    k, v = ly["kv2"](ctx).chunk(2, -1)
    x = x + ly["out2"](dc.attention_bhld(_heads(q, H), _heads(k, H), _heads(v, H), "int8_turing"))
    return x + dc.int8_geglu_ff(F.layer_norm(x, d, g3, b3), ly["proj"], ly["ff"])


# ---------------------------------------------------------------- work and tolerance

def work(c):
    """Inputs and int8 weights read once, outputs written once; two operations
    per multiply-add of the products (softmax and glue not counted)."""
    kind = c["kind"]
    e = 4 if c["dtype"] == "fp32" else 2
    wbytes = sum(n * k + 4 * n + (e * n if b else 0) for n, k, b in _layer_shapes(c).values())
    if kind == "linear":
        M, K, N = c["M"], c["K"], c["N"]
        return {"bytes": wbytes + e * M * (K + N), "flops": 2 * M * K * N}
    if kind == "geglu":
        M, d = c["M"], c["dim"]
        return {"bytes": wbytes + 2 * e * M * d, "flops": 2 * M * d * 12 * d}
    if kind == "mlp":
        M, d = c["M"], c["dim"]
        return {"bytes": wbytes + 2 * e * M * d, "flops": 2 * M * d * 8 * d}
    if kind == "modlin":
        M, K, N = c["M"], c["K"], c["N"]
        return {"bytes": wbytes + e * (M * (K + N) + 2 * K), "flops": 2 * M * K * N}
    if kind == "gated":
        M, K, N = c["M"], c["K1"] + c["K2"], c["N"]
        return {"bytes": wbytes + e * (M * (K + 2 * N) + N), "flops": 2 * M * K * N}
    if kind == "qknorm":
        n = c["B"] * c["L"] * c["H"] * c["D"]
        return {"bytes": 6 * e * n + 8 * c["L"] * c["D"], "flops": 0}
    if kind == "attn":
        B, H, Lq, Lk, D = c["B"], c["H"], c["Lq"], c["Lk"], c["D"]
        return {"bytes": 2 * e * B * H * D * (Lq + Lk), "flops": 4 * B * H * Lq * Lk * D}
    B, L, d, x = c["B"], c["L"], c["dim"], c["ctx"]
    gemm = 2 * B * (L * d * d * (3 + 1 + 1 + 1 + 12) + x * c["ctx_dim"] * 2 * d)
    return {"bytes": wbytes + e * B * (2 * L * d + x * c["ctx_dim"]), "flops": gemm + 4 * B * L * d * (L + x)}


def tolerance(c):
    """The outputs are rounded to their type once (``linear``, ``modlin``,
    ``attn``) or a few times, and an int8 code on a rounding boundary may fall
    either way where the sums before it are taken in another order."""
    if c["dtype"] == "fp32":
        return {"rel": 2e-4}
    one = 4e-3 if c["dtype"] == "bf16" else 1e-3
    return {"rel": {"linear": one, "modlin": one, "qknorm": one, "gated": 1.5 * one, "mlp": 2.5 * one,
                    "geglu": 2.5 * one, "attn": 2 * one, "block": 6 * one}[c["kind"]]}


# ---------------------------------------------------------------- 64-bit statement

def _hadamard():
    h4 = torch.ones(4, 4, dtype=torch.float64) - 2 * torch.flip(torch.eye(4, dtype=torch.float64), (0,))
    h = h4
    for _ in range(3):
        h = torch.kron(h, h4)
    return (h / 16).cuda()


def _codes(x, group):
    """int8 codes (as float64) and row scales of the rows of x, rotated by ``group``."""
    if group:
        x = (x.reshape(-1, group) @ _hadamard()).view(x.shape)
    s = (x.abs().amax(-1, keepdim=True) / 127).clamp_min(1e-30)
    return torch.round(x / s).clamp(-128, 127), s


def _lin64(x, w, b):
    """The W8A8 layer on rows x (float64): its codes are part of what it computes."""
    q, sx = _codes(x, _group(w.shape[1]))
    qw, sw = _codes(w.double(), _group(w.shape[1]))
    y = (q @ qw.t()) * sx * sw.t()
    return y if b is None else y + b.double()


def _attn64(q, k, v, quantized):
    """(B, L, H, D) float64 q / k / v -> (B, Lq, H * D), one head at a time."""
    B, Lq, H, D = q.shape
    Lk = k.shape[1]
    o = torch.empty(B, Lq, H, D, dtype=torch.float64, device=q.device)
    for b in range(B):
        for h in range(H):
            qh, kh = q[b, :, h], k[b, :, h]
            if quantized:   # q per token, k per 64 keys after taking its mean off
                qc, qs = _codes(qh, 0)
                kh = kh - kh.mean(0, keepdim=True)
                pad = F.pad(kh, (0, 0, 0, -Lk % 64)).view(-1, 64 * D)
                kc, ks = _codes(pad, 0)
                qh, kh = qc * qs, (kc * ks).reshape(-1, D)[:Lk]
            p = torch.softmax((qh @ kh.t()) * D ** -0.5, -1)
            o[b, :, h] = p @ v[b, :, h]
    return o.reshape(B, Lq, H * D)


def exact(c, seed):
    s = _inputs(c, seed)
    w, kind = s["w"], c["kind"]
    f = {k: t.double() for k, t in s.items() if isinstance(t, torch.Tensor)}
    if kind == "linear":
        return _lin64(f["x"], *w["lin"])
    if kind == "geglu":
        a, g = _lin64(f["x"], *w["proj"]).chunk(2, -1)
        return _lin64(a * F.gelu(g), *w["out"])
    if kind == "mlp":
        h = _lin64(f["x"], *w["l1"])
        return _lin64(F.gelu(h, approximate="tanh" if c["act"] == "tanh" else "none"), *w["l2"])
    if kind == "modlin":
        return _lin64(F.layer_norm(f["x"], (c["K"],), eps=1e-6) * f["sc1"] + f["sh"], *w["lin"])
    if kind == "gated":
        x = torch.cat((f["attn"], F.gelu(f["mlp"], approximate="tanh")), -1)
        return f["res"] + f["gate"] * _lin64(x, *w["lin"])
    if kind == "qknorm":
        def side(x, wt):
            n = x * torch.rsqrt(x.square().mean(-1, keepdim=True) + 1e-6) * wt
            pe = f["pe"][:, :, None]
            a, b = n[..., 0::2], n[..., 1::2]
            return torch.stack((pe[..., 0, 0] * a + pe[..., 0, 1] * b, pe[..., 1, 0] * a + pe[..., 1, 1] * b), -1).flatten(-2)
        x = f["qkv"]
        return side(x[:, :, 0], f["wq"]), side(x[:, :, 1], f["wk"]), x[:, :, 2]
    if kind == "attn":
        q, k, v = (f[n].unflatten(-1, (c["H"], c["D"])) for n in "qkv")
        return _attn64(q, k, v, True)
    (g1, b1), (g2, b2), (g3, b3) = [[t.double() for t in n] for n in s["norms"]]
    B, L, d, H = c["B"], c["L"], (c["dim"],), c["H"]

    def lin(name, x):
        return _lin64(x.reshape(-1, x.shape[-1]), *w[name]).unflatten(0, x.shape[:-1])

    def split(t):
        return t.unflatten(-1, (H, -1))

    x = f["x"]
    q, k, v = lin("qkv", F.layer_norm(x, d, g1, b1)).chunk(3, -1)
    x = x + lin("out1", _attn64(split(q), split(k), split(v), True))
    q = lin("q2", F.layer_norm(x, d, g2, b2))
    k, v = lin("kv2", f["ctx"]).chunk(2, -1)
    x = x + lin("out2", _attn64(split(q), split(k), split(v), False))
    a, g = lin("proj", F.layer_norm(x, d, g3, b3)).chunk(2, -1)
    return x + lin("ff", a * F.gelu(g))

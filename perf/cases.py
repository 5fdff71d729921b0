"""The work this package's speed is judged by: its quantized layers, called as a worker's denoiser calls them.

Every case goes through a public entry point, eagerly, with weights laid out once in ``prepare``. The shapes are
the ones the package's benchmark and tests use (the Flux-shaped denoiser: hidden 3072, MLP 12288, 24 heads of
128, 4096 image + 512 text tokens, rank 32, group 64) and ragged sizes around them. ``exact`` restates each path
in 64 bits with plain torch; values the path stores in 16 bits between its layers are rounded there too, since
the next layer's quantizer sees the rounded ones.
"""

from __future__ import annotations

import math
import os
import sys

import torch
import torch.nn.functional as F

_ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
_PKG = os.path.join(_ROOT, "python-gen-worker_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

DEV = "cuda"
BF16, F16 = torch.bfloat16, torch.float16
GROUP = 64
HEAD = 128


# ---------------------------------------------------------------------------
# the cases
# ---------------------------------------------------------------------------

def listed():
    return [
        # one token through an adaLN modulation linear: 57 of these open every denoising step, latency-bound
        {"name": "w4a4_one_token", "kind": "w4a4", "m": 1, "n": 18432, "k": 3072, "rank": 32, "out": "bf16", "gelu": False},
        # a short, odd-length text sequence through a fused QKV projection: a small grid
        {"name": "w4a4_qkv_333", "kind": "w4a4", "m": 333, "n": 9216, "k": 3072, "rank": 32, "out": "bf16", "gelu": False},
        # the headline layer: 4096 image + 512 text tokens through an attention output projection
        {"name": "w4a4_4608", "kind": "w4a4", "m": 4608, "n": 3072, "k": 3072, "rank": 32, "out": "bf16", "gelu": False},
        # the largest single layer: QKV of a batch of images (or one at a higher resolution), fp16 out
        {"name": "w4a4_qkv_16384", "kind": "w4a4", "m": 16384, "n": 9216, "k": 3072, "rank": 32, "out": "fp16", "gelu": False},
        # a block's MLP: fc1, GELU and fc2 with the second quantization fused into the first GEMM
        {"name": "w4a4_mlp_4608", "kind": "mlp", "m": 4608, "d": 3072, "h": 12288, "rank": 32},
        # the operators a worker's own module calls (quantize, low-rank down, GEMM with the low-rank epilogue)
        {"name": "svdq_ops_1024", "kind": "ops", "m": 1024, "n": 9216, "k": 3072, "rank": 32},
        # int8 layers: a small batch of tokens, and the QKV projection of a full image
        {"name": "w8a8_256", "kind": "w8a8", "m": 256, "n": 3072, "k": 3072, "mode": "rowwise", "static": False, "out": "bf16"},
        {"name": "w8a8_qkv_4608", "kind": "w8a8", "m": 4608, "n": 9216, "k": 3072, "mode": "rowwise", "static": False, "out": "bf16"},
        # the modulation linear as an svdq checkpoint stores it (AWQ W4A16), one token
        {"name": "awq_one_token", "kind": "awq", "m": 1, "n": 18432, "k": 3072},
        # a layer of an nvfp4 checkpoint, dynamic second-level scale
        {"name": "nvfp4_4608", "kind": "nvfp4", "m": 4608, "n": 3072, "k": 3072, "static": False},
        # joint attention over image and text tokens
        {"name": "attention_4608", "kind": "attention", "m": 4608, "keys": 4608, "heads": 24},
        # the denoiser end to end with one dual and one single block, all linears W4A4, the blocks' streams on
        {"name": "dit_1_1", "kind": "dit", "img": 4096, "txt": 512},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _mult(rng, lo, hi, step):
    return max(lo // step, _log(rng, lo, hi) // step) * step


_LARGEST = 2.0 * 16384 * 9216 * 3072


def draw(rng):
    while True:
        c = _draw(rng)
        if work(c)["flops"] <= _LARGEST:
            return c


def _draw(rng):
    kind = rng.choice(("w4a4", "w4a4", "w4a4", "mlp", "ops", "w8a8", "w8a8", "awq", "nvfp4", "attention", "dit"))
    m = _log(rng, 1, 16384)
    n, k = _mult(rng, 512, 18432, 16), _mult(rng, 64, 15360, 64)
    rank = rng.choice((16, 32, 32, 64, 128))
    if kind == "w4a4":
        return {"kind": kind, "m": m, "n": n, "k": k, "rank": rng.choice((0, rank, rank)),
                "out": rng.choice(("bf16", "bf16", "fp16")), "gelu": rng.random() < 0.25}
    if kind == "mlp":
        return {"kind": kind, "m": m, "d": _mult(rng, 512, 4096, 128), "h": _mult(rng, 1024, 15360, 128), "rank": rank}
    if kind == "ops":
        return {"kind": kind, "m": m, "n": n, "k": max(k, 256), "rank": rank}
    if kind == "w8a8":
        return {"kind": kind, "m": m, "n": n, "k": max(k, 256), "mode": rng.choice(("rowwise", "rowwise", "pertensor")),
                "static": rng.random() < 0.3, "out": rng.choice(("bf16", "bf16", "fp16"))}
    if kind == "awq":
        return {"kind": kind, "m": _log(rng, 1, 64), "n": n, "k": _mult(rng, 512, 15360, 128)}
    if kind == "nvfp4":
        return {"kind": kind, "m": m, "n": n, "k": max(k, 256), "static": rng.random() < 0.5}
    if kind == "attention":
        return {"kind": kind, "m": _log(rng, 40, 8192), "keys": _log(rng, 40, 8192), "heads": rng.choice((4, 8, 16, 24))}
    return {"kind": "dit", "img": _log(rng, 256, 1024), "txt": _log(rng, 64, 512)}


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------

class _Rand:
    """Seeded draws on the GPU."""

    def __init__(self, seed):
        self.g = torch.Generator(device=DEV).manual_seed(int(seed))

    def normal(self, *shape, std=1.0, dtype=torch.float32):
        return torch.randn(*shape, generator=self.g, device=DEV).mul_(std).to(dtype)

    def uniform(self, *shape):
        return torch.rand(*shape, generator=self.g, device=DEV)

    def activation(self, m, k, frac, scale):
        """bf16 N(0, 1) with a share of outlier channels, as denoiser activations have."""
        x = torch.randn(m, k, generator=self.g, device=DEV)
        hot = torch.randperm(k, generator=self.g, device=DEV)[: int(frac * k)]
        x[:, hot] *= scale
        return x.to(BF16)

    def smooth(self, k):
        return torch.exp(math.log(0.25) + self.uniform(k) * math.log(16.0)).to(BF16)


def _pack(codes):
    c = (codes.to(torch.int16) & 0xF).to(torch.uint8)
    return c[..., 0::2] | (c[..., 1::2] << 4)


def _unpack(packed):
    lo, hi = (packed & 0xF).to(torch.int8), (packed >> 4).to(torch.int8)
    c = torch.stack((lo, hi), dim=-1).reshape(packed.shape[0], -1)
    return torch.where(c >= 8, c - 16, c)


def _int4_weight(r, n, k):
    """N(0, 0.02) weights quantized to int4 codes with fp16 scales per 64 inputs."""
    w = r.normal(n, k, std=0.02).reshape(n, k // GROUP, GROUP)
    s = (w.abs().amax(-1) / 7.0).to(F16)
    q = (w / s.float().unsqueeze(-1)).round_().clamp_(-8, 7)
    return _pack(q.reshape(n, k)), s


def _w4a4_layer(r, n, k, rank, gelu=False, out=BF16):
    from gen_worker_amd import build_svdq_w4a4_linear

    qw, ws = _int4_weight(r, n, k)
    return build_svdq_w4a4_linear(
        qweight=qw, wscales=ws, smooth=r.smooth(k), proj_down=r.normal(k, rank, std=0.02, dtype=BF16) if rank else None,
        proj_up=r.normal(n, rank, std=0.02, dtype=BF16) if rank else None, bias=r.normal(n, std=0.02, dtype=BF16),
        activation="gelu_tanh" if gelu else None, out_dtype=out, device=DEV)


def prepare(case, seed):
    c, r, kind = case, _Rand(seed), case["kind"]
    s = {"kind": kind}
    if kind == "w4a4":
        s["mod"] = _w4a4_layer(r, c["n"], c["k"], c["rank"], c["gelu"], F16 if c["out"] == "fp16" else BF16)
        s["x"] = r.activation(c["m"], c["k"], 0.005, 30.0)
    elif kind == "mlp":
        s["fc1"] = _w4a4_layer(r, c["h"], c["d"], c["rank"], gelu=True)
        s["fc2"] = _w4a4_layer(r, c["d"], c["h"], c["rank"])
        s["x"] = r.activation(c["m"], c["d"], 0.005, 30.0)
    elif kind == "ops":
        import gen_worker_amd  # noqa: F401  (registers the operators)

        qw, ws = _int4_weight(r, c["n"], c["k"])
        s.update(wq=qw.t().contiguous(), ws=ws, smooth=r.smooth(c["k"]), s2=torch.ones((), device=DEV),
                 second=torch.ones(1, device=DEV), down=r.normal(c["k"], c["rank"], std=0.02, dtype=BF16),
                 up=r.normal(c["n"], c["rank"], std=0.02, dtype=BF16), bias=r.normal(c["n"], std=0.02, dtype=BF16),
                 x=r.activation(c["m"], c["k"], 0.005, 30.0))
    elif kind == "w8a8":
        from gen_worker_amd import build_int8_linear

        w = r.normal(c["n"], c["k"], std=0.02)
        ws = (w.abs().amax(-1, keepdim=True) / 127.0).clamp_(min=1e-12)
        s["x"] = r.activation(c["m"], c["k"], 0.01, 20.0)
        static = (s["x"].float().abs().amax() / 127.0).reshape(1, 1) if c["static"] else None
        s["mod"] = build_int8_linear(qweight=(w / ws).round_().clamp_(-127, 127).to(torch.int8), weight_scale=ws,
                                     bias=r.normal(c["n"], std=0.02), compute_dtype=F16 if c["out"] == "fp16" else BF16,
                                     input_scale=static, gemm_mode=c["mode"], device=DEV)
    elif kind == "awq":
        from gen_worker_amd.awq import AwqPackedLinear

        mod = AwqPackedLinear(c["k"], c["n"], bias=True, device=DEV)
        w = r.normal(c["n"], c["k"], std=0.02).reshape(c["n"], -1, GROUP)
        lo, sc = w.amin(-1), ((w.amax(-1) - w.amin(-1)) / 15.0).clamp_(min=1e-6)
        q = ((w - lo.unsqueeze(-1)) / sc.unsqueeze(-1)).round_().clamp_(0, 15).reshape(c["n"], c["k"])
        with torch.no_grad():
            mod.weight.copy_(_pack(q))
            mod.wscales.copy_(sc)
            mod.wzeros.copy_(lo)
            mod.bias.copy_(r.normal(c["n"], std=0.02))
        s["mod"], s["x"] = mod, F.silu(r.normal(c["m"], c["k"])).to(BF16)
    elif kind == "nvfp4":
        from gen_worker_amd import build_nvfp4_linear

        w = r.normal(c["n"], c["k"], std=0.02)
        ws2 = w.abs().amax() / (6.0 * 448.0)
        blocks = w.reshape(c["n"], -1, 16)
        bs = (blocks.abs().amax(-1) / (6.0 * ws2)).clamp_(2.0 ** -9, 448.0).to(torch.float8_e4m3fn)
        q = _e2m1((blocks / (bs.float().unsqueeze(-1) * ws2)).reshape(c["n"], c["k"]))
        s["x"] = r.activation(c["m"], c["k"], 0.01, 20.0)
        static = s["x"].float().abs().amax().reshape(1, 1) / (6.0 * 448.0) if c["static"] else None
        s["packed"] = (q[:, 1::2] << 4 | q[:, 0::2]).contiguous()
        s["bs"], s["ws2"], s["static"] = bs, ws2, static
        s["mod"] = build_nvfp4_linear(s["packed"], bs, ws2, bias=r.normal(c["n"], std=0.02, dtype=BF16), input_scale=static,
                                      device=DEV)
    elif kind == "attention":
        h = c["heads"]
        s["q"], s["k"] = (r.normal(t, h, HEAD, std=1.5, dtype=BF16) for t in (c["m"], c["keys"]))
        s["v"] = r.normal(c["keys"], h, HEAD, dtype=BF16)
    else:
        from gen_worker_amd.flux_dit import FluxDiT, FluxDiTConfig, inputs

        cfg = FluxDiTConfig(n_dual=1, n_single=1, img_tokens=c["img"], txt_tokens=c["txt"])
        s["mod"] = FluxDiT("w4a4", cfg, device=DEV, seed=1000 * (seed % 100000) + 1, lane="int4", streams=2)
        s["in"] = inputs(cfg, device=DEV, seed=seed)
    return s


def run(state):
    s, kind = state, state["kind"]
    with torch.no_grad():
        if kind in ("w4a4", "w8a8", "awq", "nvfp4"):
            return s["mod"](s["x"])
        if kind == "mlp":
            from gen_worker_amd.svdq import svdq_pair_forward

            return svdq_pair_forward(s["x"], s["fc1"], s["fc2"])
        if kind == "ops":
            cg = torch.ops.cozy_gen_worker
            qa, sa = cg.svdq_quant(s["x"], s["smooth"], s["s2"], False)
            la = s["x"] @ s["down"]
            y = cg.svdq_gemm_w4a4_lora(qa, sa, s["wq"], s["ws"], s["s2"], s["second"], la, s["up"], s["bias"])
            return {"y": y, "codes": qa, "scales": sa}
        if kind == "attention":
            from gen_worker_amd.flux_dit import attention

            return attention(s["q"], s["k"], s["v"])
        return s["mod"](*s["in"])


# ---------------------------------------------------------------------------
# what a pass cannot do without
# ---------------------------------------------------------------------------

def _w4a4_work(m, n, k, rank):
    """int4 codes and fp16 group scales of the weight, the 16-bit activation, factors, bias and output."""
    return (2 * m * k + n * k // 2 + 2 * n * k // GROUP + 2 * rank * (n + k) + 2 * (k + n) + 2 * m * n,
            2 * m * n * k + 2 * m * rank * (n + k))


def _attention_work(m, keys, heads):
    return 2 * heads * HEAD * (2 * m + 2 * keys), 4 * m * keys * heads * HEAD


def work(case):
    c, kind = case, case["kind"]
    if kind == "w4a4":
        b, f = _w4a4_work(c["m"], c["n"], c["k"], c["rank"])
    elif kind == "ops":
        b, f = _w4a4_work(c["m"], c["n"], c["k"], c["rank"])
        b += c["m"] * (c["k"] // 2 + 2 * c["k"] // GROUP)
    elif kind == "mlp":
        (b1, f1), (b2, f2) = (_w4a4_work(c["m"], n, k, c["rank"]) for n, k in ((c["h"], c["d"]), (c["d"], c["h"])))
        b, f = b1 + b2 - 4 * c["m"] * c["h"], f1 + f2
    elif kind == "w8a8":
        m, n, k = c["m"], c["n"], c["k"]
        b, f = 2 * m * k + n * k + 8 * n + 2 * m * n, 2 * m * n * k
    elif kind == "awq":
        m, n, k = c["m"], c["n"], c["k"]
        b, f = 2 * m * k + n * k // 2 + 4 * n * k // GROUP + 2 * n + 2 * m * n, 2 * m * n * k
    elif kind == "nvfp4":
        m, n, k = c["m"], c["n"], c["k"]
        b, f = 2 * m * k + 2 * n * k + 2 * n + 2 * m * n, 2 * m * n * k
    elif kind == "attention":
        b, f = _attention_work(c["m"], c["keys"], c["heads"])
    else:
        d, h, i, t = 3072, 12288, c["img"], c["txt"]
        s = i + t
        layers = [(i, d, 64), (t, d, 4096), (1, 2 * d, d), (i, 64, d), (1, 3 * d, d), (s, 3 * d, d), (s, h, d), (s, d, d + h)]
        for rows in (i, t):
            layers += [(1, 6 * d, d), (rows, 3 * d, d), (rows, d, d), (rows, h, d), (rows, d, h)]
        b = 2 * i * 64 + 2 * t * 4096 + 2 * i * 64 + sum(n * k // 2 + 2 * n * k // GROUP + 64 * (n + k) for _, n, k in layers)
        f = sum(_w4a4_work(m, n, k, 32)[1] for m, n, k in layers) + 2 * _attention_work(s, s, 24)[1]
    return {"bytes": int(b), "flops": int(f)}


# A 16-bit result's own rounding is 1.7e-3 of it for bf16 and 2e-4 for fp16 (root mean square); the low-rank
# activation is held in bf16 and adds a little. Behind a second quantizer (the MLP, the blocks) a value at a code
# boundary may take either neighbouring code, one part in fourteen of its group's largest value.
_TOL = {"w4a4": {"rel": 6e-3, "max": 3e-2}, "ops": {"rel": 6e-3, "max": 3e-2, "differ": 1e-5},
        "mlp": {"rel": 2.5e-2, "max": 0.2}, "w8a8": {"rel": 6e-3, "max": 2e-2}, "awq": {"rel": 6e-3, "max": 2e-2},
        "nvfp4": {"rel": 1.5e-2, "max": 4e-2}, "attention": {"rel": 8e-3, "max": 3e-2}, "dit": {"rel": 4.5e-2, "max": 0.4}}


def tolerance(case):
    return dict(_TOL[case["kind"]])


# ---------------------------------------------------------------------------
# the same in 64 bits
# ---------------------------------------------------------------------------

def _bf(x):
    return x.to(torch.float32).to(BF16).double()


def _e2m1(q):
    """e2m1 codes of q: the nearest of 0, .5, 1, 1.5, 2, 3, 4, 6, ties to the even code."""
    a = q.abs()
    c = torch.zeros_like(q, dtype=torch.uint8)
    for i, b in enumerate((0.25, 0.75, 1.25, 1.75, 2.5, 3.5, 5.0)):
        c += (a >= b) if i % 2 else (a > b)
    return c | (q < 0).to(torch.uint8) << 3


def _e2m1_values(codes):
    table = torch.tensor([0, 0.5, 1, 1.5, 2, 3, 4, 6, -0.0, -0.5, -1, -1.5, -2, -3, -4, -6], device=DEV, dtype=torch.float64)
    return table[codes.long()]


def _int4_activation(x, smooth):
    """The smoothed activation quantized to int4 per 64 inputs, dequantized again."""
    m, k = x.shape
    v = _bf(x / smooth).reshape(m, k // GROUP, GROUP)
    s = (v.abs().amax(-1, keepdim=True).float() / 7.0).clamp(2.0 ** -24, 65504.0).to(F16).double()
    return ((v / s).round().clamp(-8, 7) * s).reshape(m, k)


def _deq4(packed, scales):
    w = _unpack(packed).double().reshape(packed.shape[0], -1, GROUP)
    return (w * scales.double().unsqueeze(-1)).reshape(packed.shape[0], -1)


def _gelu(y):
    return 0.5 * y * (1.0 + torch.tanh(math.sqrt(2.0 / math.pi) * (y + 0.044715 * y ** 3)))


def _svdq64(x, mod):
    """One SVDQuant linear in 64 bits; x holds bf16 values in float64."""
    y = _int4_activation(x, mod.smooth_factor.double()) @ _deq4(mod.weight, mod.weight_scale).t()
    y = y * mod.second.double()
    if mod.rank:
        y += (x @ mod.proj_down.double()) @ mod.proj_up.double().t()
    y += mod.bias.double()
    return _gelu(y) if mod.activation else y


def _attention64(q, k, v):
    out = torch.empty(q.shape, device=DEV, dtype=torch.float64)
    for h in range(q.shape[1]):
        p = torch.softmax(q[:, h].double() @ k[:, h].double().t() / math.sqrt(HEAD), dim=-1)
        out[:, h] = p @ v[:, h].double()
    return out.reshape(q.shape[0], -1)


def _dit64(model, latents, text, temb):
    """The denoiser with one dual and one single block; activations between its parts rounded to bf16."""
    lin = lambda x, mod: _bf(_svdq64(x, mod))  # noqa: E731
    t = _bf(F.silu(temb.double()))
    cos, sin = (b.double() for b in (model.cos, model.sin))

    def modulate(x, scale, shift):
        n = F.layer_norm(x, (x.shape[-1],), eps=1e-6)
        return _bf(_bf(_bf(n) * _bf(1 + scale)) + shift)

    def rotate(x, w, at):
        x = x.reshape(x.shape[0], -1, HEAD)
        x = _bf(_bf(x * torch.rsqrt(x.pow(2).mean(-1, keepdim=True) + 1e-6)) * w.double())
        cs, sn = cos[at: at + x.shape[0]], sin[at: at + x.shape[0]]
        a, b = x[..., 0::2], x[..., 1::2]
        return _bf(torch.stack((_bf(a * cs) - _bf(b * sn), _bf(a * sn) + _bf(b * cs)), dim=-1).flatten(-2))

    img, txt = lin(latents.double(), model.x_embedder), lin(text.double(), model.context_embedder)
    blk, c, nt = model.dual[0], img.shape[1], txt.shape[0]
    sides, qs, ks, vs = [], [], [], []
    for x, mod, qkv, qn, kn, at in ((txt, blk.mod_txt, blk.qkv_txt, blk.qn_txt, blk.kn_txt, 0),
                                    (img, blk.mod_img, blk.qkv_img, blk.qn_img, blk.kn_img, nt)):
        sh1, sc1, g1, sh2, sc2, g2 = lin(t, mod).chunk(6, dim=-1)
        y = lin(modulate(x, sc1, sh1), qkv)
        qs.append(rotate(y[:, :c], qn, at))
        ks.append(rotate(y[:, c:2 * c], kn, at))
        vs.append(y[:, 2 * c:].reshape(-1, c // HEAD, HEAD))
        sides.append((g1, sh2, sc2, g2))
    a = _bf(_attention64(torch.cat(qs), torch.cat(ks), torch.cat(vs)))
    done = []
    for x, (g1, sh2, sc2, g2), part, o, fc1, fc2 in ((txt, sides[0], a[:nt], blk.o_txt, blk.fc1_txt, blk.fc2_txt),
                                                     (img, sides[1], a[nt:], blk.o_img, blk.fc1_img, blk.fc2_img)):
        x = _bf(x + _bf(g1 * lin(part, o)))
        done.append(_bf(x + _bf(g2 * lin(lin(modulate(x, sc2, sh2), fc1), fc2))))
    x, blk = torch.cat(done), model.single[0]
    sh, sc, g = lin(t, blk.mod).chunk(3, dim=-1)
    n = modulate(x, sc, sh)
    y = lin(n, blk.qkv)
    a = _bf(_attention64(rotate(y[:, :c], blk.qn, 0), rotate(y[:, c:2 * c], blk.kn, 0), y[:, 2 * c:].reshape(-1, c // HEAD, HEAD)))
    x = _bf(x + _bf(g * lin(torch.cat((a, lin(n, blk.mlp)), dim=-1), blk.proj_out)))
    scale, shift = lin(t, model.norm_out).chunk(2, dim=-1)
    return _svdq64(modulate(x[nt:], scale, shift), model.proj_out)


def exact(case, seed):
    s, kind = prepare(case, seed), case["kind"]
    with torch.no_grad():
        if kind == "w4a4":
            return _svdq64(s["x"].double(), s["mod"])
        if kind == "mlp":
            return _svdq64(_bf(_svdq64(s["x"].double(), s["fc1"])), s["fc2"])
        if kind == "ops":
            x = s["x"].double()
            y = _int4_activation(x, s["smooth"].double()) @ _deq4(s["wq"].t(), s["ws"]).t()
            y += (x @ s["down"].double()) @ s["up"].double().t() + s["bias"].double()
            return {"y": y, "codes": None, "scales": None}
        if kind == "w8a8":
            x, mod = s["x"].double(), s["mod"]
            if mod.input_scale is not None:
                sa = mod.input_scale.double()
            else:
                amax = x.abs().amax() if case["mode"] == "pertensor" else x.abs().amax(-1, keepdim=True)
                sa = (amax.float() / 127.0).clamp(min=1e-12).double()
            q = (x / sa).round().clamp(-127, 127)
            return (q @ mod.weight.double().t()) * sa * mod.weight_scale.double().t() + mod.bias.double()
        if kind == "awq":
            mod = s["mod"]
            codes = torch.stack((mod.weight & 0xF, mod.weight >> 4), dim=-1).reshape(case["n"], -1, GROUP).double()
            w = _bf(codes * mod.wscales.double().unsqueeze(-1) + mod.wzeros.double().unsqueeze(-1))
            return s["x"].double() @ w.reshape(case["n"], -1).t() + mod.bias.double()
        if kind == "nvfp4":
            x = s["x"].float()
            s2 = s["static"] if s["static"] is not None else x.abs().amax() / (6.0 * 448.0)
            xb = x.reshape(case["m"], -1, 16)
            sc = (xb.abs().amax(-1, keepdim=True) / (6.0 * s2)).clamp(2.0 ** -9, 448.0).to(torch.float8_e4m3fn).float()
            xq = (_e2m1_values(_e2m1(xb / (sc * s2))) * sc).reshape(case["m"], -1)
            codes = torch.stack((s["packed"] & 0xF, s["packed"] >> 4), dim=-1).reshape(case["n"], -1, 16)
            w = (_e2m1_values(codes) * s["bs"].double().unsqueeze(-1)).reshape(case["n"], -1)
            return (xq @ w.t()) * (s2.double() * s["ws2"].double()) + s["mod"].bias.double()
        if kind == "attention":
            return _attention64(s["q"], s["k"], s["v"])
        return _dit64(s["mod"], *s["in"])

"""The work this framework is measured on: its layers and blocks as the DiT steps, text encoders
and VAE decoders call them, each through a public entry point, over the sizes they are run at.

A case is a dict of plain values whose "kind" is one of

  linear   a bf16 linear module (ops_impl.linear.ColumnParallelLinear), any number of rows
  fp8      an fp8 linear module (quant.linear.FP8Linear): per-token e4m3 or MXFP8, activations
           quantized in the call
  attn     joint / self attention (ops_impl.attention.attention), unmasked
  padded   joint attention to [image | right-padded text] (ops_impl.attention.joint_ring_attention)
  cross    cross attention of many video tokens to the text (ops_impl.attention.cross_attention)
  t5       a T5 or UMT5 text encoder (text.t5.T5Encoder) of a few layers, bf16 or fp32
  vae      FLUX's VAE decoder (vae.decoder.VaeDecoder)
  flux     a FLUX denoise step (dit.flux.FluxDiT) of one double and two single blocks

The shapes are the repository's model configurations; sizes vary with resolution, prompt length
and clip length. `exact` states each of them in plain torch at 64 bits.
"""

from __future__ import annotations

import dataclasses
import math

import torch
import torch.nn.functional as F

from difflet_amd.backends.rocm.ops_impl import attention as ops_attention
from difflet_amd.backends.rocm.ops_impl.linear import ColumnParallelLinear
from difflet_amd.dit import flux as dit_flux
from difflet_amd.quant.linear import FP8Linear
from difflet_amd.text import t5
from difflet_amd.vae import decoder as vae

DEV = "cuda:0"
BF16 = torch.bfloat16

# (in, out) of the linears: FLUX and Qwen-Image (hidden 3072, MLP 12288, fused single block,
# embedders, per-block modulation), Wan (hidden 5120, FFN 13824), T5-XXL (4096, FFN 10240)
LINEARS = [(3072, 3072), (3072, 9216), (3072, 12288), (12288, 3072), (3072, 21504), (15360, 3072),
           (4096, 3072), (3584, 3072), (64, 3072), (3072, 64), (3072, 18432), (768, 3072),
           (5120, 5120), (5120, 15360), (5120, 13824), (13824, 5120), (4096, 5120), (4096, 10240),
           (10240, 4096), (4096, 12288)]
# the linears that the quantization targets name
FP8_LINEARS = [(3072, 3072), (3072, 9216), (3072, 12288), (12288, 3072), (3072, 21504),
               (15360, 3072), (5120, 5120), (5120, 13824), (13824, 5120), (5120, 10240)]
MOST_FLOPS = 4.6e12  # a drawn case's matrix work stays below the largest listed linear's


def listed():
    return [
        # one request's adaLN modulation of one double block: a single row, bound by the weight
        dict(name="linear_1_row", kind="linear", m=1, k=3072, n=18432),
        # the prompt embedding's projection into FLUX: 512 rows, a small launch
        dict(name="linear_text", kind="linear", m=512, k=4096, n=3072),
        # Qwen-Image's MLP over the 83 x 83 image tokens of 1328 x 1328: a large ragged launch
        dict(name="linear_image", kind="linear", m=6889, k=3072, n=12288),
        # the FLUX single block's output projection at 1024 x 1024, per-token fp8
        dict(name="fp8_tokens", kind="fp8", format="fp8_rowwise", m=4608, k=15360, n=3072),
        # Wan's FFN over the 32760 video tokens of 480p x 81 frames, MXFP8: the largest linear
        dict(name="mx_video", kind="fp8", format="mxfp8", m=32760, k=5120, n=13824),
        # FLUX's joint attention at 1024 x 1024
        dict(name="attn_joint", kind="attn", dtype="bf16", heads=24, s=4608),
        # Qwen-Image's joint attention at 1328 x 1328, a 93-token prompt padded to 256
        dict(name="attn_padded", kind="padded", heads=24, s=6889, text=256, valid=93),
        # Wan's cross attention from 480p x 81 frames to the 512-token prompt
        dict(name="attn_cross", kind="cross", heads=40, s=32760, text=512),
        # FLUX's T5-XXL layers on a 512-token prompt, bf16
        dict(name="t5_bf16", kind="t5", umt5=False, dtype="bf16", layers=2, batch=1, s=512,
             valid=512),
        # Wan's UMT5-XXL layers on a padded prompt of 226 tokens and its negative prompt, fp32
        dict(name="umt5_fp32", kind="t5", umt5=True, dtype="fp32", layers=1, batch=2, s=226,
             valid=61),
        # FLUX's VAE decode to 1024 x 1024
        dict(name="vae_1024", kind="vae", h=128, w=128),
        # the whole call: a denoise step at 1024 x 1024 with a 512-token prompt
        dict(name="flux_step", kind="flux", h=64, w=64, text=512),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["linear", "linear", "fp8", "attn", "padded", "cross", "t5", "t5", "vae",
                       "flux"])
    if kind == "linear":
        k, n = rng.choice(LINEARS)
        return dict(kind=kind, m=_log(rng, 1, min(32760, MOST_FLOPS / (2 * k * n))), k=k, n=n)
    if kind == "fp8":
        k, n = rng.choice(FP8_LINEARS)
        return dict(kind=kind, format=rng.choice(["fp8_rowwise", "mxfp8"]),
                    m=_log(rng, 16, min(32760, MOST_FLOPS / (2 * k * n))), k=k, n=n)
    if kind == "attn":
        return dict(kind=kind, dtype=rng.choice(["bf16", "bf16", "bf16", "fp16"]),
                    heads=rng.choice([24, 40]), s=_log(rng, 300, 12000))
    if kind == "padded":
        text = _log(rng, 32, 1024)
        return dict(kind=kind, heads=24, s=rng.randint(16, 96) * rng.randint(16, 96), text=text,
                    valid=rng.randint(1, text))
    if kind == "cross":
        return dict(kind=kind, heads=40, s=rng.randint(1, 21) * rng.randint(24, 30) *
                    rng.randint(40, 52), text=_log(rng, 64, 512))
    if kind == "t5":
        umt5 = rng.random() < 0.5
        s = _log(rng, 16, 512)
        dtype = rng.choice(["bf16", "bf16", "fp32"])
        return dict(kind=kind, umt5=umt5, dtype=dtype, layers=1 if dtype == "fp32" else 2,
                    batch=rng.randint(1, 2), s=s, valid=rng.randint(1, s) if umt5 else s)
    if kind == "vae":
        return dict(kind=kind, h=2 * rng.randint(12, 64), w=2 * rng.randint(12, 64))
    return dict(kind=kind, h=rng.randint(16, 64), w=rng.randint(16, 64), text=_log(rng, 64, 512))


# ------------------------------------------------------------------------------ inputs
def _gen(seed, salt):
    return torch.Generator(device=DEV).manual_seed(int(seed) * 1009 + salt)


def _randn(seed, salt, *shape, std=1.0, dtype=BF16):
    x = torch.randn(shape, generator=_gen(seed, salt), device=DEV, dtype=torch.float32)
    return (x * std).to(dtype)


def _dense_linear(c, seed):
    """(x, weight, bias) of a linear case: normalized activations, N(0, 0.02) weights."""
    return (_randn(seed, 1, c["m"], c["k"]), _randn(seed, 2, c["n"], c["k"], std=0.02),
            _randn(seed, 3, c["n"], std=0.02))


def _qkv(c, seed):
    """q, k, v [1, heads, tokens, 128] as the model's projections lay them out: one [tokens,
    3 hidden] buffer. q and k are RMS-normalized rows, so scores are of order one."""
    dt = torch.float16 if c.get("dtype") == "fp16" else BF16
    h, s, text = c["heads"], c["s"], c.get("text", 0)
    split = lambda t: [x.view(1, -1, h, 128).transpose(1, 2)  # noqa: E731
                       for x in t.split(h * 128, dim=-1)]
    if c["kind"] == "cross":
        q = split(_randn(seed, 1, s, h * 128, dtype=dt))
        return q + split(_randn(seed, 2, text, 2 * h * 128, dtype=dt))
    out = split(_randn(seed, 1, s, 3 * h * 128, dtype=dt))
    if text:
        out += split(_randn(seed, 2, text, 3 * h * 128, dtype=dt))
    return out


def _t5_parts(c, seed):
    cfg = dataclasses.replace(t5.UMT5_XXL if c["umt5"] else t5.T5_XXL, num_layers=c["layers"])
    dtype = BF16 if c["dtype"] == "bf16" else torch.float32
    ids = torch.randint(3, 32000, (c["batch"], c["s"]), generator=_gen(seed, 1), device=DEV)
    mask = None
    if c["umt5"]:  # right-padded prompts: the first as long as `valid`, the next half of it
        mask = torch.zeros(c["batch"], c["s"], dtype=torch.int64, device=DEV)
        for b in range(c["batch"]):
            mask[b, : max(1, c["valid"] >> b)] = 1
        ids = ids * mask
    return cfg, dtype, t5.random_param_source(cfg, seed, DEV, dtype), ids, mask


def _flux_parts(c, seed):
    cfg = dit_flux.FluxConfig(n_double=1, n_single=2)
    inputs = dict(latents=_randn(seed, 1, 1, c["h"] * c["w"], cfg.in_channels),
                  text=_randn(seed, 2, 1, c["text"], cfg.txt_dim),
                  pooled=_randn(seed, 3, 1, cfg.pooled_dim),
                  timestep=torch.rand(1, generator=_gen(seed, 4), device=DEV),
                  guidance=torch.full((1,), 3.5, device=DEV))
    return cfg, dit_flux.random_param_source(cfg, seed, DEV), inputs


def prepare(case, seed):
    c = case
    if c["kind"] == "linear":
        x, w, b = _dense_linear(c, seed)
        lin = ColumnParallelLinear(c["k"], c["n"], dtype=BF16, device="meta")
        lin.weight = torch.nn.Parameter(w, requires_grad=False)
        lin.bias = torch.nn.Parameter(b, requires_grad=False)
        return c, lin, x
    if c["kind"] == "fp8":
        x, w, b = _dense_linear(c, seed)
        lin = FP8Linear(c["k"], c["n"], device=DEV, format=c["format"])
        lin.load_from_dense_(w, b)
        lin.prepare_kernel_()
        return c, lin, x
    if c["kind"] in ("attn", "cross"):
        return c, _qkv(c, seed), None
    if c["kind"] == "padded":
        return c, _qkv(c, seed), torch.tensor([c["valid"]], dtype=torch.int32, device=DEV)
    if c["kind"] == "t5":
        cfg, dtype, source, ids, mask = _t5_parts(c, seed)
        return c, t5.T5Encoder(cfg, source, dtype=dtype, device=DEV), (ids, mask)
    if c["kind"] == "vae":
        dec = vae.VaeDecoder(vae.FLUX_VAE, vae.random_param_source(vae.FLUX_VAE, seed, DEV, BF16),
                             dtype=BF16, device=DEV)
        return c, dec, _randn(seed, 1, 1, 16, c["h"], c["w"])
    cfg, source, inputs = _flux_parts(c, seed)
    return c, dit_flux.FluxDiT(cfg, source, "bf16", DEV), inputs


def run(state):
    c, obj, x = state
    kind = c["kind"]
    if kind in ("linear", "fp8"):
        return obj(x)
    if kind == "attn":
        return ops_attention.attention(*obj, scale=128 ** -0.5)
    if kind == "cross":
        return ops_attention.cross_attention(*obj, scale=128 ** -0.5)
    if kind == "padded":
        q, k, v, tq, tk, tv = obj
        return ops_attention.joint_ring_attention(q, k, v, tk, tv, scale=128 ** -0.5,
                                                  text_valid_len=x)
    if kind == "t5":
        return obj.forward(*x)
    if kind == "vae":
        return obj.decode(x)
    return obj.forward(x["latents"], x["text"], x["pooled"], x["timestep"], x["guidance"],
                       (c["h"], c["w"]))


# ------------------------------------------------------------------------------ work
def _attn_work(heads, sq, sk, keys=None):
    return dict(flops=4 * heads * 128 * sq * (keys or sk),
                bytes=2 * heads * 128 * (2 * sq + 2 * (keys or sk)))


def work(case):
    c = case
    if c["kind"] in ("linear", "fp8"):
        m, k, n = c["m"], c["k"], c["n"]
        wb = {"fp8_rowwise": n * (k + 4), "mxfp8": n * (k + k // 32)}.get(c.get("format"),
                                                                         2 * n * k)
        return dict(flops=2 * m * k * n, bytes=2 * m * (k + n) + wb + 2 * n)
    if c["kind"] == "attn":
        return _attn_work(c["heads"], c["s"], c["s"])
    if c["kind"] == "cross":
        return _attn_work(c["heads"], c["s"], c["text"])
    if c["kind"] == "padded":  # the padded keys need not be read
        return _attn_work(c["heads"], c["s"], 0, c["s"] + c["valid"])
    if c["kind"] == "t5":
        cfg = t5.T5_XXL
        es = 2 if c["dtype"] == "bf16" else 4
        per = 4 * cfg.d_model * cfg.inner_dim + 3 * cfg.d_model * cfg.d_ff
        rows = c["batch"] * c["s"]
        flops = c["layers"] * (2 * rows * per + 4 * rows * c["s"] * cfg.inner_dim)
        return dict(flops=flops, bytes=es * (c["layers"] * per + 2 * rows * cfg.d_model))
    if c["kind"] == "vae":
        cfg, px = vae.FLUX_VAE, c["h"] * c["w"]
        shapes = vae.param_shapes(cfg)
        flops, at = 0, {"conv_in": 0, "mid_block": 0, "conv_out": 6}
        for name, shp in shapes.items():
            if len(shp) < 2:
                continue
            up = 2 * int(name.split(".")[2]) if "up_blocks" in name else at[name.split(".")[1]]
            if "upsamplers" in name:
                up += 2
            flops += 2 * math.prod(shp) * (px << up)
        flops += 4 * px * px * cfg.block_out_channels[-1]
        return dict(flops=flops, bytes=2 * (sum(math.prod(s) for s in shapes.values())
                                            + 16 * px + 3 * 64 * px))
    cfg = dit_flux.FluxConfig(n_double=1, n_single=2)
    d, f, st, si = cfg.hidden, cfg.mlp, c["text"], c["h"] * c["w"]
    s = st + si
    flops = (2 * s * (4 * d * d + 2 * d * f) * 3 + 3 * 4 * s * s * d
             + 2 * st * cfg.txt_dim * d + 4 * si * cfg.in_channels * d)
    params = sum(math.prod(v) for v in dit_flux.flux_param_shapes(cfg).values())
    return dict(flops=flops, bytes=2 * (params + 2 * si * cfg.in_channels + st * cfg.txt_dim))


def tolerance(case):
    # about four times what the path shows against `exact`: one bf16 (fp16) rounding of the
    # output for a linear, the rounded probabilities too for attention, the roundings of every
    # stored activation for the models
    if case.get("dtype") == "fp32":
        return {"rel": 6e-6, "max": 2e-4}
    if case.get("dtype") == "fp16":
        return {"rel": 0.0012, "max": 0.012}
    return {
        "linear": {"rel": 0.007, "max": 0.03},
        "fp8": {"rel": 0.007, "max": 0.03},
        "attn": {"rel": 0.01, "max": 0.1},
        "padded": {"rel": 0.01, "max": 0.1},
        "cross": {"rel": 0.01, "max": 0.1},
        "t5": {"rel": 0.02, "max": 0.3},
        "vae": {"rel": 0.03, "max": 0.5},
        "flux": {"rel": 0.03, "max": 0.5},
    }[case["kind"]]


# ------------------------------------------------------------------------------ 64 bits
def _mm(x, w, b=None):
    """x w^T + b in 64 bits over the last dim, rows in chunks."""
    w = w.double()
    y = torch.cat([p.double() @ w.t() for p in x.reshape(-1, x.shape[-1]).split(8192)])
    y = y.reshape(*x.shape[:-1], w.shape[0])
    return y if b is None else y + b.double()


def _attend(q, k, v, scale, bias=None):
    """softmax(q k^T scale + bias) v in 64 bits, a head and up to 4096 queries at a time."""
    out = torch.empty(q.shape, dtype=torch.float64, device=q.device)
    for b in range(q.shape[0]):
        for h in range(q.shape[1]):
            kt, vv = k[b, h].double().t().contiguous(), v[b, h].double().contiguous()
            for i in range(0, q.shape[2], 4096):
                s = q[b, h, i:i + 4096].double() @ kt * scale
                if bias is not None:
                    s = s + bias[b if bias.shape[0] > 1 else 0, h, i:i + 4096]
                out[b, h, i:i + 4096] = torch.softmax(s, dim=-1) @ vv
    return out


def _e4m3_rows(x):
    """The per-row e4m3 law: codes (as values) and fp32 scales, amax / 448 per row."""
    x = x.float()
    a = x.abs().amax(dim=-1, keepdim=True).clamp_min(2.0 ** -112)
    q = (x * (torch.full_like(a, 448.0) / a)).clamp(-448, 448).to(torch.float8_e4m3fn)
    return q.double() * (a / torch.full_like(a, 448.0)).double()


def _mx_rows(x):
    """The MXFP8 law: 512-wide tiles (and the rest as one) read in four interleaved quarters,
    each run of 32 sharing the power of two 2^(largest exponent - 7)."""
    out = []
    k = x.shape[-1]
    for k0 in range(0, k, 512):
        t = x[:, k0:k0 + 512].float()
        t = t.reshape(t.shape[0], 4, -1).transpose(1, 2).reshape(t.shape[0], -1, 32).contiguous()
        e = ((t.view(torch.int32) >> 23) & 0xff).amax(dim=-1, keepdim=True) - 7
        scale = torch.exp2(e.clamp(0, 255).double() - 127)
        q = (t.double() / scale).float().clamp(-448, 448).to(torch.float8_e4m3fn)
        q = (q.double() * scale).reshape(x.shape[0], -1, 4).transpose(1, 2)
        out.append(q.reshape(x.shape[0], -1))
    return torch.cat(out, dim=-1)


def _rms(x, w, eps):
    return x * torch.rsqrt(x.square().mean(-1, keepdim=True) + eps) * w.double()


def _gelu(x):
    return F.gelu(x, approximate="tanh")


def _exact_t5(c, seed):
    cfg, dtype, source, ids, mask = _t5_parts(c, seed)
    b, s = ids.shape
    heads = lambda t: t.view(b, s, cfg.num_heads, cfg.d_kv).transpose(1, 2)  # noqa: E731
    rel = torch.arange(s)[None, :] - torch.arange(s)[:, None]
    dist, half = rel.abs(), cfg.relative_attention_num_buckets // 2
    near = half // 2
    far = near + (torch.log(dist.float() / near) / math.log(
        cfg.relative_attention_max_distance / near) * (half - near)).to(torch.long)
    bucket = (rel > 0).long() * half + torch.where(dist < near, dist, far.clamp(max=half - 1))
    x, bias = source("shared.weight")[ids].double(), None
    for i in range(c["layers"]):
        a, m = f"encoder.block.{i}.layer.0.", f"encoder.block.{i}.layer.1."
        if bias is None or cfg.per_layer_bias:
            table = source(a + "SelfAttention.relative_attention_bias.weight").double()
            bias = table[bucket.to(DEV)].permute(2, 0, 1)[None]
            if mask is not None:
                bias = bias.masked_fill(mask[:, None, None, :] == 0, torch.finfo(torch.float32).min)
        n = _rms(x, source(a + "layer_norm.weight"), cfg.layer_norm_epsilon)
        q, k, v = (heads(_mm(n, source(a + f"SelfAttention.{p}.weight"))) for p in "qkv")
        o = _attend(q, k, v, 1.0, bias).transpose(1, 2).reshape(b, s, -1)
        x = x + _mm(o, source(a + "SelfAttention.o.weight"))
        n = _rms(x, source(m + "layer_norm.weight"), cfg.layer_norm_epsilon)
        g = _gelu(_mm(n, source(m + "DenseReluDense.wi_0.weight")))
        x = x + _mm(g * _mm(n, source(m + "DenseReluDense.wi_1.weight")),
                    source(m + "DenseReluDense.wo.weight"))
    return _rms(x, source("encoder.final_layer_norm.weight"), cfg.layer_norm_epsilon)


def _exact_vae(c, seed):
    cfg = vae.FLUX_VAE
    source = vae.random_param_source(cfg, seed, DEV, BF16)
    get = lambda n: source(n).double()  # noqa: E731

    def conv(x, name):  # x [C, H, W]; 3 x 3 (padding 1) or 1 x 1, bands of rows at a time
        w, b = get(name + ".weight"), get(name + ".bias")
        ch, hh, ww = x.shape
        if w.shape[-1] == 1:
            return (w.view(w.shape[0], ch) @ x.view(ch, -1) + b[:, None]).view(-1, hh, ww)
        xp, wf, out = F.pad(x, (1, 1, 1, 1)), w.reshape(w.shape[0], -1), []
        band = max(1, (1 << 28) // (9 * ch * ww))
        for y in range(0, hh, band):
            n = min(band, hh - y)
            cols = torch.stack([xp[:, y + ky:y + ky + n, kx:kx + ww]
                                for ky in range(3) for kx in range(3)], dim=1)
            out.append((wf @ cols.reshape(9 * ch, -1)).view(-1, n, ww))
        return torch.cat(out, dim=1) + b[:, None, None]

    def norm(x, name, silu=True):
        y = x.reshape(cfg.norm_num_groups, -1)
        y = (y - y.mean(1, keepdim=True)) * torch.rsqrt(y.var(1, unbiased=False, keepdim=True)
                                                        + vae.EPS)
        y = y.view(x.shape) * get(name + ".weight")[:, None, None] + get(name + ".bias")[:, None, None]
        return y * torch.sigmoid(y) if silu else y

    def resnet(x, pre):
        h = conv(norm(x, pre + ".norm1"), pre + ".conv1")
        h = conv(norm(h, pre + ".norm2"), pre + ".conv2")
        short = pre + ".conv_shortcut"
        return h + (conv(x, short) if short + ".weight" in shapes else x)

    shapes = vae.param_shapes(cfg)
    x = conv(_randn(seed, 1, 16, c["h"], c["w"]).double(), "decoder.conv_in")
    x = resnet(x, "decoder.mid_block.resnets.0")
    a = "decoder.mid_block.attentions.0"
    n = norm(x, a + ".group_norm", silu=False).reshape(x.shape[0], -1).t()
    q, k, v = (_mm(n, get(f"{a}.{p}.weight"), get(f"{a}.{p}.bias"))[None, None]
               for p in ("to_q", "to_k", "to_v"))
    o = _mm(_attend(q, k, v, x.shape[0] ** -0.5)[0, 0], get(a + ".to_out.0.weight"),
            get(a + ".to_out.0.bias"))
    x = resnet(x + o.t().reshape(x.shape), "decoder.mid_block.resnets.1")
    last = len(cfg.block_out_channels) - 1
    for i in range(last + 1):
        for j in range(cfg.layers_per_block + 1):
            x = resnet(x, f"decoder.up_blocks.{i}.resnets.{j}")
        if i < last:
            x = x.repeat_interleave(2, dim=1).repeat_interleave(2, dim=2)
            x = conv(x, f"decoder.up_blocks.{i}.upsamplers.0.conv")
    return conv(norm(x, "decoder.conv_norm_out"), "decoder.conv_out")[None]


def _exact_flux(c, seed):
    cfg, source, inp = _flux_parts(c, seed)
    d, eps, st = cfg.hidden, 1e-6, c["text"]
    get = lambda n: source(n).double()  # noqa: E731
    lin = lambda x, n: _mm(x, source(n + ".weight"), source(n + ".bias"))  # noqa: E731
    silu = lambda x: x * torch.sigmoid(x)  # noqa: E731

    def norm(x, shift, scale):
        y = x - x.mean(-1, keepdim=True)
        y = y * torch.rsqrt(y.square().mean(-1, keepdim=True) + eps)
        return y * (1 + scale) + shift

    def embed(t, pre):  # the step scales timestep and guidance by 1000 in bf16
        ang = (t.to(BF16) * 1000).double()[:, None] * torch.exp(
            -math.log(10000) * torch.arange(128, dtype=torch.float64, device=DEV) / 128)
        return mlp(torch.cat([ang.cos(), ang.sin()], dim=-1), pre)

    def mlp(x, pre):
        return lin(silu(lin(x, f"time_text_embed.{pre}.linear_1")),
                   f"time_text_embed.{pre}.linear_2")

    temb = (embed(inp["timestep"], "timestep_embedder") + embed(inp["guidance"], "guidance_embedder")
            + mlp(inp["pooled"], "text_embedder"))
    # positions (0, row, column), zero for the text, on axes of 16, 56 and 56 dims
    yy, xx = torch.meshgrid(torch.arange(c["h"]), torch.arange(c["w"]), indexing="ij")
    pos = F.pad(torch.stack([yy, xx], -1).reshape(-1, 2).to(DEV).double(), (1, 0, st, 0))
    ang = torch.cat([torch.outer(pos[:, i], 10000.0 ** (-torch.arange(
        0, ax, 2, dtype=torch.float64, device=DEV) / ax)) for i, ax in enumerate(cfg.axes)], 1)
    cos, sin = ang.cos(), ang.sin()

    def rope(x, w):  # [S, D] -> [heads, S, 128], normalized and rotated
        x = _rms(x.view(-1, cfg.heads, 128), w, eps).transpose(0, 1)
        a, b = x[..., 0::2], x[..., 1::2]
        return torch.stack([a * cos - b * sin, b * cos + a * sin], -1).flatten(-2)

    def attend(q, k, v):
        v = v.view(-1, cfg.heads, 128).transpose(0, 1)
        o = _attend(q[None], k[None], v[None], 128 ** -0.5)[0]
        return o.transpose(0, 1).reshape(-1, d)

    img, txt = lin(inp["latents"][0], "x_embedder"), lin(inp["text"][0], "context_embedder")
    for i in range(cfg.n_double):
        p = f"transformer_blocks.{i}."
        a = p + "attn."
        m = lin(silu(temb), p + "norm1.linear").chunk(6, -1)
        mc = lin(silu(temb), p + "norm1_context.linear").chunk(6, -1)
        n, nc = norm(img, m[0], m[1]), norm(txt, mc[0], mc[1])
        w2 = lambda t, r: get(a + t)[None].expand(r, -1)[:, None]  # noqa: E731
        both = lambda t, u: torch.cat([w2(t, st), w2(u, img.shape[0])])  # noqa: E731
        cat = lambda t, u: torch.cat([lin(nc, a + t), lin(n, a + u)])  # noqa: E731
        o = attend(rope(cat("add_q_proj", "to_q"), both("norm_added_q.weight", "norm_q.weight")),
                   rope(cat("add_k_proj", "to_k"), both("norm_added_k.weight", "norm_k.weight")),
                   cat("add_v_proj", "to_v"))
        img = img + m[2] * lin(o[st:], a + "to_out.0")
        txt = txt + mc[2] * lin(o[:st], a + "to_add_out")
        img = img + m[5] * lin(_gelu(lin(norm(img, m[3], m[4]), p + "ff.net.0.proj")), p + "ff.net.2")
        txt = txt + mc[5] * lin(_gelu(lin(norm(txt, mc[3], mc[4]), p + "ff_context.net.0.proj")),
                                p + "ff_context.net.2")
    h = torch.cat([txt, img])
    for i in range(cfg.n_single):
        p = f"single_transformer_blocks.{i}."
        shift, scale, gate = lin(silu(temb), p + "norm.linear").chunk(3, -1)
        n = norm(h, shift, scale)
        q = rope(lin(n, p + "attn.to_q"), get(p + "attn.norm_q.weight"))
        k = rope(lin(n, p + "attn.to_k"), get(p + "attn.norm_k.weight"))
        o = attend(q, k, lin(n, p + "attn.to_v"))
        h = h + gate * lin(torch.cat([o, _gelu(lin(n, p + "proj_mlp"))], -1), p + "proj_out")
    scale, shift = lin(silu(temb), "norm_out.linear").chunk(2, -1)
    return lin(norm(h[st:], shift, scale), "proj_out")[None]


def exact(case, seed):
    c = case
    if c["kind"] == "linear":
        return _mm(*_dense_linear(c, seed))
    if c["kind"] == "fp8":
        x, w, b = _dense_linear(c, seed)
        law = _mx_rows if c["format"] == "mxfp8" else _e4m3_rows
        w = law(w)
        return torch.cat([law(p) @ w.t() + b.double() for p in x.split(4096)])
    if c["kind"] in ("attn", "cross"):
        return _attend(*_qkv(c, seed), 128 ** -0.5)
    if c["kind"] == "padded":
        q, k, v, _, tk, tv = _qkv(c, seed)
        n = c["valid"]
        return _attend(q, torch.cat([k, tk[:, :, :n]], 2), torch.cat([v, tv[:, :, :n]], 2),
                       128 ** -0.5)
    if c["kind"] == "t5":
        return _exact_t5(c, seed)
    if c["kind"] == "vae":
        return _exact_vae(c, seed)
    return _exact_flux(c, seed)

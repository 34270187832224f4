"""The ping-pong attention's instance for key windows and two key segments, against the oracle's
fp32 attention on the concatenated keys: segment lengths around the 64-key tile, windows that cut
tiles, cover nothing, or differ per query, the split schedule, strided and misaligned inputs.

Tolerance: P and the output are each rounded to 16 bits (bf16: relative error up to 2^-9, fp16
2^-12), everything else is fp32, so rel L2 stays below 2^-9 + 2^-9 (2^-12 + 2^-12)."""

import math

import pytest
import torch

from oracle import ops

pytestmark = pytest.mark.gpu
SCALE = 1 / math.sqrt(128)


def rel_l2(a, b):
    a, b = a.detach().float().cpu(), b.detach().float().cpu()
    return ((a - b).norm() / b.norm().clamp_min(1e-30)).item()


TOL = {torch.bfloat16: 2.0 ** -8, torch.float16: 2.0 ** -11}


def _rand(g, b, h, s, dtype):
    """[b, h, s, 128] as a view of one [b, s, 3 h 128] projection."""
    x = torch.randn(b, s, 3 * h * 128, generator=g).to(dtype)
    return [t.view(b, s, h, 128).transpose(1, 2) for t in x.split(h * 128, dim=-1)]


def _ref(q, k, v, lo=None, hi=None):
    bounds = {} if hi is None else dict(bound_min=lo, bound_max=hi)
    return ops.attention(q.float(), k.float(), v.float(), scale=SCALE, **bounds)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("s1,s2,counts", [
    (1, 1, [0, 1]), (63, 65, [65, 1]), (64, 64, [64, 0]), (65, 63, [-70, 33]), (130, 1, [1, -1]),
    (1100, 40, [7, 40]), (1088, 0, [0, -40]), (200, 300, None), (256, 1000, [64, 999]),
])
def test_joint_attention_segments(gpu, dtype, s1, s2, counts):
    """Windows from "everything" down to none (a fully masked row averages every value)."""
    from difflet_amd.backends.rocm.ops_impl import attention as A

    print(f"joint {s1} + {s2} {counts} {dtype}", flush=True)
    g = torch.Generator().manual_seed(s1 * 7 + s2)
    q, k, v = _rand(g, 2, 3, s1, dtype)
    _, k2, v2 = _rand(g, 2, 3, s2, dtype)
    keys, vals = torch.cat([k, k2], 2), torch.cat([v, v2], 2)
    hi = valid = None
    if counts is not None:
        valid = torch.tensor(counts, dtype=torch.int32)
        hi = (s1 + valid).view(2, 1, 1, 1).expand(2, 3, s1, 1)
        valid = valid.to(gpu)
    ref = _ref(q, keys, vals, None if hi is None else torch.zeros_like(hi), hi)
    G = lambda t: t.to(gpu)  # noqa: E731
    out = A.joint_ring_attention(G(q), G(k), G(v), G(k2), G(v2), scale=SCALE, text_valid_len=valid)
    assert rel_l2(out, ref) < TOL[dtype]
    # rows the kernel cannot address where they lie: base 2 bytes off, a row stride of 129
    odd = lambda t: torch.cat([t, t[..., :1]], -1).to(gpu)[..., :128]  # noqa: E731
    out2 = A.joint_ring_attention(G(q), odd(k), odd(v), odd(k2), odd(v2), scale=SCALE,
                                  text_valid_len=valid)
    assert torch.equal(out, out2)


def test_joint_attention_split_schedule(gpu):
    """More tiles than compute units and a last wave under 90 % full: cut tiles, both segments."""
    from difflet_amd.backends.rocm.ops_impl import attention as A

    g = torch.Generator().manual_seed(3)
    q, k, v = _rand(g, 1, 20, 3400, torch.bfloat16)
    _, k2, v2 = _rand(g, 1, 20, 200, torch.bfloat16)
    hi = torch.full((1, 20, 3400, 1), 3400 + 77)
    ref = _ref(q, torch.cat([k, k2], 2), torch.cat([v, v2], 2), torch.zeros_like(hi), hi)
    G = lambda t: t.to(gpu)  # noqa: E731
    out = A.joint_ring_attention(G(q), G(k), G(v), G(k2), G(v2), scale=SCALE,
                                 text_valid_len=torch.tensor([77], device=gpu))
    assert rel_l2(out, ref) < TOL[torch.bfloat16]


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("scale", [SCALE, 3.0, 1e-3])
def test_bounded_attention_per_query_windows(gpu, dtype, scale):
    """Per-query windows over 1025 keys on the ping-pong kernel: edges at tile borders, empty and
    reversed windows, windows past either end."""
    from difflet_amd.backends.rocm.ops_impl import attention as A

    print(f"bounded {dtype} {scale}", flush=True)
    g = torch.Generator().manual_seed(11)
    q, _, _ = _rand(g, 1, 2, 300, dtype)
    _, k, v = _rand(g, 1, 2, 1025, dtype)
    lo = torch.randint(-100, 1100, (1, 2, 300, 1), generator=g)
    hi = lo + torch.randint(-50, 700, (1, 2, 300, 1), generator=g)
    for i, (a, b) in enumerate([(0, 64), (64, 128), (63, 65), (1024, 1025), (0, 1025), (5, 5),
                                (1025, 2000), (-9, 0), (0, 1)]):
        lo[..., i, :], hi[..., i, :] = a, b
    ref = ops.attention(q.float(), k.float(), v.float(), scale=scale, bound_min=lo, bound_max=hi)
    out = A.attention(q.to(gpu), k.to(gpu), v.to(gpu), scale=scale, bound_min=lo.to(gpu),
                      bound_max=hi.to(gpu))
    assert rel_l2(out, ref) < TOL[dtype]


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("d", [64, 128])
@pytest.mark.parametrize("sq,sk,padded", [(1, 1, False), (33, 64, True), (128, 65, True),
                                          (129, 200, False), (226, 226, True)])
def test_relative_bias_attention(gpu, dtype, d, sq, sk, padded):
    """The relative-position bias read by its diagonals, with key padding (a batch element whose
    keys are all padding averages v), against the expanded additive mask. fp32: sums of d and sk
    terms in fp32, rel L2 < 1e-5."""
    from difflet_amd import kernels

    print(f"relative bias {dtype} {d} {sq} {sk} {padded}", flush=True)
    g = torch.Generator().manual_seed(sq + sk)
    q, k, v = (torch.randn(2, 3, s, d, generator=g).to(dtype) for s in (sq, sk, sk))
    diag = torch.randn(3, sq + sk + 2, generator=g)
    j = torch.arange(sk)[None, :] - torch.arange(sq)[:, None] + sq - 1
    bias, keep = diag[:, j][None].expand(2, -1, -1, -1), None
    if padded:
        keep = torch.rand(2, sk, generator=g) > 0.4
        keep[1] = False
        bias = bias.masked_fill(~keep[:, None, None, :], torch.finfo(torch.float32).min)
    ref = ops.attention(q.float(), k.float(), v.float(), scale=0.3, attention_mask=bias)
    out = kernels.attention_relative_bias(q.to(gpu), k.to(gpu), v.to(gpu), scale=0.3,
                                          diag=diag.to(gpu),
                                          key_keep=None if keep is None else keep.to(gpu))
    assert rel_l2(out, ref) < TOL.get(dtype, 1e-5)

"""The rocm kernels as torch custom operators (namespace ``difflet_rocm``).

The op modules call the HIP kernels through these operators, not through ctypes directly: to
``torch.compile`` each one is a single opaque node with a fake (meta) implementation that gives
the output's shape and dtype, so Dynamo traces a block that uses them without a graph break and
Inductor compiles the torch code around them. This is what the reference's CUDA and TPU backends
do for their own fused kernels (difflet/backends/cuda/hunyuan_video_15/modeling.py:73-100,
difflet/backends/tpu/ops_impl/collectives.py:99-150).

A custom_op's Python layers cost about 10 us a call, as much as a short linear on the device. So
the operators of the linears and the attention each have a twin, ``<name>_infer``, with the same
implementation and fake but a bare dispatcher registration; the functions here call the twin for
device tensors that need no gradient, in plain eager execution (_eager). Everything else (compiled
and recorded graphs, functorch transforms, inputs that require grad, whose backward custom_op
refuses, host tensors) goes to the custom_op. The twin's own backward refuses too.

Every operator is functional: it allocates and returns a new contiguous tensor and mutates no
argument. Shape and dtype checks that raise for unsupported inputs stay in the op modules, so
they also run while tracing.
"""

from __future__ import annotations

from typing import Optional

import torch
import torch.nn.functional as F

from difflet_amd import kernels

Tensor = torch.Tensor

_INFER = torch.library.Library("difflet_rocm", "FRAGMENT")  # noqa: TOR901


def _infer_twin(op, impl, fake):
    """The operator <op's name>_infer of op's signature: impl on the device, fake for tracing, and
    as the custom_op no formula for the backward."""
    schema = op._opoverload._schema
    name = schema.name.split("::")[1]
    _INFER.define(str(schema).split("::")[1].replace(f"{name}(", f"{name}_infer(", 1))
    _INFER.impl(f"{name}_infer", impl, "CUDA")
    torch.library.register_fake(f"difflet_rocm::{name}_infer", fake, lib=_INFER)

    def no_backward(ctx, *grads):
        raise RuntimeError(f"difflet_rocm::{name} has no backward: it runs inference only")

    torch.library.register_autograd(f"difflet_rocm::{name}_infer", no_backward, lib=_INFER)
    return getattr(torch.ops.difflet_rocm, f"{name}_infer").default


def _plain(*tensors: Optional[Tensor]) -> bool:
    """Device tensors, none of which needs a gradient."""
    grad = torch.is_grad_enabled()
    for t in tensors:
        if t is not None and (not t.is_cuda or (grad and t.requires_grad)):
            return False
    return True


_functorch_level = torch._C._functorch.peek_interpreter_stack
_dispatch_modes = torch._C._len_torch_dispatch_stack
_pre_dispatch_modes = torch._ops._len_torch_dispatch_stack_pre_dispatch
_jit_trace = torch._C._is_tracing
_forward_ad = torch.autograd.forward_ad
_TENSORS = frozenset((Tensor, torch.nn.Parameter, type(None)))
#: a twin is called at the device's key, below autograd as custom_op's implementations run: the
#: kernel there is only for calls that come another way
_DEVICE = torch._C.DispatchKeySet(torch._C.DispatchKey.CUDA)


def _eager() -> bool:
    """Nothing records, transforms or differentiates the calls: no torch.compile, jit or dispatch
    mode (make_fx, fake tensors), no functorch level (a batched tensor denies the gradient that
    the tensor under it needs), no forward-mode level."""
    return not (torch.compiler.is_compiling() or _functorch_level() is not None
                or _dispatch_modes() or _pre_dispatch_modes() or _jit_trace()
                or _forward_ad._current_level >= 0)


def _inference(*tensors: Optional[Tensor]) -> bool:
    """Whether a twin can stand in for its custom_op: plain eager execution, plain device tensors
    (no subclasses), no gradient."""
    return _eager() and _TENSORS.issuperset(map(type, tensors)) and _plain(*tensors)


# ---------------------------------------------------------------------------------- attention
def _attention_impl(q: Tensor, k: Tensor, v: Tensor, scale: float, causal: bool,
                    attention_mask: Optional[Tensor], bound_min: Optional[Tensor],
                    bound_max: Optional[Tensor]) -> Tensor:
    """difflet_rocm_attention: (B, H, S, D) or (B*H, S, D) q/k/v, output in v's dtype."""
    return kernels.attention(q, k, v, scale=scale, causal=causal, attention_mask=attention_mask,
                             bound_min=bound_min, bound_max=bound_max).contiguous()


def _attention_fake(q, k, v, scale, causal, attention_mask, bound_min, bound_max):
    return q.new_empty((*q.shape[:-1], v.shape[-1]), dtype=v.dtype)


_attention_op = torch.library.custom_op("difflet_rocm::attention", _attention_impl, mutates_args=())
_attention_op.register_fake(_attention_fake)
_attention_infer = _infer_twin(_attention_op, _attention_impl, _attention_fake)


def attention(q: Tensor, k: Tensor, v: Tensor, scale: float, causal: bool,
              attention_mask: Optional[Tensor], bound_min: Optional[Tensor],
              bound_max: Optional[Tensor]) -> Tensor:
    if _inference(q, k, v, attention_mask, bound_min, bound_max):
        return _attention_infer.redispatch(_DEVICE, q, k, v, scale, causal, attention_mask,
                                           bound_min, bound_max)
    return _attention_op(q, k, v, scale, causal, attention_mask, bound_min, bound_max)


def _attention_joint_impl(q: Tensor, k: Tensor, v: Tensor, k2: Tensor, v2: Tensor, scale: float,
                          key_count: Optional[Tensor], count_offset: int) -> Tensor:
    """difflet_rocm_attention_joint: (B, H, S, 128) q over the keys [k | k2], the first
    key_count[b] + count_offset of them when key_count is given."""
    return kernels.attention_joint(q, k, v, k2, v2, scale=scale, key_count=key_count,
                                   count_offset=count_offset)


def _attention_joint_fake(q, k, v, k2, v2, scale, key_count, count_offset):
    return q.new_empty(q.shape)


_attention_joint_op = torch.library.custom_op("difflet_rocm::attention_joint",
                                              _attention_joint_impl, mutates_args=())
_attention_joint_op.register_fake(_attention_joint_fake)
_attention_joint_infer = _infer_twin(_attention_joint_op, _attention_joint_impl,
                                     _attention_joint_fake)


def attention_joint(q: Tensor, k: Tensor, v: Tensor, k2: Tensor, v2: Tensor, scale: float,
                    key_count: Optional[Tensor], count_offset: int) -> Tensor:
    if _inference(q, k, v, k2, v2, key_count):
        return _attention_joint_infer.redispatch(_DEVICE, q, k, v, k2, v2, scale, key_count,
                                                 count_offset)
    return _attention_joint_op(q, k, v, k2, v2, scale, key_count, count_offset)


# ------------------------------------------------------------------------------------- linear
#: up to this many input rows a linear may run on the GEMV kernel (HBM-bound on the weight)
GEMV_ROWS = 8


def _gemv_stages(m: int, k: int) -> bool:
    """The GEMV kernel stages m rows of x in LDS: m (rounded up to 1, 2, 4 or 8) x k <= 16384."""
    return (m <= GEMV_ROWS and k % 8 == 0
            and {1: 1, 2: 2}.get(m, 4 if m <= 4 else 8) * k <= 16384)


def _gemv_fits(m: int, k: int, n: int) -> bool:
    """Whether the GEMV is the faster kernel. From two rows on its reads of x bound it (3072 x 18432:
    2 rows 34 us, 4 rows 56, the GEMM's 64-row tiles 26), so there it keeps the widths the GEMM
    would have to pad the weight for."""
    return _gemv_stages(m, k) and (m == 1 or k % 64 != 0 or n % 4 != 0)


def _linear_impl(x: Tensor, w: Tensor, bias: Optional[Tensor], out_features: int) -> Tensor:
    """y [M, out_features] bf16 = x [M, K'] @ w[:out_features, :K']^T + bias, where w [N', K'] may be
    the zero-padded weight (K' a multiple of 64, N' of 4); x is padded to K' here."""
    m, kx = x.shape
    n_pad, k_pad = w.shape
    if m == 0:
        return x.new_empty((0, out_features), dtype=torch.bfloat16)
    as_given = m <= GEMV_ROWS and n_pad == out_features and k_pad == kx
    if as_given and _gemv_fits(m, kx, n_pad):
        return kernels.gemv(x, w, bias)
    try:
        return _linear_gemm(x, w, bias, out_features)
    except (TypeError, ValueError, NotImplementedError):
        # what the GEMM refuses (rows of x that overlap or are off 16 bytes, a bias off 8, 4 GiB and
        # more) the GEMV takes: it copies x, reads the bias value by value, addresses in 64 bits
        if as_given and _gemv_stages(m, kx):
            return kernels.gemv(x, w, bias)
        raise


def _linear_gemm(x: Tensor, w: Tensor, bias: Optional[Tensor], out_features: int) -> Tensor:
    kx, (n_pad, k_pad) = x.shape[1], w.shape
    if kx != k_pad:
        x = F.pad(x, (0, k_pad - kx))
    if bias is not None and bias.shape[0] != n_pad:
        bias = F.pad(bias, (0, n_pad - bias.shape[0]))
    y = kernels.gemm_call("bf16", x if x.stride(-1) == 1 else x.contiguous(), w, bias)
    return y if n_pad == out_features else y[:, :out_features].contiguous()


def _linear_fake(x, w, bias, out_features):
    return x.new_empty((x.shape[0], out_features), dtype=torch.bfloat16)


_linear_op = torch.library.custom_op("difflet_rocm::linear", _linear_impl, mutates_args=())
_linear_op.register_fake(_linear_fake)
_linear_infer = _infer_twin(_linear_op, _linear_impl, _linear_fake)


def linear(x: Tensor, w: Tensor, bias: Optional[Tensor], out_features: int) -> Tensor:
    if _inference(x, w, bias):
        return _linear_infer.redispatch(_DEVICE, x, w, bias, out_features)
    return _linear_op(x, w, bias, out_features)


def _linear_f32_impl(x: Tensor, w: Tensor, bias: Optional[Tensor], out_features: int) -> Tensor:
    """y [M, out_features] fp32 = x [M, K'] @ w[:out_features, :K']^T + bias on the fp32 GEMM,
    where w [N', K'] may be the zero-padded weight (K' and N' multiples of 4)."""
    m, kx = x.shape
    n_pad, k_pad = w.shape
    if m == 0:
        return x.new_empty((0, out_features), dtype=torch.float32)
    if kx != k_pad:
        x = F.pad(x, (0, k_pad - kx))
    if bias is not None and bias.shape[0] != n_pad:
        bias = F.pad(bias, (0, n_pad - bias.shape[0]))
    y = kernels.gemm_f32(x.contiguous(), w, None if bias is None else bias.contiguous(),
                         workspace="call")
    return y if n_pad == out_features else y[:, :out_features].contiguous()


def _linear_f32_fake(x, w, bias, out_features):
    return x.new_empty((x.shape[0], out_features), dtype=torch.float32)


_linear_f32_op = torch.library.custom_op("difflet_rocm::linear_f32", _linear_f32_impl,
                                         mutates_args=())
_linear_f32_op.register_fake(_linear_f32_fake)
_linear_f32_infer = _infer_twin(_linear_f32_op, _linear_f32_impl, _linear_f32_fake)


def linear_f32(x: Tensor, w: Tensor, bias: Optional[Tensor], out_features: int) -> Tensor:
    if _inference(x, w, bias):
        return _linear_f32_infer.redispatch(_DEVICE, x, w, bias, out_features)
    return _linear_f32_op(x, w, bias, out_features)


def _fp8_linear_impl(x: Tensor, w_kernel: Tensor, w_scale: Tensor, bias: Optional[Tensor],
               mx: bool) -> Tensor:
    """The fp8 twins' matmul: x [M, K] bf16 quantized per token (per-channel weights) or per MX
    block in swizzle order (mx), then the fp8 GEMM with fp32 accumulation, bf16 [M, N] out."""
    if mx:
        aq, asc = kernels.quantize_mxfp8(x, swizzled=True)
    else:
        aq, asc = kernels.quantize_fp8_rowwise(x)
    return kernels.gemm_call("mx" if mx else "fp8", aq, w_kernel, bias, asc, w_scale)


def _fp8_linear_fake(x, w_kernel, w_scale, bias, mx):
    return x.new_empty((x.shape[0], w_kernel.shape[0]), dtype=torch.bfloat16)


_fp8_linear_op = torch.library.custom_op("difflet_rocm::fp8_linear", _fp8_linear_impl,
                                         mutates_args=())
_fp8_linear_op.register_fake(_fp8_linear_fake)
_fp8_linear_infer = _infer_twin(_fp8_linear_op, _fp8_linear_impl, _fp8_linear_fake)


def fp8_linear(x: Tensor, w_kernel: Tensor, w_scale: Tensor, bias: Optional[Tensor],
               mx: bool) -> Tensor:
    if _inference(x, w_kernel, w_scale, bias):
        return _fp8_linear_infer.redispatch(_DEVICE, x, w_kernel, w_scale, bias, mx)
    return _fp8_linear_op(x, w_kernel, w_scale, bias, mx)


# ---------------------------------------------------------------------------- norms, rotary
@torch.library.custom_op("difflet_rocm::rms_norm", mutates_args=())
def rms_norm(x: Tensor, weight: Optional[Tensor], eps: float) -> Tensor:
    """difflet_rocm_rms_norm: the fp32 RMSNorm law, one cast back to x's dtype."""
    return kernels.rms_norm(x, weight, eps)


@rms_norm.register_fake
def _(x, weight, eps):
    return x.new_empty(x.shape)


@torch.library.custom_op("difflet_rocm::layer_norm", mutates_args=())
def layer_norm(x: Tensor, weight: Optional[Tensor], bias: Optional[Tensor], eps: float) -> Tensor:
    """difflet_rocm_layernorm_modulate with one_plus = 0: LN(x) * weight + bias, fp32 stats."""
    return kernels.layernorm_modulate(x, weight, bias, eps=eps, one_plus=False)


@layer_norm.register_fake
def _(x, weight, bias, eps):
    return x.new_empty(x.shape)


@torch.library.custom_op("difflet_rocm::rope", mutates_args=())
def rope(x: Tensor, cos: Tensor, sin: Tensor, law: int) -> Tensor:
    """difflet_rocm_rope on x [..., S, D] with fp32 tables [S, D]; law 0 rotates in fp32
    (apply_rotary_emb_fp32), law 1 in the input dtype (apply_rotary_emb)."""
    return kernels.rope(x, cos, sin, law=law)


@rope.register_fake
def _(x, cos, sin, law):
    return x.new_empty(x.shape)


__all__ = ["attention", "fp8_linear", "layer_norm", "linear", "rms_norm", "rope"]

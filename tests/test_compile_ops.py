"""The custom-operator registration and the per-block compile helpers, on the CPU: every
``difflet_rocm::*`` operator has a schema and a fake implementation that gives the real one's
output shape and dtype (checked under FakeTensorMode, where no kernel runs), and the compile
helpers wrap exactly the repeated blocks. The compiled GPU path is test_gpu_compile.py."""

from __future__ import annotations

import pytest
import torch
import torch.nn as nn
from torch._subclasses.fake_tensor import FakeTensorMode

from difflet_amd.backends.rocm import compile as rc
from difflet_amd.backends.rocm.ops_impl import library  # noqa: F401  (registers the ops)

OPS = ("attention", "linear", "fp8_linear", "rms_norm", "layer_norm", "rope")


def test_every_op_is_registered_with_a_schema():
    for name in OPS:
        op = getattr(torch.ops.difflet_rocm, name).default
        assert op._schema.name == f"difflet_rocm::{name}"
        # functional: no argument is written
        assert not any(a.alias_info is not None and a.alias_info.is_write
                       for a in op._schema.arguments), name


def test_fake_implementations_give_shapes_and_dtypes():
    ops = torch.ops.difflet_rocm
    with FakeTensorMode():
        bf = dict(dtype=torch.bfloat16)
        q = torch.empty(1, 4, 300, 128, **bf)
        kv = torch.empty(1, 4, 77, 128, **bf)
        o = ops.attention(q, kv, kv, 0.1, False, None, None, None)
        assert o.shape == (1, 4, 300, 128) and o.dtype == torch.bfloat16
        o = ops.attention(q.reshape(4, 300, 128), kv.reshape(4, 77, 128),
                          kv.reshape(4, 77, 128).half(), 1.0, True, None, None, None)
        assert o.shape == (4, 300, 128) and o.dtype == torch.float16
        x = torch.empty(33, 384, **bf)
        y = ops.linear(x, torch.empty(100, 384, **bf), None, 99)
        assert y.shape == (33, 99) and y.dtype == torch.bfloat16
        y = ops.fp8_linear(x, torch.empty(256, 384, dtype=torch.uint8),
                           torch.empty(256, dtype=torch.float32), None, False)
        assert y.shape == (33, 256) and y.dtype == torch.bfloat16
        h = torch.empty(2, 9, 4, 128, dtype=torch.float32)
        assert ops.rms_norm(h, None, 1e-6).shape == h.shape
        assert ops.layer_norm(x, None, None, 1e-6).dtype == torch.bfloat16
        r = ops.rope(q, torch.empty(300, 128), torch.empty(300, 128), 1)
        assert r.shape == q.shape and r.dtype == q.dtype


class _Flux(nn.Module):
    def __init__(self):
        super().__init__()
        self.transformer_blocks = nn.ModuleList([nn.Linear(4, 4) for _ in range(2)])
        self.single_transformer_blocks = nn.ModuleList([nn.Linear(4, 4) for _ in range(3)])
        self.proj_out = nn.Linear(4, 4)


class _Wan(nn.Module):
    def __init__(self):
        super().__init__()
        self.blocks = nn.ModuleList([nn.Linear(4, 4)])


def test_repeated_blocks_and_compile_blocks():
    flux = _Flux()
    assert [len(b) for b in rc.repeated_blocks(flux)] == [2, 3]
    assert [len(b) for b in rc.repeated_blocks(_Wan())] == [1]
    outer = nn.Module()
    outer.transformer = _Flux()
    assert len(rc.repeated_blocks(outer)) == 2
    n = rc.compile_repeated_blocks_(flux, mode="default")
    assert n == 5
    assert all(type(b).__name__ == "OptimizedModule" for bl in rc.repeated_blocks(flux) for b in bl)
    assert isinstance(flux.proj_out, nn.Linear)  # the module around the blocks stays eager
    with pytest.raises(ValueError, match="repeated block lists"):
        rc.compile_repeated_blocks_(nn.Linear(2, 2))


def test_compile_options_extend_the_mode():
    blocks = nn.ModuleList([nn.Linear(2, 2)])
    assert rc.compile_blocks([blocks], dynamic=False, options={"max_autotune": False}) == 1
    assert rc.COMPILE_MODE == "max-autotune-no-cudagraphs"


def test_infer_twins_mirror_the_custom_ops():
    """The twin that eager inference calls: same signature, same fake; not taken for host tensors
    or tensors that require grad."""
    ops = torch.ops.difflet_rocm
    for name in ("attention", "attention_joint", "linear", "linear_f32", "fp8_linear"):
        a = getattr(ops, name).default._schema
        b = getattr(ops, f"{name}_infer").default._schema
        assert str(a).split("(", 1)[1] == str(b).split("(", 1)[1]
    with FakeTensorMode():
        x = torch.empty(33, 384, dtype=torch.bfloat16, device="cuda")
        w = torch.empty(100, 384, dtype=torch.bfloat16, device="cuda")
        assert library._plain(x, w, None) and not library._plain(x, w.requires_grad_())
        with torch.no_grad():
            assert library._plain(x, w)
        assert not library._plain(torch.empty(3))
        y = library.linear(x, w, None, 99)  # w requires grad: the custom op
        assert y.shape == (33, 99) and y.requires_grad
        y = library.linear(x, w.detach(), None, 99)
        assert y.shape == (33, 99) and y.dtype == torch.bfloat16 and y.is_cuda


def _linear_args():
    bf = dict(dtype=torch.bfloat16, device="cuda")
    return torch.empty(5, 33, 384, **bf), torch.empty(100, 384, **bf)


def _grad_nodes(y):
    seen, todo = set(), [y.grad_fn]
    while todo:
        node = todo.pop()
        if node is not None and node not in seen:
            seen.add(node)
            todo += [n for n, _ in node.next_functions]
    return {n.name() for n in seen}


@pytest.mark.parametrize("batched", [False, True])
@pytest.mark.parametrize("call", ["linear", "linear_infer"])
def test_gradients_are_refused_also_under_vmap(call, batched):
    """Inputs that need a gradient get the node whose backward raises, whether the call comes through
    library.linear or names the twin, and where vmap's batched tensor hides the gradient."""
    with FakeTensorMode():
        x, w = _linear_args()
        x.requires_grad_()
        fn = library.linear if call == "linear" else torch.ops.difflet_rocm.linear_infer
        f = lambda r: fn(r, w, None, 100)  # noqa: E731
        names = _grad_nodes(torch.vmap(f)(x) if batched else f(x[0]))
    assert any(n.startswith("GeneratedBackwardFor_difflet_rocm_linear") for n in names), names
    assert not any("NotImplemented" in n for n in names), names


@pytest.mark.parametrize("pre_dispatch", [False, True])
def test_recorded_graphs_hold_the_custom_op(pre_dispatch):
    """A graph recorded with inputs that need no gradient may be replayed with ones that do."""
    from torch.fx.experimental.proxy_tensor import make_fx

    with FakeTensorMode():
        x, w = _linear_args()
        gm = make_fx(lambda a: library.linear(a, w, None, 100), pre_dispatch=pre_dispatch)(x[0])
    calls = [n.target for n in gm.graph.nodes if n.op == "call_function"]
    assert torch.ops.difflet_rocm.linear.default in calls
    assert torch.ops.difflet_rocm.linear_infer.default not in calls


def test_twins_are_for_plain_eager_execution_only():
    import torch.autograd.forward_ad as fwd
    from torch.utils._python_dispatch import TorchDispatchMode

    class Mode(TorchDispatchMode):
        pass

    assert library._eager()
    with Mode():
        assert not library._eager()
    with fwd.dual_level():
        assert not library._eager()
    seen = []
    torch.vmap(lambda t: (seen.append(library._eager()), t)[1])(torch.zeros(2))
    torch.func.grad(lambda t: (seen.append(library._eager()), t.sum())[1])(torch.zeros(2))
    torch.jit.trace(lambda t: (seen.append(library._eager()), t + 1)[1], torch.zeros(2),
                    check_trace=False)
    assert seen == [False, False, False]
    assert library._eager()

"""GEMM launches of few tiles (64-, 128- and 256-row tiles, K whole or cut into pieces): every
element type and both epilogues at the edges of tiles, K stages and pieces, against the fp32
reference; scratch full of NaN patterns; strided and 8-byte aligned outputs; graph replays.

Tolerance: the products are exact in fp32 and the output is rounded once to bf16 (relative error
up to 2^-9, rms below 2^-9): rel L2 < 2^-9 plus 2e-4 for fp32 sums in another order. The gated
epilogue adds a rounded residual of the same size: the same bound."""

import pytest
import torch

from difflet_amd import _lib, kernels
from test_gpu_gemm_split import _operands, _reference, rel_l2, rnd

pytestmark = pytest.mark.gpu
TOL = 2.0 ** -9 + 2e-4

# (m, n, k): one row tile and its edges, two and three row tiles, narrow and ragged n, one K stage,
# K that pieces divide unevenly (MXFP8 in units of 4 stages), many column tiles
SHAPES = [(9, 4, 128), (64, 128, 128), (65, 132, 256), (63, 3076, 3072), (128, 512, 15360),
          (129, 252, 4096), (200, 3072, 6912), (257, 128, 7808), (512, 5120, 5120),
          (1024, 3072, 12288), (1500, 5120, 1280), (2047, 3072, 3072), (16, 18432, 3072)]


@pytest.mark.parametrize("kind", ["bf16", "fp8", "mx"])
@pytest.mark.parametrize("m,n,k", SHAPES)
def test_small_gemm_matches_the_reference(gpu, kind, m, n, k):
    print(f"small gemm {kind} m={m} n={n} k={k}", flush=True)
    g = torch.Generator().manual_seed(m + n + k)
    a, w, b = rnd(g, m, k), rnd(g, n, k, std=0.05), rnd(g, n, std=0.1)
    aq, wq, sa, sw = _operands(kind, a, w, gpu)
    ref = _reference(kind, a, w, b)
    bg = b.to(gpu)
    ws = torch.full((96 << 20,), 0xff, dtype=torch.uint8, device=gpu)  # NaN patterns
    outs = []
    for workspace in (None, "call", ws):
        c = torch.full((m, n + 12), float("nan"), dtype=torch.bfloat16, device=gpu)[:, 4:n + 4]
        kernels.gemm_grouped([kernels.Problem(aq, wq, c, bg, a_scale=sa, w_scale=sw)], kind=kind,
                             workspace=workspace)
        outs.append(c)
        assert rel_l2(c, ref) < TOL
    assert torch.equal(outs[1], outs[2])  # the plan does not depend on where the scratch lies
    # gate * (acc + bias) + residual written over the residual
    res, gate = rnd(g, m, n).to(gpu), rnd(g, 1, n).to(gpu)
    want = res.float().cpu() + gate.float().cpu() * ref
    kernels.gemm_grouped([kernels.Problem(aq, wq, res, bg, gate, res, a_scale=sa, w_scale=sw)],
                         kind=kind, epilogue=_lib.EPI_GATE_RESIDUAL, workspace="call")
    assert rel_l2(res, want) < TOL


def test_small_gemm_in_a_replayed_graph(gpu):
    """K pieces under capture: scratch from the graph's pool, each replay equal to eager."""
    from difflet_amd.backends.rocm.ops_impl import library

    g = torch.Generator().manual_seed(5)
    x, w, b = rnd(g, 128, 12288).to(gpu), rnd(g, 3072, 12288, std=0.05).to(gpu), rnd(g, 3072).to(gpu)
    assert _lib.load().difflet_rocm_gemm_scratch_bytes(0, 128, 3072, 12288) > 0
    want = library.linear(x, w, b, 3072)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        y = library.linear(x, w, b, 3072)
    for i in range(3):
        y.zero_()
        x2 = rnd(g, 128, 12288).to(gpu) if i == 1 else x
        eager = library.linear(x2, w, b, 3072)
        if i == 1:
            x.copy_(x2)
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(y, eager)
    assert not torch.equal(y, want)


@pytest.mark.parametrize("m,n,k", [(1, 4, 4), (63, 124, 36), (64, 128, 64), (65, 132, 100),
                                   (16, 12288, 4096), (129, 260, 4092), (452, 4096, 1024),
                                   (300, 512, 10240), (4200, 384, 516)])
def test_fp32_gemm(gpu, m, n, k):
    """fp32 GEMM: partial K stages, strided operands, residual in place; K whole and cut. Sums of k
    products in fp32 against 64 bits: error of the sum below sqrt(k) 2^-24 relative, 1e-5 at most."""
    print(f"fp32 gemm m={m} n={n} k={k}", flush=True)
    g = torch.Generator().manual_seed(m + n + k)
    a = torch.randn(m, k + 8, generator=g)[:, 4:k + 4]
    w = torch.randn(n, k + 4, generator=g)[:, :k]
    b, r = torch.randn(n, generator=g), torch.randn(m, n, generator=g)
    ref = a.double() @ w.double().t() + b.double()
    ag, wg = torch.zeros(m, k + 8).to(gpu)[:, 4:k + 4], torch.zeros(n, k + 4).to(gpu)[:, :k]
    ag.copy_(a), wg.copy_(w)
    for workspace in (None, "call"):
        y = kernels.gemm_f32(ag, wg, b.to(gpu), workspace=workspace)
        assert ((y.double().cpu() - ref).norm() / ref.norm()).item() < 1e-5
        y = r.to(gpu)
        kernels.gemm_f32(ag, wg, b.to(gpu), residual=y, out=y, workspace=workspace)
        assert ((y.double().cpu() - ref - r.double()).norm() / ref.norm()).item() < 1e-5


@pytest.mark.parametrize("kind", ["bf16", "fp8", "mx"])
@pytest.mark.parametrize("m,n,k", [(6889, 3072, 6144), (6700, 12288, 10240)])
def test_linear_call_split_schedule_on_scratch(gpu, kind, m, n, k):
    """A last wave of tiles cut over the XCDs on scratch of the call, which nobody zeroed: equal on
    reruns over garbage, and to whole tiles within fp32 summation order (2e-3, a bf16 step)."""
    if kind != "bf16":
        k *= 2  # the same number of K stages
    print(f"split on scratch {kind} m={m} n={n} k={k}", flush=True)
    g = torch.Generator(device=gpu).manual_seed(m)
    a = torch.randn(m, k, generator=g, device=gpu).bfloat16()
    w = (torch.randn(n, k, generator=g, device=gpu) * 0.05).bfloat16()
    aq, wq, sa, sw = _operands(kind, a, w, gpu)
    kid = {"bf16": 0, "fp8": 1, "mx": 2}[kind]
    nbytes = _lib.load().difflet_rocm_gemm_scratch_bytes(kid, m, n, k)
    assert nbytes == _lib.load().difflet_rocm_gemm_workspace_bytes()  # the split schedule's
    outs = []
    for _ in range(2):
        torch.full((nbytes,), 0xff, dtype=torch.uint8, device=gpu)  # freed: the scratch's garbage
        outs.append(kernels.gemm_call(kind, aq, wq, None, sa, sw))
    assert torch.equal(outs[0], outs[1])
    whole = torch.empty_like(outs[0])
    kernels.gemm_grouped([kernels.Problem(aq, wq, whole, a_scale=sa, w_scale=sw)], kind=kind)
    d = (outs[0].float() - whole.float()).norm() / whole.float().norm()
    assert d.item() < 2e-3


@pytest.mark.parametrize("kind,m,n,k", [("bf16", 128, 3072, 12288), ("bf16", 6889, 3072, 6144),
                                        ("fp8", 6889, 3072, 12288), ("f32", 16, 4096, 4096)])
def test_calls_without_memory_for_scratch(gpu, monkeypatch, kind, m, n, k):
    """Scratch only saves time: where torch has no memory for it the call runs with K whole, equal up
    to the order of fp32 sums (a bf16 step, 2e-3; fp32 1e-5)."""
    print(f"no scratch {kind} m={m} n={n} k={k}", flush=True)
    g = torch.Generator().manual_seed(m)
    a, w = rnd(g, m, k), rnd(g, n, k, std=0.05)
    kid = {"bf16": 0, "fp8": 1, "mx": 2, "f32": 3}[kind]
    assert _lib.load().difflet_rocm_gemm_scratch_bytes(kid, m, n, k) > 0
    if kind == "f32":
        a, w = a.float().to(gpu), w.float().to(gpu)
        calls = [lambda: kernels.gemm_f32(a, w, workspace="call")]
    else:
        aq, wq, sa, sw = _operands(kind, a, w, gpu)

        def grouped():
            c = torch.empty(m, n, dtype=torch.bfloat16, device=gpu)
            kernels.gemm_grouped([kernels.Problem(aq, wq, c, a_scale=sa, w_scale=sw)], kind=kind,
                                 workspace="call")
            return c

        calls = [grouped, lambda: kernels.gemm_call(kind, aq, wq, None, sa, sw)]
    want = [f() for f in calls]
    empty = torch.empty

    def no_scratch(*args, **kwargs):
        if kwargs.get("dtype") is torch.uint8:
            raise torch.OutOfMemoryError("no memory left")
        return empty(*args, **kwargs)

    monkeypatch.setattr(torch, "empty", no_scratch)
    got = [f() for f in calls]
    monkeypatch.undo()
    for x, y in zip(got, want):
        d = (x.float() - y.float()).norm() / y.float().norm()
        assert d.item() < (1e-5 if kind == "f32" else 2e-3)


@pytest.mark.parametrize("m,s,k", [(2, 32760, 5120), (5, 16384, 3072), (70, 8400, 2048)])
def test_rows_far_apart(gpu, m, s, k):
    """The last token of each of m batch elements: rows 34 to 335 MB apart, so that a tile's rows past
    m would lie 4 GiB and more past its first. Small tiles, the linear op's, and with two problems
    in a launch the 256 x 256 ones."""
    from difflet_amd.backends.rocm.ops_impl import library

    print(f"rows far apart m={m} s={s} k={k}", flush=True)
    g = torch.Generator(device=gpu).manual_seed(m)
    x = torch.empty(m, s, k, dtype=torch.bfloat16, device=gpu)[:, -1]
    x.normal_(generator=g)
    w = torch.empty(384, k, dtype=torch.bfloat16, device=gpu).normal_(std=0.05, generator=g)
    want = kernels.gemm_call("bf16", x.contiguous(), w, None)
    assert rel_l2(want, x.float() @ w.float().t()) < TOL
    assert torch.equal(kernels.gemm_call("bf16", x, w, None), want)
    assert torch.equal(library.linear(x, w, None, 384), want)
    c = [torch.empty_like(want) for _ in range(4)]
    kernels.gemm_grouped([kernels.Problem(t, w, y) for t, y in zip((x, x.contiguous()), c[:2])])
    kernels.linear(x, w, epilogue=_lib.EPI_GELU, out=c[2])
    kernels.linear(x.contiguous(), w, epilogue=_lib.EPI_GELU, out=c[3])
    assert torch.equal(c[0], c[1]) and torch.equal(c[2], c[3])
    assert rel_l2(c[0], want.float()) < TOL


def test_fp32_gemm_above_4_gib(gpu):
    """A weight past 4 GiB and K off the 32-float stage: the stage's missing values are zeros, not the
    weight's 2^32 - 16 bytes on (infinite here in row 1044495, which every row but its own ignores)."""
    n, k, hit = (1 << 20) + 64, 1028, (1 << 32) // (1028 * 4)
    w = torch.full((n, k), 0.5, device=gpu)
    w[hit] = float("inf")
    a = torch.ones(3, k, device=gpu)
    y = kernels.gemm_f32(a, w, workspace="call")
    assert torch.isinf(y[:, hit]).all()
    y[:, hit] = 0.5 * k
    assert bool((y == 0.5 * k).all())  # sums of halves: exact

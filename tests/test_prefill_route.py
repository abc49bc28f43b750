"""linear()'s route above AUTO_PREFILL_ROWS rows (CPU: the kernels are replaced by a recorder and a plain product): plain
calls take the int4 prefill GEMM where prefill_path says, calls that torch differentiates or transforms keep dequantize +
BLAS there and so their gradients, tangents and batches."""
from types import SimpleNamespace

import pytest
import torch
import torch.autograd.forward_ad as fwad
import torch.utils.flop_counter

from lowbit import _native, ops

N, K, M = 8320, 128, 600                                    # a wide layer, more rows than AUTO_PREFILL_ROWS


@pytest.fixture
def layer(monkeypatch):
    w = torch.randn(N, K, generator=torch.Generator().manual_seed(1)).half()
    taken = []

    def fake(name, result):
        def call(*args, **kwargs):
            taken.append(name)
            return result(*args, **kwargs)
        return call
    monkeypatch.setattr(ops, "prefill", fake("prefill", lambda x, wq: x.detach() @ w.t()))
    monkeypatch.setattr(ops, "dequant", fake("dequant", lambda *a: w))
    monkeypatch.setattr(ops, "ext", lambda: SimpleNamespace(w4_gemm_prefill=fake(
        "prefill+bias", lambda x, p, s, g, epilogue, bias, **own: (x.detach() @ w.t()).add_(bias.detach()))))
    wq = SimpleNamespace(n=N, k=K, packed=None, packed_v3=None, packed_mma=object(), scales=None, group=128)
    assert ops.prefill_path(M, wq) and not ops._prefill_without_blas(M, wq)
    return wq, w, taken


def test_plain_calls_take_the_int4_gemm(layer):
    wq, w, taken = layer
    x = torch.randn(M, K).half()
    ops.linear(x, wq)
    with torch.no_grad():
        ops.linear(x.clone().requires_grad_(), wq)
    ops.linear(torch.nn.Parameter(x, requires_grad=False), wq)
    assert taken == ["prefill"] * 3


def near(a, b):                                             # fp16 products of 128 unit-variance terms
    return torch.allclose(a.float(), b.float(), rtol=2e-2, atol=0.1)


def test_transformed_calls_keep_blas(layer):
    wq, w, taken = layer
    x = torch.randn(M, K).half().requires_grad_()
    ops.linear(x, wq).backward(torch.eye(M, N).half())
    assert near(x.grad, w[:M])
    with fwad.dual_level():
        t = torch.randn(M, K).half()
        out = ops.linear(fwad.make_dual(torch.randn(M, K).half(), t), wq)
        assert near(fwad.unpack_dual(out).tangent, t @ w.t())
    xs = torch.randn(2, M, K).half()
    assert near(torch.func.vmap(lambda a: ops.linear(a, wq))(xs), xs @ w.t())
    x3 = torch.randn(M, 2, K).half()
    assert near(ops.linear(x3, wq), x3 @ w.t())
    assert taken == ["dequant"] * 4


def test_the_bias_counts_as_x_does(layer):
    wq, w, taken = layer
    x = torch.randn(M, K).half()
    b = torch.randn(N).half()
    with torch.no_grad():
        ops.linear(x, wq, bias=b.clone().requires_grad_())
    for plain in (b, torch.nn.Parameter(b, requires_grad=False), b.float()):
        assert near(ops.linear(x, wq, bias=plain), x @ w.t() + b)
    assert taken == ["prefill+bias"] * 4
    taken.clear()
    for bias in (torch.nn.Parameter(b.clone()), b.float().requires_grad_(), b.view(1, N).clone().requires_grad_()):
        y = ops.linear(x, wq, bias=bias)
        assert y.requires_grad
        y.float().sum().backward()
        assert torch.equal(bias.grad.view(N).float(), torch.full((N,), float(M)))
    got = torch.func.grad(lambda a: ops.linear(x, wq, bias=a).float().sum())(b)
    assert torch.equal(got, torch.full((N,), float(M)).half())
    with fwad.dual_level():
        t = torch.randn(N).half()
        out = ops.linear(x, wq, bias=fwad.make_dual(b.clone(), t))
        assert torch.equal(fwad.unpack_dual(out).tangent, t.expand(M, N))

    class Sub(torch.Tensor):
        pass
    assert type(ops.linear(x, wq, bias=b.as_subclass(Sub))) is Sub
    assert taken == ["dequant"] * 6


def test_x_off_the_16_byte_grid_keeps_blas(layer):
    """A contiguous view that starts on any fp16 element was served by the BLAS GEMM; the int4 GEMM refuses it."""
    wq, w, taken = layer
    x = torch.randn(M, K).half()
    buf = torch.empty(M * K + 8, dtype=torch.float16)
    for off in (1, 2, 4, 8):
        at = buf[off:off + M * K].view(M, K).copy_(x)
        assert at.is_contiguous() and near(ops.linear(at, wq), x @ w.t())
    wide = torch.empty(M, K + 1, dtype=torch.float16)[:, 1:].copy_(x)        # copied to its own, aligned, memory
    assert near(ops.linear(wide, wq), x @ w.t())
    assert taken == ["dequant"] * 3 + ["prefill"] * 2


def test_calls_under_a_mode_keep_blas(layer):
    wq, w, taken = layer
    x = torch.randn(M, K).half()
    with torch.utils.flop_counter.FlopCounterMode(display=False) as count:
        ops.linear(x, wq)
    assert count.get_total_flops() == 2 * M * N * K

    class Mode(torch.overrides.TorchFunctionMode):
        seen = 0

        def __torch_function__(self, func, types, args=(), kwargs=None):
            Mode.seen += func is torch.nn.functional.linear
            return func(*args, **(kwargs or {}))
    with Mode():
        ops.linear(x, wq)
    with torch.device("cpu"):
        ops.linear(x, wq)
    assert Mode.seen == 1 and taken == ["dequant", "dequant", "prefill"]


@pytest.mark.parametrize("m,n,k,want", [
    (512, 8192, 2048, True), (513, 8192, 2048, False), (513, 4096, 8960, True), (1024, 8193, 2048, True),
    (1025, 4096, 8960, False), (1024, 4097, 2048, False), (1400, 22016, 2048, True), (1400, 18944, 3584, False),
    (2048, 18944, 3584, True), (2048, 22016, 2048, False), (2048, 16384, 3584, False), (2049, 18944, 3584, False),
    (2048, 4096, 4096, True), (2049, 4096, 4096, False), (5000, 256, 16384, True)])
def test_rule(m, n, k, want):
    assert ops.prefill_path(m, SimpleNamespace(n=n, k=k, packed=None, packed_v3=None, packed_mma=object())) is want


def test_results_are_plain_tensors(monkeypatch):
    class Sub(torch.Tensor):
        pass
    monkeypatch.setattr(_native, "torch", torch)
    x = torch.randn(3, 8).half()
    for v in (x, x.as_subclass(Sub), torch.nn.Parameter(x)):
        y = _native._output_rows(v, 3, 5)
        assert type(y) is torch.Tensor and y.shape == (3, 5) and y.dtype is torch.float16 and not y.requires_grad


@pytest.mark.parametrize("workspace", [0, 16384, 16384 + (1 << 20), 16384 + (64 << 20)])
def test_prefill_plans_fit(workspace):
    """The launch shape of the prefill GEMM over its range (host only): every tile is covered once, whole or in splits of
    at least four chunks, with an arrival counter a split tile and partials within the workspace; whole tiles before split
    ones fill whole rounds, so that the workgroup numbering of both starts on a multiple of the eight XCDs."""
    import ctypes
    p = (ctypes.c_int * 5)()
    shapes = set()
    for k in (128, 384, 896, 2048, 3584, 11008, 18944):
        for n in (1, 64, 250, 1536, 2048, 2560, 4604, 11008, 18944, 22016):
            for m in (1, 64, 65, 100, 200, 333, 512, 700, 1000, 1400, 2048, 5000):
                _native.check(_native.lib().lowbit_w4_prefill_plan(m, n, k, workspace, p))
                rows, cols, split, whole, groups = p
                shapes.add((rows, cols, split > 1, whole > 0))
                tiles = -(-m // rows) * -(-n // cols)
                rest = tiles - whole
                assert groups == whole + split * rest and whole >= 0 and rest >= 0
                assert rest == 0 or split > 1 and k // 128 >= 4 * split and rest <= 4096
                assert rest == 0 or whole % 256 == 0
                assert rest == 0 or 16384 + rest * split * rows * cols * 4 <= workspace
    assert {s[:2] for s in shapes} == {(64, 64), (64, 128), (96, 256), (128, 128)}
    if workspace > 1 << 25:
        assert {s[:2] for s in shapes if s[2] and s[3]} >= {(96, 256), (128, 128)}

"""The prefill GEMM at the edges of its tile shapes (64, 96 and 128 activation rows; 64, 128 and 256 weight rows), its K
splits and its output path (16-byte pieces, or element by element for widths and addresses that do not allow them),
against the fp64 product of the exactly dequantized weights; and the routes above AUTO_PREFILL_ROWS rows.

Bound (assert_rounds): half an fp16 ulp plus 2^-16 of the outputs' RMS for the fp32 sums."""
import ctypes

import pytest
import torch
import torch.nn.functional as F

from lowbit import _native, ops
from test_gpu_kernels import make_weight
from test_gpu_prefill import assert_rounds, prefill, ulps

pytestmark = pytest.mark.gpu


def plan(m, k, n):
    """(activation rows, weight rows of a tile; K split; whole tiles; workgroups) of the launch"""
    p = (ctypes.c_int * 5)()
    _native.check(_native.lib().lowbit_w4_prefill_plan(m, n, k, _native.PREFILL_WORKSPACE_BYTES, p))
    return tuple(p)


# rows at, before and after a multiple of 64, 96 and 128; N at and off multiples of 256, 64, 16, 8, 4 and 2; one chunk of
# K, an odd count, and long K (splits)
@pytest.mark.parametrize("m,k,n", [
    (64, 128, 64), (65, 128, 250), (95, 384, 257), (96, 640, 1000), (97, 256, 1004), (127, 1152, 998), (128, 896, 4864),
    (129, 2048, 2050), (191, 11008, 130), (192, 8960, 1536), (193, 4096, 72), (255, 1536, 8961), (257, 128, 8960),
    (65, 128, 5), (333, 2048, 11004), (333, 2048, 11003), (700, 2048, 2560), (385, 1024, 11008), (1025, 640, 4099), (640, 384, 22016)])
def test_tile_edges(cuda, m, k, n):
    wq, *_, gen = make_weight(k, n, m + k + n, layouts=("mma",), sd=0.02)
    x = torch.randn(m, k, generator=gen).half().cuda()
    w = ops.dequant(wq, "mma").double()
    y = prefill(x, wq)
    assert_rounds(y, x.double() @ w.t())
    assert torch.equal(prefill(x, wq), y)
    bias = torch.randn(n, generator=gen).half().cuda()
    assert torch.equal(prefill(x, wq, _native.EPI_BIAS, bias), y + bias)
    res = torch.randn(m, n, generator=gen).half().cuda()
    want = res + y
    prefill(x, wq, _native.EPI_RESIDUAL, res, out=res)
    assert torch.equal(res, want)


# whole tiles and split ones in one launch: the tiles that fill whole rounds of the chip take a workgroup each, those of the
# last round K in pieces, with counters and partials numbered from the first of them
@pytest.mark.parametrize("m,k,n,tile", [
    (1000, 2048, 12320, (96, 256)), (1000, 2048, 12322, (96, 256)), (1400, 1536, 5995, (128, 128)),
    (1400, 1536, 6000, (128, 128)), (2047, 3584, 4604, (128, 128)), (700, 2048, 11984, (64, 128)),
    (700, 2048, 11989, (64, 128)), (700, 3584, 18944, (96, 256))])
def test_whole_and_split_tiles(cuda, m, k, n, tile):
    got = plan(m, k, n)
    assert got[:2] == tile and got[2] > 1 and 0 < got[3] < got[4], got
    gen = torch.Generator(device="cuda").manual_seed(m + n)
    wq = ops.W4Weight.from_float(0.02 * torch.randn(n, k, generator=gen, device="cuda"), 128, ("mma",))
    x = torch.randn(m, k, generator=gen, device="cuda").half()
    y = prefill(x, wq)
    assert_rounds(y, x.double() @ ops.dequant(wq, "mma").double().t())
    assert torch.equal(prefill(x, wq), y)
    bias = torch.randn(n, generator=gen, device="cuda").half()
    assert torch.equal(prefill(x, wq, _native.EPI_BIAS, bias), y + bias)
    res = torch.randn(m, n, generator=gen, device="cuda").half()
    want = res + y
    prefill(x, wq, _native.EPI_RESIDUAL, res, out=res)
    assert torch.equal(res, want)
    if n % 16 == 0:
        gu = y.view(m, -1, 2, 8)
        act = (F.silu(gu[:, :, 0]) * gu[:, :, 1]).reshape(m, -1)
        assert ulps(prefill(x, wq, _native.EPI_SILU_MUL), act) <= 1


@pytest.mark.parametrize("m,k,n,tile", [(129, 2048, 2050, (64, 64)), (191, 11008, 130, (64, 64)), (700, 2048, 2560, (64, 64)),
                                        (192, 8960, 1536, (64, 64)), (1025, 640, 4099, (64, 128)), (640, 384, 22016, (128, 128)),
                                        (333, 2048, 11004, (96, 256)), (333, 2048, 11003, (96, 256))])
def test_tile_edges_cover_the_shapes(cuda, m, k, n, tile):
    """The shapes of test_tile_edges that are there for a tile shape or a K split still take it."""
    got = plan(m, k, n)
    assert got[:2] == tile, got
    if k > 8000:
        assert got[2] > 1 and got[3] == 0, got


def test_output_at_any_address(cuda):
    wq, *_, gen = make_weight(512, 768, 3, layouts=("mma",), sd=0.02)
    x = torch.randn(200, 512, generator=gen).half().cuda()
    y = prefill(x, wq)
    for off in (1, 2, 4):                                   # 2-, 4- and 8-byte aligned outputs and residuals
        buf = torch.zeros(200 * 768 + 2 * off, dtype=torch.float16, device="cuda")
        out = buf[off:off + 200 * 768].view(200, 768)
        assert torch.equal(prefill(x, wq, out=out), y)
        assert int(torch.count_nonzero(buf[:off])) == 0 and int(torch.count_nonzero(buf[off + 200 * 768:])) == 0
        res = torch.randn(200, 768, generator=gen).half().cuda()
        out.copy_(res)
        assert torch.equal(prefill(x, wq, _native.EPI_RESIDUAL, out, out=out), res + y)


@pytest.mark.parametrize("m,k,n", [(512, 256, 8192), (513, 256, 8192), (1024, 2048, 11008), (1025, 256, 1536), (1100, 256, 17920), (1300, 256, 13000), (2048, 256, 11008),
                                   (2048, 2048, 2560), (2049, 256, 2048)])
def test_linear_agrees_on_both_prefill_routes(cuda, m, k, n):
    """linear() on either side of the routing rule equals the product of the dequantized weights, with and without a
    bias, whichever GEMM it takes."""
    wq, *_, gen = make_weight(k, n, m + n, layouts=("mma",), sd=0.02)
    x = torch.randn(m, k, generator=gen).half().cuda()
    bias = torch.randn(n, generator=gen).half().cuda()
    y = ops.linear(x, wq)
    assert_rounds(y, x.double() @ ops.dequant(wq, "mma").double().t())
    assert torch.equal(ops.linear(x, wq, bias=bias), y + bias)


def test_captured_calls_share_no_scratch(cuda):
    """Calls above AUTO_PREFILL_ROWS rows, with K split over workgroups, captured on one stream into graphs that are then
    replayed at the same time on two streams, between eager calls: every replay gives the eager result. The stream has
    captured before it has run any, and its first eager call comes after that."""
    wq, *_, gen = make_weight(11008, 2048, 5, layouts=("mma",), sd=0.02)
    bias = torch.randn(2048, generator=gen).half().cuda()
    xs = [torch.randn(600, 11008, generator=gen).half().cuda() for _ in range(2)]
    assert ops.prefill_path(600, wq) and not ops._prefill_without_blas(600, wq) and plan(600, 11008, 2048)[2] > 1
    want = [ops.linear(x, wq, bias=bias) for x in xs]
    side = torch.cuda.Stream()
    graphs, outs = [torch.cuda.CUDAGraph() for _ in xs], []
    for g, x in zip(graphs, xs):
        with torch.cuda.graph(g, stream=side):
            for _ in range(4):
                y = ops.linear(x, wq, bias=bias)
            outs.append(y)
    with torch.cuda.stream(side):
        eager = ops.linear(xs[0], wq, bias=bias)
    torch.cuda.synchronize()
    assert torch.equal(eager, want[0])
    streams = [torch.cuda.Stream() for _ in xs]
    for _ in range(3):
        for y in outs:
            y.zero_()
        torch.cuda.synchronize()
        for g, s in zip(graphs, streams):
            with torch.cuda.stream(s):
                g.replay()
        torch.cuda.synchronize()
        for y, w in zip(outs, want):
            assert torch.equal(y, w)
        assert torch.equal(ops.linear(xs[1], wq, bias=bias), want[1])

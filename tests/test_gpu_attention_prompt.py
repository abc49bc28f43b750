"""The prompt attention kernel (lowbit_attention from 384 query rows per KV head) against causal softmax attention in
fp64, at the sizes where its tiling can go wrong: row tiles of 64 and 32 that end inside a token's heads, key blocks of
64 and 128 that end on and beside a position, key partitions, positions out of order, rows without keys.

Bound: the outputs are fp16 (2^-11 relative to each value, at most 2^-11 of the row's largest) and everything before
them is fp32 or a split that keeps 2^-20; 2^-10 of the outputs' norm leaves a factor of two over the rounding.
"""
import math

import pytest
import torch

from lowbit import ops

pytestmark = pytest.mark.gpu
BOUND = 2.0 ** -10


def attend(q, k, v, positions, scale):
    m, hq, _ = q.shape
    grp = hq // k.shape[0]
    out = torch.empty(m, hq, 128, dtype=torch.float64, device=q.device)
    mask = torch.arange(k.shape[1], device=q.device)[None, :] > positions[:, None]
    for h in range(hq):
        s = (q[:, h].double() @ k[h // grp].double().t().contiguous()) * scale
        out[:, h] = torch.softmax(s.masked_fill(mask, -math.inf), -1) @ v[h // grp].double()
    return out


def case(m, hq, hkv, L, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    q = (2 * torch.randn(m, hq, 128, generator=g, device="cuda")).half()
    k = torch.randn(hkv, L, 128, generator=g, device="cuda").half()
    v = torch.randn(hkv, L, 128, generator=g, device="cuda").half()
    return q, k, v


def check(q, k, v, positions, scale, written, split=True):
    out = torch.empty(q.shape[0], q.shape[1] * 128, dtype=torch.float16, device="cuda")
    ops.ext().attention(q, k, v, positions, out, q.shape[1], k.shape[0], k.shape[1], scale, split=split)
    want = attend(q, k[:, :written], v[:, :written], positions, scale).view(q.shape[0], -1)
    err = (out.double() - want).norm() / want.norm()
    assert err < BOUND, float(err)
    return out


# tokens, query heads, KV heads, cached rows, cache length: (rows per KV head = tokens * group) % 64 and % 32 of every
# kind; keys that end at block edges (64 and 128) and one to either side; short and long caches (both tilings)
@pytest.mark.parametrize("m,hq,hkv,past,L", [
    (48, 16, 2, 0, 64), (64, 12, 2, 0, 64), (65, 28, 4, 0, 128), (49, 16, 2, 15, 64), (384, 2, 2, 0, 384),
    (385, 4, 4, 0, 512), (200, 4, 2, 63, 320), (129, 16, 4, 127, 256), (97, 12, 2, 31, 128), (55, 28, 4, 1100, 1200),
    (48, 16, 2, 976, 1024), (48, 16, 2, 977, 1088), (301, 16, 2, 2000, 4096), (700, 16, 2, 0, 1024)])
def test_prompt_attention(cuda, m, hq, hkv, past, L):
    q, k, v = case(m, hq, hkv, L, m + past)
    k[:, past + m:] = float("nan")                          # never written
    v[:, past + m:] = float("nan")
    pos = torch.arange(past, past + m, device="cuda")
    one = check(q, k, v, pos, 128 ** -0.5, past + m)
    assert torch.equal(one, check(q, k, v, pos, 128 ** -0.5, past + m))
    check(q, k, v, pos, 128 ** -0.5, past + m, split=False)


@pytest.mark.parametrize("L", [200, 1500])
def test_prompt_attention_positions_in_any_order(cuda, L):
    m = 96
    q, k, v = case(m, 16, 2, L, L)
    pos = torch.randperm(L, generator=torch.Generator().manual_seed(L))[:m].cuda()
    check(q, k, v, pos, 128 ** -0.5, L)
    check(q, k, v, torch.zeros(m, dtype=torch.long, device="cuda"), 128 ** -0.5, L)


@pytest.mark.parametrize("scale", [-0.1, 0.0, 1e-30, 3.0])
def test_prompt_attention_scales(cuda, scale):
    q, k, v = case(96, 12, 2, 320, 5)
    check(q, k, v, torch.arange(224, 320, device="cuda"), scale, 320)


# few rows over long caches: the same kernel with up to 64 key partitions (64 rows a workgroup, or 32 beyond 128 rows), below
# and above the lengths where it starts, positions well short of the cache's end, and partitions that hold no key
@pytest.mark.parametrize("m,hq,hkv,L,last", [
    (1, 28, 4, 4608, 4600), (1, 16, 2, 16384, 16383), (1, 12, 2, 10752, 40), (1, 4, 4, 32064, 32000), (2, 12, 2, 4096, 4095),
    (3, 28, 4, 2048, 1029), (4, 16, 2, 2112, 2111), (16, 16, 2, 4096, 700), (17, 16, 2, 6400, 6399), (47, 16, 2, 2048, 2000),
    (54, 28, 4, 2304, 2176)])
def test_long_cache_attention(cuda, m, hq, hkv, L, last):
    q, k, v = case(m, hq, hkv, L, m + last)
    k[:, last + 1:] = float("nan")
    v[:, last + 1:] = float("nan")
    pos = torch.arange(last + 1 - m, last + 1, device="cuda")
    one = check(q, k, v, pos, 128 ** -0.5, last + 1)
    assert torch.equal(one, check(q, k, v, pos, 128 ** -0.5, last + 1))
    check(q, k, v, torch.zeros(m, dtype=torch.long, device="cuda"), 128 ** -0.5, last + 1)


def test_long_cache_attention_then_projection(cuda):
    """lowbit_w4_attention_linear on a long cache: attention (merged by itself there), then the projection."""
    from lowbit import _native
    hq, hkv, L = 16, 2, 8192
    q, k, v = case(1, hq, hkv, L, 4)
    pos = torch.tensor([8000], device="cuda")
    wq = ops.W4Weight.from_float(0.02 * torch.randn(512, hq * 128, device="cuda"), 128, ("mma",))
    attn = torch.empty(1, hq * 128, dtype=torch.float16, device="cuda")
    ext = ops.ext()
    ext.attention(q, k, v, pos, attn, hq, hkv, L, 128 ** -0.5)
    want = ext.w4_linear_fused(attn, wq.packed_mma, wq.scales, 128, _native.EPI_STORE)
    got = ext.w4_attention_linear(q, k, v, pos, hq, hkv, L, 128 ** -0.5, wq.packed_mma, wq.scales, 128, _native.EPI_STORE)
    assert torch.equal(got, want)


def test_prompt_attention_of_growing_scores(cuda):
    """Every block of keys raises the rows' maximum far past the lag of the running reference, then lowers it again."""
    q, k, v = case(64, 16, 2, 1024, 9)
    k *= torch.linspace(0.05, 4.0, 1024, device="cuda").half()[None, :, None]
    pos = torch.arange(960, 1024, device="cuda")
    check(q, k, v, pos, 128 ** -0.5, 1024)
    check(q, k.flip(1).contiguous(), v, pos, 128 ** -0.5, 1024)


@pytest.mark.parametrize("m,drop,floor", [(1, 20.0, 39), (1, 24.0, 39), (1, 26.0, 39), (2, 26.0, 39), (16, 25.0, 32),
                                          (64, 26.0, 32)])
def test_long_tail_of_small_weights(cuda, m, drop, floor):
    """One key of weight 1 and value 0 beside tens of thousands of weights of 2^-drop, whose sum alone makes the output.
    Weights are good to 2^-39 of the largest below 32 rows per KV head and to 2^-32 from there on, 2^(drop - 39) or
    2^(drop - 32) of these; the outputs are fp16."""
    L, hq, hkv = 64000, 16, 2
    q = torch.zeros(m, hq, 128, device="cuda").half()
    q[..., 0] = 1
    k = torch.zeros(hkv, L, 128, device="cuda").half()
    k[:, 100, 0] = 128.0
    v = (1 + 0.25 * torch.randn(hkv, L, 128, generator=torch.Generator(device="cuda").manual_seed(6), device="cuda")).half()
    v[:, 100] = 0
    scale = drop * math.log(2.0) / 128.0
    pos = torch.full((m,), L - 1, device="cuda")
    out = torch.empty(m, hq * 128, dtype=torch.float16, device="cuda")
    ops.ext().attention(q, k, v, pos, out, hq, hkv, L, scale)
    want = attend(q, k, v, pos, scale).view(m, -1)
    assert bool((want > 1e-4).all())
    err = (out.double() - want).norm() / want.norm()
    assert err < BOUND + 2.0 ** (drop - floor), float(err)


# bounds far above the keys: the kernel is chosen on the device by the last token's position, one token, few rows (attend_heads
# below), up to 128 and 383 rows and prompts (attend_mfma below), keys on either side of each line and at partition edges;
# the last column sends the last token's position below the others'
@pytest.mark.parametrize("m,hq,hkv,L,keys", [
    (1, 16, 2, 8192, (1, 2, 127, 128, 129, 2049, 3124, 3125, 3126, 8192)), (1, 28, 4, 4608, (33, 1785, 1786, 1787, 4608)),
    (1, 16, 8, 16384, (64, 3125, 9000)), (3, 28, 4, 2048, (3, 500, 904, 905, 2048)), (2, 12, 2, 4096, (2, 3166, 3167, 4000)),
    (4, 16, 2, 4096, (4, 64, 65, 2047, 2048, 4096)), (16, 16, 2, 4096, (16, 31, 700, 2048, 3000)),
    (17, 16, 2, 2560, (17, 65, 600, 2047, 2048, 2560)), (16, 16, 16, 4096, (16, 3000)), (30, 12, 2, 4096, (40, 700, 3000)),
    (48, 16, 2, 4096, (48, 64, 65, 191, 192, 1500)), (55, 28, 4, 1200, (55, 192, 567, 1200)), (96, 12, 2, 2048, (96, 191, 400)),
    (200, 16, 2, 2048, (200, 300, 2048)), (400, 4, 4, 1664, (400, 1600)), (8, 8, 8, 8192, (8, 5000))])
def test_bound_above_the_keys(cuda, m, hq, hkv, L, keys):
    q, k, v = case(m, hq, hkv, L, m + L)
    clean = k, v
    for n in keys:
        k, v = clean[0].clone(), clean[1].clone()
        k[:, n:] = float("nan")
        v[:, n:] = float("nan")
        pos = torch.arange(n - m, n, device="cuda") if n >= m else torch.full((m,), n - 1, device="cuda")
        one = check(q, k, v, pos, 128 ** -0.5, n)
        assert torch.equal(one, check(q, k, v, pos, 128 ** -0.5, n))
        check(q, k, v, pos.flip(0).contiguous(), 128 ** -0.5, n)
        if n >= m:
            last_low = pos.clone()
            last_low[-1] = 0
            check(q, k, v, last_low, 128 ** -0.5, n)


@pytest.mark.parametrize("m,hq,hkv,L", [(1, 16, 2, 8192), (3, 28, 4, 4096), (16, 16, 2, 8192), (24, 16, 2, 2560),
                                        (64, 16, 2, 4096)])
def test_captured_once_for_every_position(cuda, m, hq, hkv, L):
    """A graph captured at one position serves the others: every replay has the eager call's bits, on both sides of the
    line and back, with eager calls between the replays."""
    q, k, v = case(m, hq, hkv, L, 3 * m)
    pos = torch.arange(m, device="cuda")
    out = torch.empty(m, hq * 128, dtype=torch.float16, device="cuda")
    call = lambda o: ops.ext().attention(q, k, v, pos, o, hq, hkv, L, 128 ** -0.5)
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        call(out)
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g, stream=side):
        call(out)
    for first in (0, 100, L - m, 30, 1000, 2500 if L > 2600 else 1500, 7):
        pos.copy_(torch.arange(first, first + m, device="cuda"))
        eager = torch.empty_like(out)
        call(eager)
        out.zero_()
        torch.cuda.synchronize()
        g.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, eager), first
        check(q, k, v, pos, 128 ** -0.5, first + m)


@pytest.mark.parametrize("m,hq,hkv,L,last", [(47, 16, 2, 2048, 2000), (54, 28, 4, 2304, 2176), (18, 28, 4, 2560, 2500),
                                             (47, 16, 2, 2048, 60)])
def test_long_cache_attention_in_a_workspace_of_its_size(cuda, m, hq, hkv, L, last):
    """Steps whose 16 partitions the Python binding's workspace does not hold, through the C ABI: with a workspace that
    holds them exactly and one that falls 16 bytes short (the other kernel), and nothing written past either."""
    from lowbit import _native
    q, k, v = case(m, hq, hkv, L, m)
    k[:, last + 1:] = float("nan")
    v[:, last + 1:] = float("nan")
    pos = torch.arange(last + 1 - m, last + 1, device="cuda")
    want = attend(q, k[:, :last + 1], v[:, :last + 1], pos, 128 ** -0.5).view(m, -1)
    need = 4096 + 16 * m * hq * 132 * 4
    for size in (need, need - 16, 2 * need):
        ws = torch.full((size + 4096,), 171, dtype=torch.uint8, device="cuda")
        out = torch.empty(m, hq * 128, dtype=torch.float16, device="cuda")
        _native.check(_native.lib().lowbit_attention(
            _native.ptr(q), _native.ptr(k), _native.ptr(v), _native.ptr(pos), _native.ptr(out), m, hq, hkv, L, L, 128 ** -0.5,
            _native.ptr(ws), size, torch.cuda.current_stream().cuda_stream))
        err = (out.double() - want).norm() / want.norm()
        assert err < BOUND, (size, float(err))
        assert bool((ws[size:] == 171).all()) and bool((ws[:4096] == 171).all())

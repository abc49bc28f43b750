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

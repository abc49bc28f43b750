"""The quantizer's kernel for groups of 32, 64 and 128 against the kernel of a wave per group, which the library takes for
tensors that 16-byte loads do not fit: the same bytes and scales on the same weights, with and without the clip search, for
every data type, at row and group counts that leave waves partly idle, and on weights beside rounding boundaries, zeros,
values whose scale overflows or underflows, infinities and NaNs."""
import pytest
import torch

from lowbit import ops

pytestmark = pytest.mark.gpu
CLIP = (1.0, 0.975, 0.95, 0.925, 0.9, 0.875, 0.85, 0.825, 0.8, 0.775, 0.75)


def both(w, group, grid):
    n, k = w.shape
    buf = torch.empty(n * k + 1, dtype=w.dtype, device="cuda")
    off = buf[1:].view(n, k)                                # not 16-byte aligned
    off.copy_(w)
    a, b = ops.ext().w4_quantize(w, group, grid), ops.ext().w4_quantize(off, group, grid)
    assert torch.equal(a[0], b[0])
    assert torch.equal(a[1].view(torch.int16), b[1].view(torch.int16))


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16, torch.float32])
@pytest.mark.parametrize("n,k,group", [(1, 32, 32), (3, 96, 32), (7, 64, 64), (5, 320, 64), (1, 128, 128), (37, 896, 128),
                                       (301, 2048, 128), (64, 4096, 32)])
def test_same_bits_as_a_wave_per_group(cuda, n, k, group, dtype):
    g = torch.Generator(device="cuda").manual_seed(n + k)
    w = (torch.randn(n, k, generator=g, device="cuda") * 0.02).to(dtype)
    for grid in (None, CLIP, (0.5,), (1.0, 1.0, 0.9)):
        both(w, group, grid)


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16, torch.float32])
def test_same_bits_on_hard_values(cuda, dtype):
    g = torch.Generator(device="cuda").manual_seed(1)
    half = (torch.randint(-15, 16, (256, 256), generator=g, device="cuda").float() + 0.0) * 0.5   # half-integer multiples
    scale = torch.rand(256, 1, generator=g, device="cuda").half().float()
    rows = [half * scale, half * scale * (1 + torch.randint(-3, 4, (256, 256), generator=g, device="cuda") * 2.0 ** -23)]
    big = torch.randn(256, 256, generator=g, device="cuda")
    rows += [big * 1e-7, big * 6e4, big * 3e5, big * 0.0]
    special = big.clone()
    special[::3, ::17] = float("inf")
    special[1::3, ::29] = float("nan")
    special[2::3, 5] = -float("inf")
    rows.append(special)
    for w in rows:
        for group in (32, 64, 128):
            for grid in (None, CLIP):
                both(w.to(dtype).contiguous(), group, grid)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_same_bits_where_quotients_overflow(cuda, dtype):
    """Clip factors near 0 on weights near fp32's largest value: finite scales whose quotients pass fp32's range."""
    g = torch.Generator(device="cuda").manual_seed(3)
    w = (torch.randn(64, 256, generator=g, device="cuda").clamp(-3, 3) * 1e38).to(dtype)
    assert bool(torch.isfinite(w).all())
    for group in (32, 64, 128):
        for grid in ((1e-38,), (1e-37, 3e-38, 1e-38, 3e-39), (2e-38, 1.0), (0.0,)):
            both(w, group, grid)
        both(torch.cat([w[:3], w[3:6] * 1e-38]), group, (1e-38, 1.0))

"""The fp16-weight MFMA head kernel (lowbit_f16_gemv beyond 8 rows) where its ring and tiles can go wrong: fewer chunks of K
than the ring holds, one more and many; 9, 16, 17, 33, 48, 49 and 64 rows; N beside multiples of 64, 16 and 4; the shorter
ring of many-row, short-K weights.

Bound: half an fp16 ulp of the result plus 2^-16 of the outputs' RMS for the fp32 sums, against the fp64 product."""
import pytest
import torch

from lowbit import ops
from test_gpu_prefill import assert_rounds

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("k", [128, 256, 384, 512, 640, 2048, 3584])
@pytest.mark.parametrize("m,n", [(9, 63), (10, 64), (16, 65), (17, 1000), (32, 258), (33, 16), (48, 129), (49, 70), (64, 515)])
def test_head_rows(cuda, m, n, k):
    g = torch.Generator(device="cuda").manual_seed(m + n + k)
    x = torch.randn(m, k, generator=g, device="cuda").half()
    w = (torch.randn(n, k, generator=g, device="cuda") * 0.02).half()
    y = ops.ext().f16_gemv(x, w)
    assert_rounds(y, x.double() @ w.double().t())
    assert torch.equal(ops.ext().f16_gemv(x, w), y)


@pytest.mark.parametrize("k", [128, 256, 384, 1536, 1664])
@pytest.mark.parametrize("m,n", [(33, 16385), (48, 16450), (49, 16384), (64, 16516)])
def test_head_rows_short_ring(cuda, m, n, k):
    test_head_rows(cuda, m, n, k)


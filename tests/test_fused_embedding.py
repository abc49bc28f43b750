"""The fused decoder's embedding lookup on the CPU (no layers, the final norm replaced by a copy): the rows of
F.embedding for the id types that it takes, at lengths on either side of the gather, and no others."""
from types import SimpleNamespace

import pytest
import torch

from lowbit import fused, ops


@pytest.fixture
def model(monkeypatch):
    monkeypatch.setattr(ops, "ext", lambda: SimpleNamespace(rmsnorm=lambda h, w, eps, out: out.copy_(h)))
    f = object.__new__(fused.FusedQwen2)
    f.embed = torch.randn(50, 8, generator=torch.Generator().manual_seed(2)).half()
    f.hidden, f.hq, f.head_dim, f.quant, f.layers, f.final_norm, f.eps, f.max_len = 8, 1, 128, "int4", [], None, 1e-6, 32
    f.logits = lambda xn, pick: xn
    return f


@pytest.mark.parametrize("m", [1, 4, 16, 17, 30])
@pytest.mark.parametrize("dtype", [torch.int32, torch.int64])
def test_rows_of_the_ids(model, m, dtype):
    ids = torch.randperm(50, generator=torch.Generator().manual_seed(m))[:m].to(dtype)
    assert torch.equal(model(ids, torch.arange(m)), model.embed[ids.long()])
    every = torch.arange(50).to(dtype)[::3][:m]              # a strided view
    assert torch.equal(model(every, torch.arange(every.shape[0])), model.embed[every.long()])


@pytest.mark.parametrize("ids", [torch.tensor([3, 50]), torch.tensor([-1, 3]), torch.tensor([1.0, 2.0]),
                                 torch.tensor([1, 2], dtype=torch.int16), torch.tensor([1, 2], dtype=torch.uint8)])
def test_other_ids_are_refused(model, ids):
    with pytest.raises((IndexError, RuntimeError)):
        model(ids, torch.arange(2))

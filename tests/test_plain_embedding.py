"""Which embeddings the batched decode step reads as rows of their weight (host only)."""
from types import SimpleNamespace

import pytest
import torch


class _Wrapped(torch.nn.Parameter):
    """A weight that is not what its memory holds (a quantized or sharded one)."""


def _half(**kw):
    return torch.nn.Embedding(10, 16, **kw).half().requires_grad_(False)


def _with(change):
    e = _half()
    change(e)
    return e


def _weight(e, w):
    e.weight = torch.nn.Parameter(w, requires_grad=False)


@pytest.mark.parametrize("emb,plain", [
    (_half(), True), (_half(padding_idx=0), True), (torch.nn.Embedding(10, 16), False), (_half(max_norm=1.0), False),
    (torch.nn.EmbeddingBag(10, 16).half(), False),
    (_with(lambda e: e.register_forward_hook(lambda *a: None)), False),
    (_with(lambda e: e.register_forward_pre_hook(lambda *a: None)), False),
    (_with(lambda e: setattr(e, "forward", lambda t: t)), False),
    (_with(lambda e: _weight(e, torch.zeros(16, 10, dtype=torch.float16).t())), False),
    (_with(lambda e: _weight(e, torch.zeros(161, dtype=torch.float16)[1:].view(10, 16))), False),
    (_with(lambda e: _weight(e, torch.zeros(10, 16, dtype=torch.float16, device="meta"))), False),
    (_with(lambda e: setattr(e, "weight", _Wrapped(torch.zeros(10, 16).half(), requires_grad=False))), False)])
def test_plain_embedding(emb, plain):
    from leankv_amd.engine import BatchedEngine

    step = SimpleNamespace(tok=torch.zeros(2, dtype=torch.long))
    assert BatchedEngine._plain_embedding(step, emb) is plain

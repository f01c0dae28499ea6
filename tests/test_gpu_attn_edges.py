"""Decode attention over packed KV at the edges of its work split: blocks of 32 tokens to a wave, 16 waves to a
block, splits of whole 256-token units, 1 to 16 query heads per kv head, and sequences far shorter than their batch's
longest, against fp64 attention over the dequantized cache (the oracle), at the bound of the other attention tests."""
import pytest
import torch
from oracle import teal as ot
from test_gpu_kernels import RTOL, _attn_case, _paged_tq_case

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("B,Hq,Hkv,cold,bits", [
    (1, 8, 8, 31, 3), (1, 32, 8, 32, 4), (1, 16, 1, 33, 3), (2, 30, 2, 255, 1), (1, 28, 2, 256, 2), (1, 14, 1, 257, 4),
    (1, 32, 8, 511, 3), (1, 32, 8, 512, 1), (5, 8, 4, 513, 2), (3, 24, 8, 545, 3), (33, 8, 8, 290, 3), (1, 2, 1, 2049, 4)])
def test_split_edges(cuda, B, Hq, Hkv, cold, bits):
    out, ref = _attn_case(B, Hq, Hkv, cold + 64, 64, seed=cold + bits, dev=cuda, bits=bits)
    assert torch.isfinite(out).all()
    assert ot.max_rel_err(out.numpy(), ref.numpy()) < RTOL


@pytest.mark.parametrize("lens,Hq,Hkv,hot,ps,bits", [
    ([1500, 64, 65, 1, 96, 97], 16, 2, 64, 16, 3), ([320, 577, 1, 2113], 16, 1, 64, 128, 4),
    ([300, 17, 49, 600], 8, 8, 16, 32, 1), ([1100, 321, 129, 128], 24, 4, 128, 64, 2)])
def test_paged_mixed_lengths(cuda, lens, Hq, Hkv, hot, ps, bits):
    out, ref = _paged_tq_case(lens, Hq, Hkv, hot, ps, bits, seed=sum(lens) % 1000 + ps, dev=cuda)
    assert torch.isfinite(out).all()
    assert ot.max_rel_err(out.numpy(), ref.numpy()) < RTOL

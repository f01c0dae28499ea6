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


@pytest.mark.parametrize("bits", [1, 2, 3, 4])
@pytest.mark.parametrize("Hq,Hkv,n", [(32, 8, 1), (32, 8, 65), (8, 8, 96), (16, 1, 97), (14, 1, 319), (32, 8, 320),
                                      (32, 2, 321), (30, 2, 576), (24, 8, 600)])
def test_both_block_sizes(cuda, Hq, Hkv, n, bits):
    """The same tokens by blocks of 8 waves (a bound that one round of 256-token splits covers) and of 16 (a bound whose
    splits are longer), dense and paged, against fp64 attention."""
    from leankv_amd import kernels
    from leankv_amd.turboquant.codebook import get_codebook_tensors
    from leankv_amd.turboquant.rotation import generate_rotation_matrix

    hot, ps, cap = 64, 16, 131072 // Hkv
    g = torch.Generator(device=cuda).manual_seed(n + bits)
    rb, cold = kernels.packed_row_bytes(bits), max(0, n - 64)
    cent = get_codebook_tensors(128, bits, cuda)[0]
    pis = [generate_rotation_matrix(128, cuda, seed=42 + j) for j in range(2)]
    q = torch.randn(1, Hq, 128, generator=g, device=cuda).half()
    store, full = [], []
    for pi in pis:
        idx = torch.randint(0, 1 << bits, (1, Hkv, cap, 128), generator=g, device=cuda, dtype=torch.uint8)
        w = {1: 1, 2: 2}.get(bits, 4)
        sh = torch.arange(8 // w, device=cuda, dtype=torch.uint8) * w
        codes = (idx.view(1, Hkv, cap, rb, 8 // w) << sh).sum(-1, dtype=torch.uint8)
        norms = torch.rand(1, Hkv, cap, generator=g, device=cuda) * 8 + 8
        ring = torch.randn(1, Hkv, hot, 128, generator=g, device=cuda).half()
        store.append((codes, norms, ring))
        x = cent.double()[idx[:, :, :cold].long()] @ pi.double() * norms[:, :, :cold].double().unsqueeze(-1)
        slots = torch.arange(cold, n, device=cuda) % hot
        full.append(torch.cat([x, ring[:, :, slots].double()], dim=2)[0].repeat_interleave(Hq // Hkv, dim=0))
    s = (full[0] @ q[0].double().unsqueeze(-1)).squeeze(-1) / 128 ** 0.5
    ref = (torch.softmax(s, -1).unsqueeze(1) @ full[1]).squeeze(1).float().cpu()
    (kc, kn, kh), (vc, vn, vh) = store
    seq = torch.tensor([n], dtype=torch.int32, device=cuda)
    npg = -(-max(cold, 1) // ps)
    perm = torch.randperm(npg, generator=g, device=cuda)  # page p of the sequence is pool page perm[p]

    def pool(t):
        t = t[0, :, :npg * ps].reshape(Hkv, npg, ps, *t.shape[3:]).transpose(0, 1)
        out = torch.empty_like(t, memory_format=torch.contiguous_format)
        out[perm] = t
        return out

    pools = [pool(t) for t in (kc, kn, vc, vn)]
    table = [torch.tensor([0, npg], dtype=torch.int32, device=cuda), perm.int()]
    for bound in (max(n, 2048), cap + hot):
        out = kernels.tq_decode_attn(q, kc, kn, vc, vn, kh, vh, *pis, cent, bits, seq, bound)
        assert ot.max_rel_err(out[0].cpu().numpy(), ref.numpy()) < RTOL
        out = kernels.tq_paged_decode_attn(q, *pools, kh, vh, *pis, cent, bits, *table, seq, bound)
        assert ot.max_rel_err(out[0].cpu().numpy(), ref.numpy()) < RTOL

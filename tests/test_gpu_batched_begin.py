"""lkv_batched_begin: the start of a batched decode step (embedding rows, their RMSNorm, the position's RoPE factors)."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("B,Z", [(1, 8), (2, 256), (3, 264), (16, 4096), (33, 1000), (2, 10240)])
def test_batched_begin_equals_its_parts(B, Z):
    from leankv_amd import kernels as K

    g = torch.Generator(device="cuda").manual_seed(Z)
    emb, w, cos, sin = (torch.randn(s, generator=g, device="cuda").half() for s in ((50, Z), (Z,), (9, 128), (9, 128)))
    tok = torch.randint(0, 50, (B,), generator=g, device="cuda")
    tok[0], tok[-1] = 0, 49
    for p in (0, 5, 8):
        pos = torch.tensor([p], dtype=torch.int32, device="cuda")
        x, h, c, s = K.batched_begin(tok, emb, w, 1e-5, cos, sin, pos)
        ref = emb[tok].view(B, 1, Z)
        assert torch.equal(x, ref) and torch.equal(h, K.rms_norm(ref, w, 1e-5))
        assert torch.equal(c.view(-1), cos[p]) and torch.equal(s.view(-1), sin[p])
    # past the tables: clamped to their ends
    tok[0], tok[-1] = -3, 50
    x, _, c, _ = K.batched_begin(tok, emb, w, 1e-5, cos, sin, torch.tensor([9], dtype=torch.int32, device="cuda"))
    assert torch.equal(x[-1, 0], emb[49]) and torch.equal(c.view(-1), cos[8])
    assert B == 1 or torch.equal(x[0, 0], emb[0])

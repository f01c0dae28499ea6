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


def test_other_embeddings_keep_their_module():
    """An embedding that does more than hand out fp16 rows runs as a module: the step is the same bit for bit."""
    from leankv_amd.engine import BatchedEngine, random_mistral
    from leankv_amd.turboquant.cache import TurboQuantCache

    model = random_mistral(device="cuda", seed=0, vocab_size=512, hidden_size=512, intermediate_size=1024,
                           num_hidden_layers=2, num_attention_heads=4, num_key_value_heads=2, head_dim=128,
                           max_position_embeddings=512)
    emb = model.model.embed_tokens
    plain = type(emb).forward

    def steps():
        cache = TurboQuantCache(num_layers=2, hot_buffer_size=16, device="cuda", max_seq_len=128)
        g = torch.Generator(device="cuda").manual_seed(3)
        for i in range(2):
            cache.update(*(torch.randn(3, 2, 40, 128, generator=g, device="cuda").half() for _ in range(2)), i)
        eng = BatchedEngine(model, cache, 3)
        eng.set_position(40)
        out = []
        for t in range(4):  # the first eager, the others replayed
            eng.tok.copy_(torch.tensor([t, 511 - t, 7 * t], device="cuda"))
            eng.step()
            out.append(eng.logits.clone())
        return eng._plain_embedding(emb), torch.stack(out)

    took, want = steps()
    assert took and torch.isfinite(want).all()
    calls = []
    handle = emb.register_forward_hook(lambda mod, args, out: calls.append(1))
    took, got = steps()
    handle.remove()
    assert not took and calls and torch.equal(got, want)
    emb.forward = lambda tok: plain(emb, tok)
    took, got = steps()
    del emb.forward
    assert not took and torch.equal(got, want)

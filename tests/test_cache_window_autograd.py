"""Updates of several tokens inside the hot window: on the host, and followed by autograd in both modes."""
import pytest
import torch
from torch.autograd import forward_ad


def _cache(hot=16, device="cpu", **kw):
    from leankv_amd.turboquant.cache import TurboQuantCache

    return TurboQuantCache(num_layers=1, hot_buffer_size=hot, device=device, max_seq_len=64, **kw)


def _kv(S, seed=0, device="cpu", B=2, H=3):
    g = torch.Generator().manual_seed(seed)
    return tuple(torch.randn(B, H, S, 128, generator=g).half().to(device) for _ in range(2))


def test_host_cache_inside_the_window():
    c = _cache()
    parts = [_kv(5, 1), _kv(4, 2), _kv(7, 3)]
    for k, v in parts:
        got = c.update(k, v, 0)
    for g, j in zip(got, (0, 1)):
        assert torch.equal(g, torch.cat([p[j] for p in parts], dim=2))


def test_gradients_reach_the_keys_and_values():
    c = _cache()
    (k0, v0), (k1, v1) = _kv(6, 4), _kv(9, 5)
    for t in (k0, v0, k1, v1):
        t.requires_grad_()
    c.update(k0, v0, 0)
    k, v = c.update(k1, v1, 0)
    (wk, wv) = _kv(15, 6)
    ((k.float() * wk.float()).sum() + (v.float() * wv.float()).sum()).backward()
    for t, w in ((k0, wk[:, :, :6]), (k1, wk[:, :, 6:]), (v0, wv[:, :, :6]), (v1, wv[:, :, 6:])):
        assert torch.equal(t.grad, w)


def test_forward_mode_tangents_reach_the_result():
    c = _cache()
    (k, v), (tk, tv) = _kv(7, 7), _kv(7, 8)
    with forward_ad.dual_level():
        out = c.update(forward_ad.make_dual(k, tk), forward_ad.make_dual(v, tv), 0)
        assert all(torch.equal(forward_ad.unpack_dual(o).tangent, t) for o, t in zip(out, (tk, tv)))


@pytest.mark.gpu
@pytest.mark.parametrize("p0,S", [(0, 2), (0, 40), (10, 3), (10, 30), (20, 5), (40, 33)])
def test_followed_update_equals_the_kernel(p0, S):
    """Values bit for bit those of the one-launch update; gradients of the tokens in the window, none past it."""
    (k0, v0), (k1, v1) = _kv(max(p0, 2), 9, "cuda"), _kv(S, 10, "cuda")
    outs = []
    for follow in (False, True):
        c = _cache(device="cuda")
        if p0:
            c.update(k0, v0, 0)
        k, v = (t.clone().requires_grad_(follow) for t in (k1, v1))
        out = c.update(k, v, 0)
        outs.append([t.detach() for t in (*out, c._k_codes[0], c._k_norms[0], c._v_codes[0], c._v_norms[0], c._k_hot[0],
                                          c._v_hot[0])])
    assert all(torch.equal(a, b) for a, b in zip(*outs))
    (out[0].float().sum() + 2 * out[1].float().sum()).backward()
    seen = (torch.arange(S, device="cuda") >= S - 16).half().view(1, 1, S, 1)
    assert torch.equal(k.grad, seen.expand_as(k)) and torch.equal(v.grad, (2 * seen).expand_as(v))

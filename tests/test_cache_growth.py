"""Growing a cache layer's store: contents kept, and no more memory at the peak than parts replaced one by one need."""
import pytest
import torch

B, H, HOT = 2, 8, 16


def _cache(cap, device):
    from leankv_amd.turboquant.cache import TurboQuantCache

    return TurboQuantCache(num_layers=1, hot_buffer_size=HOT, device=device, max_seq_len=cap)


@pytest.mark.parametrize("cap,own", [(40, False), (20000, True)])
def test_large_parts_have_buffers_of_their_own(cap, own):
    c = _cache(cap, "cpu")
    c._alloc(0, B, H, cap)
    parts = [getattr(c, n)[0] for n in ("_k_codes", "_v_codes", "_k_norms", "_v_norms")]
    assert all(t.is_contiguous() and not t.any() and t.shape[:3] == (B, H, cap) for t in parts)
    assert all((t.untyped_storage().nbytes() == t.nbytes) is own for t in parts)


@pytest.mark.gpu
def test_growth_peak():
    """Doubling holds at most the old store, the new codes of both sides and no old codes of the first: five times one
    side's codes, and the norms."""
    cap = 1 << 18
    c = _cache(cap, "cuda")
    c._alloc(0, B, H, cap)
    codes, norms = c._k_codes[0].nbytes, c._k_norms[0].nbytes
    c._k_codes[0][:, :, -1] = 7
    torch.cuda.synchronize()
    base = torch.cuda.memory_allocated()
    torch.cuda.reset_peak_memory_stats()
    c._ensure_cap(0, cap + 1)
    peak = torch.cuda.max_memory_allocated() - base
    assert peak <= 3 * codes + 2 * norms + (1 << 20)  # five times, two of them in the base
    assert c.cold_capacity(0) == 2 * cap
    k = c._k_codes[0]
    assert bool((k[:, :, cap - 1] == 7).all()) and not k[:, :, :cap - 1].any() and not k[:, :, cap:].any()


@pytest.mark.gpu
@pytest.mark.parametrize("sizes", [[30, 60], [20, 1, 1, 200], [10, 5, 90]])
def test_an_update_that_grows_the_store(sizes):
    """The same tokens in a store that grows and in one that holds them all."""
    g = torch.Generator().manual_seed(sum(sizes))
    parts = [[torch.randn(B, H, s, 128, generator=g).half().cuda() for _ in range(2)] for s in sizes]
    small, large = _cache(8, "cuda"), _cache(512, "cuda")
    for k, v in parts:
        got, want = small.update(k, v, 0), large.update(k, v, 0)
        assert all(torch.equal(a, b) for a, b in zip(got, want))
    assert small.storage_generation > large.storage_generation

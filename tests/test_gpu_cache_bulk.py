"""lkv_tq_cache_bulk_update: S new tokens of one layer in one launch (leankv/turboquant/cache.py:84-159).

Expected contents come from a token-by-token restatement: tokens below T - hot are quantized (lkv_tq_quantize of
the fp16 rows widened to fp32, the same arithmetic, so bytes and norms are equal bit for bit), the others sit in ring
slot p % hot."""
import pytest
import torch

pytestmark = pytest.mark.gpu

# (p0, S, hot): empty window, part-filled and full; fewer and more new tokens than the window; tile edges
SHAPES = [(0, 2, 64), (0, 64, 64), (0, 65, 64), (0, 333, 64), (1, 63, 64), (40, 30, 64), (40, 300, 64), (63, 17, 64),
          (64, 2, 64), (64, 64, 64), (70, 63, 64), (130, 200, 64), (5, 3, 1), (0, 5, 1), (250, 16, 256), (300, 31, 16)]


@pytest.mark.parametrize("bits", [1, 2, 3, 4])
@pytest.mark.parametrize("p0,S,hot", SHAPES)
def test_bulk_update_equals_token_by_token(p0, S, hot, bits):
    from leankv_amd import kernels as K
    from leankv_amd.turboquant.codebook import get_codebook_tensors
    from leankv_amd.turboquant.rotation import generate_rotation_matrix

    dev, B, H, D = "cuda", 2, 3, 128
    T, rb = p0 + S, K.packed_row_bytes(bits)
    cap = max(1, T - hot) + 5
    g = torch.Generator().manual_seed(7 * p0 + S + bits)
    bounds = get_codebook_tensors(D, bits, dev)[1][1:-1].contiguous()
    sides = []
    for j in range(2):
        x = torch.randn(B, H, T, D, generator=g).half().to(dev)
        x[0, 0, T // 2] = 0
        pi = generate_rotation_matrix(D, dev, seed=42 + j)
        codes, norms = K.tq_quantize(x.float(), pi, bounds, bits)
        hotb = torch.full((B, H, hot, D), 9.0, dtype=torch.float16, device=dev)
        for p in range(max(0, p0 - hot), p0):
            hotb[:, :, p % hot] = x[:, :, p]
        new = x[:, :, p0:]
        # the layouts attention hands over: a transposed [B, S, H, D] view, and a slice of a longer tensor
        new = new.transpose(1, 2).contiguous().transpose(1, 2) if j else new
        want = hotb.clone()
        for p in range(max(p0, T - hot), T):
            want[:, :, p % hot] = x[:, :, p]
        sides.append(dict(new=new, pi=pi, codes=codes, norms=norms, hot=hotb, want=want,
                          c=torch.full((B, H, cap, rb), 0xA5, dtype=torch.uint8, device=dev),
                          n=torch.full((B, H, cap), -7.0, device=dev)))
    k, v = sides
    K.tq_cache_bulk_update(k["new"], v["new"], p0, k["hot"], v["hot"], k["c"], k["n"], v["c"], v["n"], k["pi"], v["pi"],
                           bounds, bits)
    c0, c1 = max(0, p0 - hot), max(0, T - hot)
    for s in sides:
        assert torch.equal(s["hot"], s["want"])
        assert torch.equal(s["c"][:, :, c0:c1], s["codes"][:, :, c0:c1])
        assert torch.equal(s["n"][:, :, c0:c1], s["norms"][:, :, c0:c1])
        for t, fill in ((s["c"], 0xA5), (s["n"], -7.0)):  # nothing else of the store is written
            assert bool((t[:, :, :c0] == fill).all()) and bool((t[:, :, c1:] == fill).all())


def test_bulk_update_refuses_bad_calls():
    from leankv_amd import kernels as K
    from leankv_amd._lib import LeanKVError

    def call(S=4, p0=62, cap=8, dtype=torch.float16, hot=64):
        z = lambda *s, dt=torch.float16: torch.zeros(*s, dtype=dt, device="cuda")  # noqa: E731
        x = z(1, 1, S, 128, dt=dtype)
        K.tq_cache_bulk_update(x, x, p0, z(1, 1, hot, 128), z(1, 1, hot, 128), z(1, 1, cap, 64, dt=torch.uint8),
                               z(1, 1, cap, dt=torch.float32), z(1, 1, cap, 64, dt=torch.uint8),
                               z(1, 1, cap, dt=torch.float32), z(128, 128, dt=torch.float32),
                               z(128, 128, dt=torch.float32), z(7, dt=torch.float32), 3)

    call()
    with pytest.raises(LeanKVError):
        call(S=20)  # 18 cold tokens do not fit 8 rows
    with pytest.raises(LeanKVError):
        call(dtype=torch.float32)


def _layouts(x):
    """[B, H, S, 128] tensors equal to x that lie in memory as callers may hand them over."""
    B, H, S, D = x.shape
    off = torch.empty(x.numel() + 1, dtype=x.dtype, device=x.device)[1:].view(x.shape)
    wide = torch.empty(B, H, S, 2 * D, dtype=x.dtype, device=x.device)[..., ::2]
    odd = torch.empty(B, H, S, D + 1, dtype=x.dtype, device=x.device)[..., :D]
    rows = torch.empty(S, H, B, D, dtype=x.dtype, device=x.device).permute(2, 1, 0, 3)
    last = torch.empty(H, S, D, B, dtype=x.dtype, device=x.device).permute(3, 0, 1, 2)  # B = 1: strides (1, ..)
    for nm, t in (("offset", off), ("strided", wide), ("odd rows", odd), ("seq first", rows), ("batch last", last)):
        yield nm, t.copy_(x)


@pytest.mark.parametrize("B,H,S", [(1, 3, 70), (2, 1, 5), (1, 1, 66), (2, 3, 130)])
def test_update_takes_any_layout(B, H, S):
    """Rows at any offset, of any strides, with free strides of single sizes."""
    from leankv_amd.turboquant.cache import TurboQuantCache

    def run(k, v):
        c = TurboQuantCache(num_layers=1, hot_buffer_size=64, device="cuda", max_seq_len=256)
        return c.update(k, v, 0)

    g = torch.Generator(device="cuda").manual_seed(S)
    k, v = (torch.randn(B, H, S, 128, generator=g, device="cuda").half() for _ in range(2))
    want = run(k, v)
    for (nm, kk), (_, vv) in zip(_layouts(k), _layouts(v)):
        got = run(kk, vv)
        assert all(torch.equal(a, b) for a, b in zip(got, want)), nm


def test_update_of_another_batch_is_refused():
    """As many rows of another batch and head count: refused, the cache as it was."""
    from leankv_amd._lib import LeanKVError
    from leankv_amd.turboquant.cache import TurboQuantCache

    c = TurboQuantCache(num_layers=1, hot_buffer_size=16, device="cuda", max_seq_len=64)
    x = torch.randn(2, 4, 20, 128, device="cuda").half()
    want = c.update(x, x, 0)
    y = torch.randn(4, 2, 5, 128, device="cuda").half()
    with pytest.raises(LeanKVError):
        c.update(y, y, 0)
    assert c.get_seq_length(0) == 20 and all(torch.equal(a, b) for a, b in zip(c[0], want))


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_update_of_other_types(dtype):
    """Keys and values of a model's own type: the cache of their fp16 values, handed back in the cache's type."""
    from leankv_amd.turboquant.cache import TurboQuantCache

    g = torch.Generator(device="cuda").manual_seed(5)
    parts = [[torch.randn(2, 3, S, 128, generator=g, device="cuda").to(dtype) for _ in range(2)] for S in (30, 50, 1, 20)]
    a = TurboQuantCache(num_layers=1, hot_buffer_size=16, device="cuda", max_seq_len=128, dtype=dtype)
    b = TurboQuantCache(num_layers=1, hot_buffer_size=16, device="cuda", max_seq_len=128)
    for k, v in parts:
        got, want = a.update(k, v, 0), b.update(k.half(), v.half(), 0)
        assert all(x.dtype == dtype and torch.equal(x, y.to(dtype)) for x, y in zip(got, want))


def test_update_and_read_on_another_stream():
    """Layouts that are copied first, on a stream that is kept busy: launched there, temporaries kept until used."""
    from leankv_amd.turboquant.cache import TurboQuantCache

    g = torch.Generator(device="cuda").manual_seed(6)
    parts = [[torch.randn(2, 3, 256, S, generator=g, device="cuda").half()[:, :, ::2].transpose(2, 3) for _ in range(2)]
             for S in (300, 40, 7)]

    def run():
        c = TurboQuantCache(num_layers=1, hot_buffer_size=64, device="cuda", max_seq_len=512)
        return [t for k, v in parts for t in c.update(k, v, 0)]

    want = run()
    torch.cuda.synchronize()
    s = torch.cuda.Stream()
    with torch.cuda.stream(s):
        x = torch.randn(4096, 4096, device="cuda")
        for _ in range(4):
            x = x @ x * 1e-3
        got = run()
    s.synchronize()
    assert all(torch.equal(a, b) for a, b in zip(got, want))

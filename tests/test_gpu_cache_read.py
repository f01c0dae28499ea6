"""lkv_tq_cache_read: a layer's K and V in position order (leankv/turboquant/cache.py:169-189) in one launch."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def _store(B, H, n, hot, bits, seed=0):
    """Random codes and norms of a layer, its rotations, centroids and rings (plus a capacity past the cold part)."""
    from leankv_amd import kernels as K
    from leankv_amd.turboquant.codebook import get_codebook_tensors
    from leankv_amd.turboquant.rotation import generate_rotation_matrix

    g = torch.Generator().manual_seed(seed)
    cold, rb = max(0, n - hot), K.packed_row_bytes(bits)
    cap = cold + 9
    out = []
    for j in range(2):
        codes = torch.randint(0, 256, (B, H, cap, rb), generator=g, dtype=torch.uint8)
        if bits == 3:
            codes &= 0x77
        out += [codes.cuda(), (torch.rand(B, H, cap, generator=g) * 20).cuda()]
    rings = [torch.randn(B, H, hot, 128, generator=g).half().cuda() for _ in range(2)]
    pis = [generate_rotation_matrix(128, "cuda", seed=42 + j) for j in range(2)]
    return out, rings, pis, get_codebook_tensors(128, bits, "cuda")[0], cold


def _exact(codes, norms, pi, cent, bits):
    from leankv_amd.turboquant.quantizer import _unpack_indices

    c = cent.double()[_unpack_indices(codes, bits, 128)]
    return (c @ pi.double()) * norms.double().unsqueeze(-1)


@pytest.mark.parametrize("bits", [1, 2, 3, 4])
@pytest.mark.parametrize("B,H,n,hot", [(1, 1, 1, 64), (2, 3, 64, 64), (2, 3, 65, 64), (1, 5, 80, 64), (3, 2, 97, 64),
                                       (1, 8, 5000, 64), (2, 8, 777, 256), (1, 2, 40, 1)])
def test_cache_read(B, H, n, hot, bits):
    from leankv_amd import kernels as K

    (kc, kn, vc, vn), rings, pis, cent, cold = _store(B, H, n, hot, bits)
    got = K.tq_cache_read(kc, kn, vc, vn, *rings, *pis, cent, bits, n)
    slots = torch.arange(cold, n, device="cuda") % hot
    for out, codes, norms, ring, pi in zip(got, (kc, vc), (kn, vn), rings, pis):
        assert torch.equal(out[:, :, cold:], ring[:, :, slots])
        if not cold:
            continue
        ref = _exact(codes[:, :, :cold], norms[:, :, :cold], pi, cent, bits)
        # half an fp16 ulp of the value, plus fp32 rounding: the split parts carry 2^-22 of each of 128 products and
        # the accumulators 2^-24 per step of sums no larger than |c| |Pi| <= the row's norm
        tol = ref.abs() * 2.0 ** -11 + 2.0 ** -25 + ref.norm(dim=-1, keepdim=True) * 2.0 ** -20
        assert bool(((out[:, :, :cold].double() - ref).abs() <= tol).all())


@pytest.mark.parametrize("bits", [1, 2, 3, 4])
def test_cache_read_is_as_exact_as_fp32_dequantize(bits):
    """The values that are not the 64-bit result rounded to fp16: no more than of the fp32 MFMA chain's."""
    from leankv_amd import kernels as K

    (kc, kn, vc, vn), rings, pis, cent, cold = _store(1, 8, 4096 + 64, 64, bits, seed=3)
    k, _ = K.tq_cache_read(kc, kn, vc, vn, *rings, *pis, cent, bits, 4096 + 64)
    kc, kn = kc[:, :, :cold].contiguous(), kn[:, :, :cold].contiguous()
    old = K.tq_dequantize(kc, kn, pis[0], cent, bits, out_dtype=torch.float16)
    ref = _exact(kc, kn, pis[0], cent, bits).half()
    off_new, off_old = int((k[:, :, :cold] != ref).sum()), int((old != ref).sum())
    print("bits %d: %d of %d values off the rounded 64-bit result, fp32 chain %d" % (bits, off_new, ref.numel(), off_old))
    assert off_new <= off_old + 3 * off_old ** 0.5 + 8  # counting noise

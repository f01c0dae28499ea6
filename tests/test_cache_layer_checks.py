"""The checks of a cache layer's parts before their pointers reach a kernel (host only)."""
import pytest
import torch

B, H, HOT, CAP, RB = 2, 3, 16, 40, 64
PARTS = ("k_codes", "k_norms", "v_codes", "v_norms", "k_hot", "v_hot")


def _layer(device="cpu"):
    def codes():
        return torch.zeros(B, H, CAP, RB, dtype=torch.uint8, device=device)

    def norms():
        return torch.zeros(B, H, CAP, device=device)

    def hot():
        return torch.zeros(B, H, HOT, 128, dtype=torch.float16, device=device)

    return dict(k_codes=codes(), k_norms=norms(), v_codes=codes(), v_norms=norms(), k_hot=hot(), v_hot=hot())


def _check(parts, B=B, H=H):
    from leankv_amd.kernels import _check_layer

    return _check_layer("layer", torch.device("cpu"), B, H, 3, **parts)


def test_a_layer_passes():
    assert _check(_layer()) == (HOT, CAP)


@pytest.mark.parametrize("part", PARTS)
@pytest.mark.parametrize("wrong", ["rows swapped", "device", "dtype", "strides", "flat"])
def test_a_wrong_part_is_refused(part, wrong):
    from leankv_amd._lib import LeanKVError

    parts = _layer()
    t = parts[part]
    if wrong == "rows swapped":  # as many rows, another batch
        t = t.view(H, B, *t.shape[2:])
    elif wrong == "device":
        t = t.to("meta")
    elif wrong == "dtype":
        t = t.to(torch.int32)
    elif wrong == "strides":
        t = t.transpose(0, 1).contiguous().transpose(0, 1)
    else:
        t = t.view(B * H, *t.shape[2:])
    with pytest.raises(LeanKVError):
        _check(dict(parts, **{part: t}))


def test_other_batch_with_as_many_rows_is_refused():
    """An update of [3, 2, ..] to a layer of [2, 3, ..] rows: as many rows, other sequences."""
    from leankv_amd._lib import LeanKVError

    with pytest.raises(LeanKVError):
        _check(_layer(), B=H, H=B)

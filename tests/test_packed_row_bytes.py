"""packed_row_bytes takes whatever int() takes, by its value at the call."""
import numpy as np
import pytest
import torch


def test_by_value():
    from leankv_amd.kernels import LeanKVError, packed_row_bytes

    assert [packed_row_bytes(b) for b in (1, 2, 3, 4)] == [16, 32, 64, 64]
    t = torch.tensor(1)
    assert packed_row_bytes(t) == 16
    t.fill_(2)
    assert packed_row_bytes(t) == 32
    assert packed_row_bytes(np.array(4)) == 64
    with pytest.raises(LeanKVError):
        packed_row_bytes(5)

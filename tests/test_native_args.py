"""What the library handle makes of Python arguments: a tensor is its device address where the signature has a pointer; where
it has a number, a tensor of one element is its value and any other an error.  No GPU: the calls return before any launch."""
import ctypes

import pytest
import torch

from flagrot_releaser_amd import kernels as K


def test_a_tensor_in_a_number_s_place():
    assert K.NATIVE.ask("fr_v2_chunk_bytes", 5, 16) == 2304
    assert K.NATIVE.ask("fr_v2_chunk_bytes", 5, torch.tensor(16)) == 2304
    with pytest.raises(ctypes.ArgumentError):
        K.NATIVE.ask("fr_v2_chunk_bytes", 5, torch.tensor([16, 16]))
    with pytest.raises(ctypes.ArgumentError):
        K.NATIVE.ask("fr_v2_chunk_bytes", 5, torch.tensor(16.0))


def test_pointers_and_bound_arguments():
    row = torch.zeros(4, dtype=torch.int64)
    args = (row, 0, row, 0, torch.tensor(0), 1, None, 1.0, None, 128)                       # no tokens: nothing is launched
    K.NATIVE.run("fr_head_fwht", *args)
    fn, plain = K.NATIVE.bind("fr_head_fwht", args)
    assert plain == (row.data_ptr(), 0, row.data_ptr(), 0, 0, 1, None, 1.0, None, 128) and fn(*plain) == 0

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


def test_step_writers_refuse_a_missing_ring_row_or_calibration():
    """at the C boundary: rows without names would be placed by a prompt's rule with an empty window"""
    from flagrot_releaser_amd import kivi as KV
    x = torch.zeros(64, dtype=torch.int64)
    for fmt in range(4, 10):
        full = dict(mask=x, CT=x, ring=x, dest=x, H=1)
        lacking = [dict(ring=None), dict(dest=None), dict(H=0), dict(H=-2)] + ([dict(CT=None)] if fmt in (6, 7, 9) else [])
        for less in lacking:
            a = {**full, **less}
            rc = K.NATIVE.ask("fr_step_write", fmt, x, 256, x, 1, a["H"], 16, a["mask"], a["CT"], x, None, a["ring"], a["dest"], 4, None)
            assert rc == -3 and K.NATIVE.last_error().startswith("fr_step_write"), (fmt, less, rc)
    for less in (dict(ring=None), dict(dest=None), dict(H=0)):
        a = {**dict(ring=x, dest=x, H=1), **less}
        rc = KV.NATIVE.ask("kv_step_write", x, 256, 1, a["H"], x, x, x, 0, a["ring"], a["dest"], 4, None)
        assert rc == 2 and KV.NATIVE.last_error().startswith("kv_step_write"), (less, rc)

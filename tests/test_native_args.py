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


def test_step_writers_take_one_slot_for_every_token(monkeypatch):
    """the number of tokens is the rows': slots that are fewer, of another shape, strided or elsewhere are not read"""
    from flagrot_releaser_amd import kivi as KV
    seen = []
    for lib in (K, KV):
        monkeypatch.setattr(lib.NATIVE, "run", lambda name, *a: seen.append((name, a)))
        monkeypatch.setattr(lib, "current_stream", lambda: 0)
    T, H = 3, 2
    kv, ring = torch.zeros(T, 2 * H, 128, dtype=torch.bfloat16), torch.zeros(8, 2 * H, 128, dtype=torch.bfloat16)
    dest, x = torch.arange(T), torch.zeros(4)
    calls = [lambda s: K.step_write(kv, s, "int4", x, 16, ring, dest, mask=x), lambda s: K.step_write(kv, s, "konly", x, 16, ring, dest, CT=x),
             lambda s: KV.step_write(kv, s, x, x, ring, dest)]
    good = torch.arange(T)
    for call in calls:
        for bad in (good[:2], torch.arange(T + 1), good.int(), good.view(T, 1), torch.empty(T, dtype=torch.int64, device="meta")):
            with pytest.raises(AssertionError):
                call(bad)
        assert not seen
        call(good)
        call(torch.arange(2 * T)[::2])                                 # every second one: a copy goes to the device
        packed = [next(t for t in a if isinstance(t, torch.Tensor) and t.dtype == torch.int64) for _, a in seen]
        assert packed[0].tolist() == [0, 1, 2] and packed[1].tolist() == [0, 2, 4] and packed[1].is_contiguous()
        seen.clear()
    with pytest.raises(AssertionError):
        K.step_write(kv, good, "konly", x, 16, ring, dest)             # key-only pages without their calibration


def test_partials_that_pairs_cannot_be_stored_to_are_refused():
    """head dim 128, more than one partial: outputs and (maximum, sum) move eight bytes at a time"""
    x = torch.zeros(64, dtype=torch.int64)
    at = x.data_ptr()

    def call(opart, mlpart, nsplit=2, variant=264):
        return K.NATIVE.ask("fr_v2_attn", 5, at, 512, at, at, 4, at, 1, 1, 16, nsplit, 8192, 1.0, None, None, 32, 0, 0, variant, 4, opart,
                            mlpart, at, at, 512, None, None, None, 0, 0, None, 4, 0)

    for bad in ((at + 4, at), (at, at + 4), (at + 12, at + 4)):
        assert call(*bad) == -3 and "8-byte" in K.NATIVE.last_error()
    assert call(at + 4, at, nsplit=3, variant=264 | K.GEN) == -3

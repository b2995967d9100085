"""Where a prompt's BF16 rows go (flagrot_releaser_amd.backend), on the CPU: the arguments that reach fr_ring_rows, with the
launches themselves replaced."""
import numpy as np
import pytest
import torch

from flagrot_releaser_amd import backend as BK
from flagrot_releaser_amd import kernels as K
from flagrot_releaser_amd import kivi as KV

S, W, R, HKV, G = 4, 32, 3, 2, 4                                      # R request rows and the spare one
SLOTS = S + W


@pytest.fixture
def sent(monkeypatch):
    """(base, start) of every fr_ring_rows call"""
    calls = []
    monkeypatch.setattr(K, "current_stream", lambda: 0)
    monkeypatch.setattr(KV, "current_stream", lambda: 0)
    monkeypatch.setattr(KV.NATIVE, "run", lambda name, *args: None)

    def run(name, *args):
        if name == "fr_ring_rows":
            base, sink, window, start = args[8:12]
            assert (sink, window) == (S, W) and type(base) is int and type(start) is int
            calls.append((base, start))
    monkeypatch.setattr(K.NATIVE, "run", run)
    return calls


def _layer(kind, planner=None):
    planner = planner or BK.StepPlanner(kind, HKV, G, 256, 4, R, S, W, "cpu", plan_fn=lambda B: (1, 256))
    if kind == "kivi2":
        pool = torch.zeros(32, HKV, KV.chunk_bytes(128, False), dtype=torch.uint8)
        return BK.KiviDecodeLayer(HKV, G, pool, planner, torch.zeros(HKV, 8, 128), torch.zeros(HKV, 8), torch.ones(HKV, 128))
    pool = torch.zeros(32, HKV, K.v2_chunk_bytes(16, 128, kind), dtype=torch.uint8)
    return BK.DecodeLayer(kind, HKV, G, pool, planner, wmask=torch.zeros(2 * HKV, 4, dtype=torch.uint8))


def _chunk(layer, n, req, start):
    kv, slots = torch.zeros(n, 2 * HKV, 128, dtype=torch.bfloat16), torch.arange(n)
    extra = (torch.arange(16, dtype=torch.int32),) if isinstance(layer, BK.KiviDecodeLayer) else ()
    layer.prefill_chunk(kv, slots, req, start, *extra)


@pytest.mark.parametrize("kind", ["int4a", "kivi2"])
@pytest.mark.parametrize("number", [int, np.int64, torch.tensor, lambda x: torch.tensor([x], dtype=torch.int32)])
def test_positions_and_requests_in_any_integer_form(sent, kind, number):
    layer = _layer(kind)
    _chunk(layer, 40, number(2), number(37))
    layer.prefill(torch.zeros(40, 2 * HKV, 128, dtype=torch.bfloat16), torch.arange(40), number(1))
    assert sent == [(2 * SLOTS, 37), (SLOTS, 0)]


@pytest.mark.parametrize("kind", ["int4a", "kivi2"])
def test_request_rows_follow_the_rules_of_an_index(sent, kind):
    layer = _layer(kind)
    kv, slots = torch.zeros(5, 2 * HKV, 128, dtype=torch.bfloat16), torch.arange(5)
    layer.prefill(kv, slots, -1)                                       # the spare row
    layer.prefill(kv, slots, -R - 1)
    assert sent == [(R * SLOTS, 0), (0, 0)]
    for outside in (R + 1, -R - 2):
        with pytest.raises(IndexError):
            layer.prefill(kv, slots, outside)
        with pytest.raises(IndexError):
            _chunk(layer, 5, outside, 0)
    with pytest.raises(TypeError):
        layer.prefill(kv, slots, 1.0)
    if kind == "kivi2":                                                # a chunk of these pages always refused negative rows
        with pytest.raises(IndexError):
            _chunk(layer, 5, -1, 0)
    else:
        _chunk(layer, 5, -1, 0)
        assert sent[2:] == [(R * SLOTS, 0)]


def test_rows_that_do_not_fit_the_ring_are_refused(monkeypatch):
    monkeypatch.setattr(K, "current_stream", lambda: 0)
    monkeypatch.setattr(K.NATIVE, "run", lambda name, *args: None)
    kv, dest = torch.zeros(3, 4, 128, dtype=torch.bfloat16), torch.arange(3)
    ring = torch.zeros(6, 4, 128, dtype=torch.bfloat16)
    K.ring_rows(kv, ring, dest=dest)
    K.ring_rows(kv, ring, base=2, sink=1, window=3)
    K.ring_rows(kv, ring.view(3, 2, 4, 128), dest=dest)
    for bad in (dict(ring=torch.zeros(6, 6, 128, dtype=torch.bfloat16)), dict(ring=torch.zeros(6, 2, 256, dtype=torch.bfloat16)),
                dict(ring=torch.zeros(6, 8, 64, dtype=torch.bfloat16)), dict(ring=ring[:, :2]), dict(ring=ring.float()),
                dict(ring=ring.to("meta")), dict(ring=torch.zeros(6 * 512 + 1, dtype=torch.bfloat16)[1:].view(6, 4, 128)),
                dict(dest=dest.int()), dict(dest=dest[:2]), dict(dest=dest.to("meta")), dict(dest=torch.zeros(6, dtype=torch.int64)[::2]),
                dict(dest=None, base=-1, sink=1, window=3), dict(dest=None, base=3, sink=1, window=3),
                dict(kv=kv.half()), dict(kv=kv[:, :3], ring=ring[:, :3].contiguous())):
        args = {**dict(kv=kv, ring=ring, dest=dest), **bad}
        with pytest.raises(AssertionError):
            K.ring_rows(args.pop("kv"), args.pop("ring"), **args)


@pytest.mark.parametrize("kind", ["int4a", "kivi2"])
@pytest.mark.parametrize("n", [1, 8, 9])
def test_steps_of_any_size_copy_their_rows_the_same_way(monkeypatch, kind, n):
    """one launch with the planner's destinations, whatever the number of rows: one rule for rows outside the ring"""
    calls = []
    monkeypatch.setattr(K, "current_stream", lambda: 0)
    monkeypatch.setattr(KV, "current_stream", lambda: 0)
    monkeypatch.setattr(KV.NATIVE, "run", lambda name, *args: None)
    monkeypatch.setattr(K.NATIVE, "run", lambda name, *args: calls.append((name, args)))
    planner = BK.StepPlanner(kind, HKV, G, 256, 16, 15, S, W, "cpu", plan_fn=lambda B: (1, 256))
    layer = _layer(kind, planner)
    sp = planner.prepare(torch.full((n,), 50, dtype=torch.int32), torch.zeros(n, 16, dtype=torch.int32), torch.arange(n),
                         homes=np.arange(n))
    layer.update(torch.zeros(n, 2 * HKV, 128, dtype=torch.bfloat16), sp)
    (args,) = [a for name, a in calls if name == "fr_ring_rows"]
    assert args[2] == n and args[6] is layer.ring and args[7] is sp.ring_dest and args[13] == 16 * SLOTS


def test_layers_share_the_rows_of_a_prompt_s_key_groups(monkeypatch):
    """int64 rows 0 .. of every whole group, sinks left out: one table per planner, not one per layer"""
    sent = []
    monkeypatch.setattr(K, "current_stream", lambda: 0)
    monkeypatch.setattr(KV, "current_stream", lambda: 0)
    monkeypatch.setattr(K.NATIVE, "run", lambda name, *args: None)
    monkeypatch.setattr(KV.NATIVE, "run", lambda name, *args: sent.append(args[4]) if name == "kv_k_encode" else None)
    planner = BK.StepPlanner("kivi2", HKV, G, 256, 4, R, S, W, "cpu", plan_fn=lambda B: (1, 256))
    for n in (70, 256, 300):                                          # past max_len the last two hold what the first do
        for layer in (_layer("kivi2", planner), _layer("kivi2", planner)):
            layer.prefill(torch.zeros(n, 2 * HKV, 128, dtype=torch.bfloat16), torch.arange(n), 0)
        a, b = sent[-2:]
        want = torch.arange(n // 32 * 32)
        want[:S] = -1
        assert torch.equal(a, want.view(-1, 32)) and torch.equal(a, b) and a.dtype == torch.int64 and a.is_contiguous()
        assert n > 256 or a.data_ptr() == b.data_ptr()

"""Head dim 256 decode whose parts are shared out by the sequences' lengths on the device: coverage of every token by one
part, sequences without parts, the largest batch of the rule and the first beyond it.  Against the oracle, the bar of
test_gpu_decode.py (2e-3 + 1e-2 |ref|); window rows, a start position and an empty sequence are in every case.  Which of the
two ran shows in the partials: fixed ranges write every slot of [sequence][KV head, tile][split | rows], parts by length the
first ones of [KV head, tile][parts | rows of every sequence]."""
import os
import subprocess
import sys

import pytest
import torch

from tests.test_gpu_decode import _head_dim_256

pytestmark = pytest.mark.gpu
ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
# lengths (the empty sequence of the helper comes on top); three splits of at least 512 tokens, a tile of 4 and one of 2 heads
# on 4 KV heads: 24 workgroups a sequence, shared out from 384 on (of 256 CUs)
UNEVEN = [1600, 1, 17, 64, 65, 333, 700, 1100, 2, 513, 1599, 40, 63, 128, 900, 0]
CASES = {"uneven": (UNEVEN, True), "even": ([1530] * 15, True), "the longest alone": ([1537] + [5] * 15, True),
         "64 sequences": ([1537] + list(range(1, 63)), True), "65 sequences": ([1537] + list(range(1, 64)), False),
         "few workgroups": ([1537, 300, 700], False)}


def parts_by_length(lens, nsplit, chunk, kv_start, groups):
    """how many parts a (KV head, q tile) has in all: of 16 candidate lengths the smallest whose parts fit beside the window rows'
    workgroups, two a CU; the plan's chunk if none does"""
    start = kv_start & ~63
    units = [max(0, -(-(min(n, nsplit * chunk) - start) // 64)) for n in lens]
    B, cap, total = len(lens), chunk // 64, sum(units)
    places = max(1, min(B * nsplit, 512 // groups - B))
    hi = min(cap, total // (places - B) + 1) if places > B else cap
    lo = min(hi, max(1, -(-total // places)))
    step = max(1, (hi - lo + 14) // 15)
    count = lambda m: sum(-(-u // m) for u in units)                                                # noqa: E731
    return next((count(m) for m in (min(hi, lo + step * k) for k in range(16)) if count(m) <= places), count(hi))


def check(dev, fmt, P, G, Hkv, lens, shared, kv_start=3):
    B, groups = len(lens) + 1, Hkv * ((G + 3) // 4)
    seen = []

    def partials(nsplit, chunk, written):
        seen.append(nsplit)
        if nsplit == 1 or not shared:
            assert written.all()
            return
        n = parts_by_length(lens + [0], nsplit, chunk, kv_start, groups)
        want = torch.zeros(B * (nsplit + 1), dtype=torch.bool)
        want[:n] = want[B * nsplit:] = True
        assert n < B * nsplit and (written.view(groups, -1) == want).all()

    _head_dim_256(dev, fmt, P, G, Hkv, lens=lens, seed=B, kv_start=kv_start, partials=partials)
    assert seen == [1, 3] and max(lens) > 2 * 512


@pytest.mark.parametrize("fmt,P", [("konlya", 16), ("int4a", 32)])
@pytest.mark.parametrize("name", CASES)
def test_parts_by_length(dev, name, fmt, P):
    check(dev, fmt, P, 6, 4, *CASES[name])


@pytest.mark.parametrize("fmt", ["konlya2", "int2a"])
def test_one_tile_and_a_start_beyond_the_first_units(dev, fmt):
    """2-bit pages, one q tile per KV head, tokens 0 .. 129 masked: two units of 64 tokens are no part's, and several
    sequences end before the start"""
    check(dev, fmt, 16, 4, 4, UNEVEN + UNEVEN, True, kv_start=130)


def test_fixed_ranges_by_request(dev):
    """FLAGROT_DECODE_STATIC=1 (read once, so in a process of its own)"""
    code = ("import torch\nfrom tests import test_gpu_wide_share as T\n"
            "T.check(torch.device('cuda:0'), 'konlya', 16, 6, 4, T.UNEVEN, False)\nprint('fixed ranges ok')")
    env = dict(os.environ, FLAGROT_DECODE_STATIC="1")
    r = subprocess.run([sys.executable, "-c", code], cwd=ROOT, env=env, capture_output=True, text=True, timeout=120)
    assert r.returncode == 0 and "fixed ranges ok" in r.stdout, r.stdout + r.stderr

"""Head dim 256 decode whose parts are shared out by the sequences' lengths on the device: coverage of every token by one
part, sequences without parts, the largest batch of the rule and the first beyond it.  Against the oracle, the bar of
test_gpu_decode.py (2e-3 + 1e-2 |ref|); window rows, a start position and an empty sequence are in every case."""
import pytest

from tests.test_gpu_decode import _head_dim_256

pytestmark = pytest.mark.gpu
# lengths (the empty sequence of the helper comes on top); three splits of at least 512 tokens, a tile of 4 and one of 2 heads
# on 4 KV heads: 24 workgroups a sequence, shared out from 384 on
UNEVEN = [1600, 1, 17, 64, 65, 333, 700, 1100, 2, 513, 1599, 40, 63, 128, 900, 0]
CASES = {"uneven": (UNEVEN, True), "even": ([1530] * 15, True), "the longest alone": ([1537] + [5] * 15, True),
         "64 sequences": ([1537] + list(range(1, 63)), True), "65 sequences": ([1537] + list(range(1, 64)), False),
         "few workgroups": ([1537, 300, 700], False)}


@pytest.mark.parametrize("fmt,P", [("konlya", 16), ("int4a", 32)])
@pytest.mark.parametrize("name", CASES)
def test_parts_by_length(dev, name, fmt, P):
    lens, shared = CASES[name]
    B = len(lens) + 1
    assert (B <= 64 and 2 * 3 * 8 * B >= 3 * 256) == shared and max(lens) > 2 * 512
    _head_dim_256(dev, fmt, P, 6, 4, lens=lens, seed=B)

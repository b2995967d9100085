"""The split merge of the KIVI-style decode against the same merge in FP64 over the call's own partials, where its slices of
partials can go wrong: one partial to a slice, one more than that, one round of eight to a slice and a little more, with
sequences that leave most or all partials empty; both head dims."""
import math

import pytest
import torch

from tests.test_gpu_kivi import _filled_cache

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("hd", [128, 256])
@pytest.mark.parametrize("ns", [7, 8, 63, 64, 71])
def test_merge_of_splits(dev, ns, hd):
    from flagrot_releaser_amd import kivi as KV
    Hkv, G, T, lens, tails = 2, 3, 32, [32 * ns - 5, 40, 33], [9, 0, 0]
    g = torch.Generator().manual_seed(ns)
    pool, bt, _, _ = _filled_cache(dev, lens, Hkv, g, hd=hd)
    ring = torch.randn(4 * T, 2 * Hkv, hd, generator=g).bfloat16().to(dev)
    q = torch.randn(3, Hkv * G, hd, generator=g).bfloat16().to(dev)
    num = lambda x: torch.tensor(x, dtype=torch.int32, device=dev)                                  # noqa: E731
    ws = KV.Workspace(3 * Hkv * (ns + 1), G, hd, dev)
    ws.ml = torch.cat([ws.ml, ws.ml[:1]])[1:]                                                       # pairs at 4 bytes from 8
    out = torch.full((3, Hkv * G * hd + 3), 7.0, dtype=torch.bfloat16, device=dev)                  # rows of an odd stride
    KV.attn(q, pool, bt.to(dev), num(lens), out[:, :-3], ns, 32, ws, math.log2(math.e) / math.sqrt(hd), 33, G, ring=ring,
            tail_len=num(tails), tail_idx=num([2, 0, 1]), T=T)
    ml = ws.ml.view(3, Hkv, ns + 1, G, 2).double()
    part = ws.opart.view(3, Hkv, ns + 1, G, hd).double()
    some = ml[..., 0] > float("-inf")
    top = ml[..., 0].amax(2, keepdim=True)
    w = torch.where(some, torch.exp2(ml[..., 0] - torch.where(top > float("-inf"), top, 0.0)), 0.0)
    part = torch.where(some[..., None], part, 0.0)
    total = (w * ml[..., 1]).sum(2)[..., None]
    safe = torch.where(total > 0, total, 1.0)
    want, size = (w[..., None] * part).sum(2) / safe, (w[..., None] * part.abs()).sum(2) / safe
    got = out[:, :-3].view(3, Hkv, G, hd).double()
    # FP32: exponents of up to 100 x 2^-24 and the roundings of the sums; BF16: half a unit of the result on top
    assert ((got - want).abs() <= 1e-5 * size + 2.0 ** -8 * want.abs()).all()
    assert not got[2].any() and (out[:, -3:] == 7.0).all()

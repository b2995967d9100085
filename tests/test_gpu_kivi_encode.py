"""The key group encoder at the sizes where its tiling can go wrong: calibration sets that do not fill a tile of 32
queries, end between two tiles, or need more than one round of 64, groups with missing tokens, both head dims and both
meta formats.  Codes and meta are bit-equal to the oracle given the stored flags, and a stored choice may differ from
the oracle's only where its FP64 margin is below 1e-3 (FP32 sums in another order)."""
import math

import numpy as np
import pytest
import torch

from oracle import kivi as OK
from tests.test_gpu_kivi import F8, _calib, _cb, _group_rows, _groups, _stored_key_flags

pytestmark = pytest.mark.gpu


@F8
@pytest.mark.parametrize("hd", [128, 256])
@pytest.mark.parametrize("NQ", [1, 31, 33, 65, 160])
def test_query_tiles(dev, NQ, hd, f8):
    from flagrot_releaser_amd import kivi as KV
    g = torch.Generator().manual_seed(NQ)
    NG, Hkv, qsc = 3, 2, 1 / math.sqrt(hd)
    rows, rows2, sidx, dslot = _groups(NG, Hkv, g, hd=hd)
    sidx[0, 0] = -1                                                    # a sink
    dslot = torch.cat([dslot, torch.full((1, 32), -1)])                # a group that is switched off
    sidx = torch.cat([sidx, sidx[:1]])
    qs, lz, _ = _calib(Hkv, NQ, g, hd)
    pool = torch.zeros(2 * NG + 3, Hkv, _cb(f8, hd), dtype=torch.uint8, device=dev)
    KV.k_encode(rows.to(dev), sidx.to(dev), dslot.to(dev), qs.to(dev), lz.to(dev), qsc, pool, Hkv, hd,
                src2=rows2.to(dev), f8=f8)
    torch.cuda.synchronize()
    got = pool.cpu().numpy()
    want = np.zeros_like(got)
    for n in range(NG):
        xb, valid = _group_rows(rows, rows2, sidx[n], Hkv)
        for h in range(Hkv):
            enc = OK.k_encode_group(xb[:, h], valid, qs[h].numpy(), lz[h].numpy(), qsc, f8=f8)
            local, whole = _stored_key_flags(got, dslot[n].numpy(), h, f8, hd)
            OK.pack_key_group(want, h, dslot[n].numpy(), valid, *OK.k_stored(enc, local, whole, f8=f8), f8=f8)
            assert whole == enc["useF"] or enc["marginF"] < 1e-3, (n, h, enc["marginF"])
            if not whole and not enc["useF"]:
                assert (enc["marginH"][local != enc["useH"]] < 1e-3).all(), (n, h)
    assert np.array_equal(got, want), "key codes / meta differ from the oracle given the stored flags"

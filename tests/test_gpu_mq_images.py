"""Prefill from tile images against the kernel that converts for every tile: the tiles hold the same fp16 numbers and the matrix
products run in the same order, so the partials are the same bits.  One block to several (the copies are three deep), ragged
ends, items that start inside a request, requests that share pages, heads in passes of unequal size, both code widths; the
pages of the static formats through the C entry, which the front end does not send this way."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def by_entry(MQ, q16, pool, bt, plan, G, shift, konly, int2, heads):
    """frmq_attn_images itself"""
    from flagrot_releaser_amd.native import current_stream
    Hkv = pool.shape[1]
    opart = q16.new_empty((plan.nitems, Hkv, plan.rows, 128), dtype=torch.float32)
    ml = q16.new_empty((plan.nitems, Hkv, plan.rows, 2), dtype=torch.float32)
    images = q16.new_empty(heads * plan.nblocks * MQ.IMAGE, dtype=torch.uint8)
    MQ.NATIVE.run("frmq_attn_images", q16, pool, pool.stride(0), bt, bt.stride(0), plan.tiles, plan.items, plan.nitems,
                  plan.tile_block, plan.block_recs, plan.nblocks, Hkv, G, shift, int(konly) + 2 * int(int2), images, heads, opart, ml,
                  current_stream(), plan.kmin)
    return opart, ml


@pytest.mark.parametrize("kind", ["konlya", "konlya2", "int4a", "int2a"])
@pytest.mark.parametrize("reqs,G,Hkv,shift,sink,heads", [
    ([(0, 0, 33, 33, 0)], 8, 1, 0, 0, 1),                              # one block
    ([(0, 0, 70, 190, 120), (1, 70, 230, 160, 0)], 4, 3, 0, 4, 2),     # up to three; two passes of heads; rows that see sinks only
    ([(1, 0, 64, 1100, 1036), (0, 64, 300, 500, 264), (1, 300, 301, 700, 699)], 3, 2, 40, 0, 2),
    ([(0, 0, 100, 100, 0)], 4, 2, 40, 0, 2),                           # the first forty rows see no key
    ([(0, 0, 512, 2048, 1536)], 5, 3, 0, 0, 1),
])
def test_same_partials(dev, monkeypatch, reqs, G, Hkv, shift, sink, heads, kind):
    from flagrot_releaser_amd import kernels as K
    from flagrot_releaser_amd import prefill_mq as MQ
    g = torch.Generator(device=dev).manual_seed(len(reqs) + G)
    int2, konly = kind in K.INT2_FMTS, kind in K.K2
    n, pages = reqs[-1][2], 2 * 128 + 3
    pool = torch.full((pages, Hkv, K.v2_chunk_bytes(16, 128, kind)), 255, dtype=torch.uint8, device=dev)   # free pages: NaN scales
    bt = torch.randperm(pages, generator=g, device=dev)[:256].view(2, 128).int()
    C = torch.randn(Hkv, 128, 128, generator=g, device=dev)
    CT = (C @ C.transpose(1, 2)).contiguous()
    mask = (torch.rand(2 * Hkv, 4, generator=g, device=dev) < 0.5).to(torch.uint8)
    for r in (0, 1):
        L = max(end for row, _, _, end, _ in reqs if row == r) if any(q[0] == r for q in reqs) else 0
        if L:
            pos = torch.arange(L, device=dev)
            kv = torch.randn(L, 2 * Hkv, 128, generator=g, device=dev).bfloat16()
            slots = bt[r].long()[pos // 16] * 16 + pos % 16
            if konly:
                K.cb_write(kv, slots, CT, torch.ones(Hkv, 128, device=dev), kind, pool, 16)
            else:
                K.v2_write(kv, slots, mask, 32, pool, 16, fmt=kind)
    q16 = (0.3 * torch.randn(n, G * Hkv, 128, generator=g, device=dev)).half()
    monkeypatch.setattr(MQ, "IMAGE_READS", 1)
    monkeypatch.setattr(MQ, "IMAGE_REUSE", 0)
    monkeypatch.setattr(MQ, "image_heads", lambda *_: heads)
    plan = MQ.build_plan(reqs, G, Hkv, shift, dev, sink=sink, kernel=4)
    assert plan.nblocks > 0
    if konly:
        got = MQ.attn(q16, pool, bt, plan, G, shift, True, int2)
    else:
        got = by_entry(MQ, q16, pool, bt, plan, G, shift, False, int2, heads)
    plan.nblocks = 0
    want = MQ.attn(q16, pool, bt, plan, G, shift, konly, int2)
    stored = torch.ones_like(want[1][..., 0], dtype=torch.bool)         # rows past a tile's last token are never written
    for t in range(plan.ntiles):
        first, count, used = (int(plan.tiles.view(-1, 9)[t, c]) for c in (6, 7, 3))
        stored[first:first + count, :, used * G:] = False
    assert torch.equal(got[1][stored], want[1][stored])                 # rows without a key among them: (-inf, 0)
    blind = stored & (want[1][..., 0] == float("-inf"))
    assert (want[1][blind][:, 1] == 0).all() and blind.any() == any(s < max(shift, sink) for *_, s in reqs)
    seen = stored & ~blind
    assert seen.any() and torch.equal(got[0][seen], want[0][seen])

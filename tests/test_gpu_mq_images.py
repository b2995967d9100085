"""Prefill from tile images against the kernel that converts for every tile: the tiles hold the same fp16 numbers and the matrix
products run in the same order, so the partials are the same bits.  One block to several (the copies are three deep), ragged
ends, items that start inside a request, requests that share pages, heads in passes of unequal size, both code widths."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("int2", [False, True])
@pytest.mark.parametrize("reqs,G,Hkv,shift,sink,heads", [
    ([(0, 0, 33, 33, 0)], 8, 1, 0, 0, 1),                              # one block
    ([(0, 0, 70, 190, 120), (1, 70, 230, 160, 0)], 4, 3, 0, 4, 2),     # up to three; two passes of heads
    ([(1, 0, 64, 1100, 1036), (0, 64, 300, 500, 264), (1, 300, 301, 700, 699)], 3, 2, 40, 0, 2),
    ([(0, 0, 512, 2048, 1536)], 5, 3, 0, 0, 1),
])
def test_same_partials(dev, monkeypatch, reqs, G, Hkv, shift, sink, heads, int2):
    from flagrot_releaser_amd import kernels as K
    from flagrot_releaser_amd import prefill_mq as MQ
    g = torch.Generator(device=dev).manual_seed(len(reqs) + G)
    kind = "konlya2" if int2 else "konlya"
    n, pages = reqs[-1][2], 2 * 128 + 3
    pool = torch.full((pages, Hkv, K.v2_chunk_bytes(16, 128, kind)), 255, dtype=torch.uint8, device=dev)   # free pages: NaN scales
    bt = torch.randperm(pages, generator=g, device=dev)[:256].view(2, 128).int()
    C = torch.randn(Hkv, 128, 128, generator=g, device=dev)
    CT = (C @ C.transpose(1, 2)).contiguous()
    for r in (0, 1):
        L = max(end for row, _, _, end, _ in reqs if row == r) if any(q[0] == r for q in reqs) else 0
        if L:
            pos = torch.arange(L, device=dev)
            kv = torch.randn(L, 2 * Hkv, 128, generator=g, device=dev).bfloat16()
            K.cb_write(kv, bt[r].long()[pos // 16] * 16 + pos % 16, CT, torch.ones(Hkv, 128, device=dev), kind, pool, 16)
    q16 = (0.3 * torch.randn(n, G * Hkv, 128, generator=g, device=dev)).half()
    monkeypatch.setattr(MQ, "IMAGE_READS", 1)
    monkeypatch.setattr(MQ, "IMAGE_REUSE", 0)
    monkeypatch.setattr(MQ, "image_heads", lambda *_: heads)
    plan = MQ.build_plan(reqs, G, Hkv, shift, dev, sink=sink, kernel=4)
    assert plan.nblocks > 0
    got = MQ.attn(q16, pool, bt, plan, G, shift, True, int2)
    plan.nblocks = 0
    want = MQ.attn(q16, pool, bt, plan, G, shift, True, int2)
    seen = want[1][..., 0] > float("-inf")                              # rows without a key, and those past the tile: never written
    for t in range(plan.ntiles):
        first, count, used = (int(plan.tiles.view(-1, 9)[t, c]) for c in (6, 7, 3))
        seen[first:first + count, :, used * G:] = False
    assert seen.any()
    assert torch.equal(got[1][seen], want[1][seen]) and torch.equal(got[0][seen], want[0][seen])

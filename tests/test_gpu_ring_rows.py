"""fr_ring_rows against torch indexing, bit for bit: prompts and chunks that end inside, at and past the sinks and the
window, rings without sinks or without window, centring, strided rows, both head dims, and rows named one by one."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def _want(ring, kv, kmu, pairs):
    H = kv.shape[1] // 2
    rows = kv.clone()
    if kmu is not None:
        rows[:, :H] = (kv[:, :H].float() - kmu).to(torch.bfloat16)
    for t, r in pairs:
        ring[r] = rows[t]
    return ring


@pytest.mark.parametrize("S,W,start,n", [(4, 128, 0, 700), (4, 128, 0, 100), (4, 128, 2, 1), (4, 128, 3, 131), (0, 32, 5, 33),
                                         (7, 0, 0, 3), (7, 0, 5, 20), (4, 16, 900, 5), (0, 1, 0, 1)])
@pytest.mark.parametrize("dim,centred", [(128, False), (128, True), (256, True)])
def test_prompt_rows(dev, S, W, start, n, dim, centred):
    from flagrot_releaser_amd import kernels as K
    g = torch.Generator().manual_seed(n)
    H, req = 3, 1
    wide = torch.randn(n, 2 * H + 1, dim, generator=g).bfloat16()
    kv = wide[:, :2 * H]                                               # rows with a stride of their own
    kmu = torch.randn(H, dim, generator=g) if centred else None
    ring0 = torch.randn(3 * (S + W), 2 * H, dim, generator=g).bfloat16()
    pairs = []
    for t in range(n):
        p = start + t
        if p < S or p >= start + n - W:
            pairs.append((t, req * (S + W) + (p if p < S else S + (p - S) % W)))
    ring = ring0.to(dev)
    K.ring_rows(wide.to(dev)[:, :2 * H], ring, kmu=None if kmu is None else kmu.to(dev), base=req * (S + W), sink=S, window=W,
                start=start)
    assert torch.equal(ring.cpu(), _want(ring0.clone(), kv, kmu, pairs))


def test_named_rows(dev):
    from flagrot_releaser_amd import kernels as K
    g = torch.Generator().manual_seed(2)
    H, n = 8, 65
    kv = torch.randn(n, 2 * H, 128, generator=g).bfloat16()
    kmu = torch.randn(H, 128, generator=g)
    dest = torch.randperm(200, generator=g)[:n]
    dest[7] = -1
    ring0 = torch.randn(200, 2 * H, 128, generator=g).bfloat16()
    ring = ring0.to(dev)
    K.ring_rows(kv.to(dev), ring, kmu=kmu.to(dev), dest=dest.to(dev))
    want = _want(ring0.clone(), kv, kmu, [(t, r) for t, r in enumerate(dest.tolist()) if r >= 0])
    assert torch.equal(ring.cpu(), want)


@pytest.mark.parametrize("dim", [128, 256])
@pytest.mark.parametrize("n", [1, 8, 9, 65])
def test_named_rows_as_they_are(dev, n, dim):
    """a decode step without centring; rows that the ring does not have are left out"""
    from flagrot_releaser_amd import kernels as K
    g = torch.Generator().manual_seed(n)
    H, have = 2, 120
    kv = torch.randn(n, 2 * H, dim, generator=g).bfloat16()
    dest = torch.randperm(have, generator=g)[:n]
    if n > 8:
        dest[0], dest[3], dest[5], dest[8] = have, -1, 1 << 40, -(1 << 62)
    ring0 = torch.randn(have, 2 * H, dim, generator=g).bfloat16()
    room = torch.zeros(2 * have, 2 * H, dim, dtype=torch.bfloat16, device=dev)       # rows behind the ring must stay as they are
    room[:have] = ring0.to(dev)
    K.ring_rows(kv.to(dev), room[:have], dest=dest.to(dev))
    want = _want(ring0.clone(), kv, None, [(t, r) for t, r in enumerate(dest.tolist()) if 0 <= r < have])
    assert torch.equal(room[:have].cpu(), want) and not room[have:].any()

"""The one-launch cache update of a decode step against the writer and the row copy by themselves, byte for byte: one token to
more than the decode step's writer takes, padding rows without a page slot or a ring row, rows that are views."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def _step(T, H, g, dev, strided):
    wide = torch.randn(T, 2 * H + strided, 128, generator=g, device=dev).bfloat16()
    kv = wide[:, strided:]
    slots = torch.randperm(3 * T, generator=g, device=dev)[:T]
    dest = torch.randperm(2 * T, generator=g, device=dev)[:T]
    if T > 2:
        slots[1], dest[2], dest[0] = -1, -1, 2 * T                     # no page, no ring row, past the ring
    return kv, slots, dest, torch.randn(2 * T, 2 * H, 128, generator=g, device=dev).bfloat16()


@pytest.mark.parametrize("fmt", ["konly", "konlya2", "int4", "int2a"])
@pytest.mark.parametrize("T,H,strided,centred", [(1, 1, 0, True), (3, 5, 1, True), (17, 8, 0, False), (129, 8, 2, True)])
def test_flagrot(dev, fmt, T, H, strided, centred):
    from flagrot_releaser_amd import kernels as K
    g = torch.Generator(device=dev).manual_seed(T)
    kv, slots, dest, ring = _step(T, H, g, dev, strided)
    kmu = torch.randn(H, 128, generator=g, device=dev) if centred else None
    mask = (torch.rand(2 * H, 4, generator=g, device=dev) < 0.5).to(torch.uint8)
    C = torch.randn(H, 128, 128, generator=g, device=dev)
    CT, co = (C @ C.transpose(1, 2)).contiguous(), torch.ones(H, 128, device=dev)
    pool = [torch.zeros(3 * T // 16 + 1, H, K.v2_chunk_bytes(16, 128, fmt), dtype=torch.uint8, device=dev) for _ in range(2)]
    rings = [ring, ring.clone()]
    K.step_write(kv, slots, fmt, pool[0], 16, rings[0], dest, mask=mask, CT=CT, kmu=kmu)
    if fmt in K.K2:
        K.cb_write(kv, slots, CT, co, fmt, pool[1], 16, kmu=kmu)
    else:
        K.v2_write(kv, slots, mask, 32, pool[1], 16, fmt=fmt, kmu=kmu)
    K.ring_rows(kv, rings[1], kmu=kmu, dest=dest)
    assert torch.equal(pool[0], pool[1]) and torch.equal(rings[0], rings[1])
    assert pool[0].any()


@pytest.mark.parametrize("f8", [False, True])
@pytest.mark.parametrize("T,H,strided", [(1, 1, 0), (3, 5, 1), (33, 8, 2)])
def test_kivi(dev, f8, T, H, strided):
    from flagrot_releaser_amd import kernels as K
    from flagrot_releaser_amd import kivi as KV
    g = torch.Generator(device=dev).manual_seed(T)
    kv, slots, dest, ring = _step(T, H, g, dev, strided)
    co = torch.rand(H, 128, generator=g, device=dev)
    pool = [torch.zeros(3 * T // 16 + 1, H, KV.chunk_bytes(128, f8), dtype=torch.uint8, device=dev) for _ in range(2)]
    rings = [ring, ring.clone()]
    KV.step_write(kv, slots, co, pool[0], rings[0], dest, f8=f8)
    KV.v_write(kv, slots, co, None, pool[1], H, 128, f8=f8)
    K.ring_rows(kv, rings[1], dest=dest)
    assert torch.equal(pool[0], pool[1]) and torch.equal(rings[0], rings[1])
    assert pool[0].any()

"""The static writer stores value words whole, merged or field by field, by how the slots of eight consecutive tokens lie:
whole-pool bytes against the same tokens written one call at a time (field by field, pinned by test_gpu_writers.py)."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("fmt", ["int4", "int4a", "int2a"])
@pytest.mark.parametrize("page", [16, 32])
@pytest.mark.parametrize("first", [0, 1, 5, 7, 8])
def test_runs_of_slots(fmt, page, first):
    from flagrot_releaser_amd import kernels as K
    dev = torch.device("cuda:0")
    g = torch.Generator().manual_seed(31 * first + page)
    T, H = 67, 2
    kv = torch.randn(T, 2 * H, 128, generator=g).bfloat16().to(dev)
    mask = (torch.rand(2 * H, 4, generator=g) < 0.5).to(torch.uint8).to(dev)
    slots = torch.arange(first, first + T, device=dev)
    slots[40:] += 11                                      # a second request begins inside a group of eight tokens
    slots[50] = -1
    npg = (T + first + 11) // page + 2
    pool = torch.randint(0, 256, (npg, H, K.v2_chunk_bytes(page, 128, fmt)), dtype=torch.uint8, generator=g).to(dev)
    want, got = pool.clone(), pool.clone()
    for t in range(T):
        K.v2_write(kv[t:t + 1], slots[t:t + 1].contiguous(), mask, 32, want, page, fmt=fmt)
    K.v2_write(kv, slots, mask, 32, got, page, fmt=fmt)
    assert torch.equal(got, want)

"""The selecting writer's launch forms (one workgroup per token, whole-prompt kernels) write the same pool bytes: calls on
either side of 1024 (token, head) pairs, where the form changes, against the same tokens in calls of up to 97, whose bytes
the oracle pins in test_gpu_writers.py."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def dev():
    return torch.device("cuda:0")


def _inputs(T, Hkv, D, g, dev):
    kv = torch.randn(T, 2 * Hkv, D, generator=g)
    kv[:, :Hkv, 5] *= 7
    kv[T // 2] = 0.0
    kv[T // 3, :, 32:64] *= 500.0
    kv[40:60] = kv[40:41].clone()                         # one token repeated
    kv[60:80] = 0.37                                      # constants
    kv[80:120, :, 64:96] = 0.0                            # ties in one group only
    kv[120:140] *= 1e-4
    qs = torch.randn(Hkv, 256, D, generator=g)
    qs[:, :, :8] *= 4
    CT = (qs.transpose(1, 2) @ qs / 256).transpose(1, 2).contiguous()
    kmu = torch.randn(Hkv, D, generator=g)
    return kv.bfloat16().to(dev), CT.to(dev), torch.ones(Hkv, D, device=dev), kmu.to(dev)


@pytest.mark.parametrize("D,Hkv,T", [(128, 2, 512), (128, 2, 513), (128, 3, 341), (256, 2, 512), (256, 2, 513), (256, 2, 1024),
                                     (256, 2, 1025), (256, 1, 2100)])
@pytest.mark.parametrize("page", [16, 32])
@pytest.mark.parametrize("kind", ["konly", "konlya", "konlya2"])
@pytest.mark.parametrize("first", [0, 3])                 # slots of the run: aligned to eight tokens or not
def test_forms_write_the_same_bytes(dev, kind, D, Hkv, T, first, page):
    from flagrot_releaser_amd import kernels as K
    g = torch.Generator().manual_seed(T + D + first)
    kv, CT, co, kmu = _inputs(T, Hkv, D, g, dev)
    npg = (T + first) // page + 2
    pool = torch.randint(0, 256, (npg, Hkv, K.v2_chunk_bytes(page, D, kind)), dtype=torch.uint8, generator=g).to(dev)
    slots = torch.arange(first, first + T, device=dev)
    slots[T // 4] = -1
    want, got = pool.clone(), pool.clone()
    for a in range(0, T, 97):
        K.cb_write(kv[a:a + 97], slots[a:a + 97].contiguous(), CT, co, kind, want, page, kmu=kmu)
    K.cb_write(kv, slots, CT, co, kind, got, page, kmu=kmu)
    assert torch.equal(got, want)
    if D == 128:
        got = pool.clone()
        K.cb_write3(kv, slots, CT, co, None, None, kind, got, page, split=False, kmu=kmu)
        assert torch.equal(got, want)

"""frmq_merge against the same fold in FP64: tiles of one to six items (four is where the form changes) in short and long
launches, items that saw no key (their outputs are never written), rows without any, tiles that end early, both head dims."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("fp32", [False, True])
@pytest.mark.parametrize("Dh,rows,G,N", [(128, 256, 8, 3), (128, 256, 4, 130), (128, 128, 3, 9), (128, 64, 5, 7), (256, 128, 6, 4),
                                         (256, 128, 4, 260)])
def test_fold_of_items(dev, Dh, rows, G, N, fp32):
    fold_check(dev, Dh, rows, G, N, fp32, [1 + (5 * i) % 6 for i in range(N)])


# below and above 8192 rows in the launch (one or four rows a wavefront); items around a step of 4 or 16 and around 64 lanes
@pytest.mark.parametrize("Dh,rows,G,N", [(128, 128, 1, 9), (128, 256, 3, 17), (256, 128, 5, 9), (256, 128, 1, 33)])
def test_fold_of_many_items(dev, Dh, rows, G, N):
    fold_check(dev, Dh, rows, G, N, True, [(5, 15, 16, 17, 18, 63, 64, 65, 70)[i % 9] for i in range(N)])


def fold_check(dev, Dh, rows, G, N, fp32, counts):
    from flagrot_releaser_amd import prefill_mq as MQ
    Hkv, per = 2, rows // G
    g = torch.Generator(device=dev).manual_seed(N)
    tokens = [per - (i % 3 if i % 2 else 0) for i in range(N)]
    T = torch.zeros(N, 9, dtype=torch.int32)
    T[:, 1] = T[:, 2] = torch.tensor([0] + tokens[:-1]).cumsum(0)
    T[:, 3], T[:, 7] = torch.tensor(tokens), torch.tensor(counts)
    T[:, 6] = T[:, 7].cumsum(0) - T[:, 7]
    items, m = sum(counts), sum(tokens)
    plan = MQ.Plan(ntiles=N, nitems=items, m=m, buf=T.flatten().to(dev), reqs=[], rows=rows, D=Dh)
    part = torch.randn(items, Hkv, rows, Dh, generator=g, device=dev)
    ml = torch.stack([40 * torch.rand(items, Hkv, rows, generator=g, device=dev) - 20,
                      0.5 + 99 * torch.rand(items, Hkv, rows, generator=g, device=dev)], -1)
    unseen = torch.rand(items, Hkv, rows, generator=g, device=dev) < 0.3
    ml[unseen] = torch.tensor([float("-inf"), 0.0], device=dev)
    part[unseen] = float("nan")
    out = torch.full((m, Hkv * G * Dh), 7.0, dtype=torch.bfloat16, device=dev)
    got, lse = MQ.merge(plan, part, ml, G, out=None if fp32 else out, fp32=fp32, want_lse=True)
    got = got.view(m, Hkv, G, Dh).double()
    lse = lse.view(Hkv, G, m)
    for i in range(N):
        first, used, row0 = int(T[i, 6]), tokens[i] * G, int(T[i, 1])
        x, top, mass = (t[first:first + counts[i], :, :used].double() for t in (part, ml[..., 0], ml[..., 1]))
        best = top.amax(0)
        seen = best > float("-inf")
        w = torch.exp2(top - torch.where(seen, best, torch.zeros_like(best)))             # 0 where an item saw no key
        total = (w * mass).sum(0)
        x = torch.where(w[..., None] > 0, x, torch.zeros_like(x))
        safe = torch.where(seen, total, torch.ones_like(total))
        mean, size = (w[..., None] * x).sum(0) / safe[..., None], (w[..., None] * x.abs()).sum(0) / safe[..., None]
        mine = got[row0:row0 + tokens[i]].permute(1, 0, 2, 3).reshape(Hkv, used, Dh)
        # FP32: exponents to 40 x 2^-24, a dozen roundings of 2^-24 (70 items: their weights fall off, no more of them count); BF16: half a unit of the result on top
        bar = 4e-6 * size + (0 if fp32 else 2.0 ** -8 * mean.abs()) + 1e-30
        assert ((mine - mean).abs() <= bar).all(), (i, counts[i], float(((mine - mean).abs() / bar).max()))
        mine = lse[:, :, row0:row0 + tokens[i]].permute(0, 2, 1).reshape(Hkv, used).double()
        want = torch.where(seen, (best + torch.log2(safe)) * 0.6931471805599453, best)
        assert torch.equal(mine == float("-inf"), ~seen)
        assert ((mine - want).abs()[seen] <= 1e-5).all()                                  # |lse| < 20: 2^-24 x 20, log2 to 2^-22

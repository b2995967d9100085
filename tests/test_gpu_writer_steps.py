"""The screened writer's workgroups of several 16-token steps: buffers in LDS are used again from step to step and the
undecided tokens of all steps are evaluated at the end.  Whole-pool bytes against small calls, which run one workgroup per
(token, head) and whose bytes the oracle pins in test_gpu_writers.py; exact ties, holes and odd rows lie in every step."""
import os
import subprocess
import sys

import pytest
import torch

pytestmark = pytest.mark.gpu
ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
# tokens x heads -> steps of a workgroup (what the library answers): 768 resident workgroups at head dim 128 (two steps from five
# on), 256 at 256 (at most eight)
SHAPES = [(128, 8, 2001, 2), (128, 8, 4000, 3), (128, 8, 5005, 4), (128, 8, 6203, 2), (256, 4, 2100, 3), (256, 4, 8201, 8)]


def tokens_of(D, Hkv, T):
    from flagrot_releaser_amd import kernels as K
    return K.NATIVE.ask("fr_cb_write_tokens", T, Hkv, D)


def check(kind, D, Hkv, T, page, first=5):
    from flagrot_releaser_amd import kernels as K
    dev = torch.device("cuda:0")
    g = torch.Generator().manual_seed(T + page)
    kv = torch.randn(T, 2 * Hkv, D, generator=g)
    kv[:, :Hkv, 5] *= 7
    kv *= 0.5 + torch.rand(T, 1, 1, generator=g)
    t = torch.arange(T)
    kv[t % 13 == 4] = 0.0                                  # every candidate reproduces the row: undecided
    kv[t % 37 == 9] = kv[9:10].clone()                     # one token repeated
    kv[t % 29 == 3] = 0.37                                 # constants
    kv[t % 17 == 6, :, 32:64] = 0.0                        # a tie in one group only
    kv[t % 41 == 11] *= 1e-4
    kv[t % 23 == 2, :, 64:96] *= 500.0
    qs = torch.randn(Hkv, 256, D, generator=g)
    qs[:, :, :8] *= 4
    CT = (qs.transpose(1, 2) @ qs / 256).transpose(1, 2).contiguous().to(dev)
    co = torch.ones(Hkv, D, device=dev)
    kv = kv.bfloat16().to(dev)
    slots = first + t
    slots[t >= T // 2] += 3                                # a second run of slots
    slots[t % 19 == 8] = -1
    slots = slots.to(dev)
    npg = (T + first + 3) // page + 2
    pool = torch.randint(0, 256, (npg, Hkv, K.v2_chunk_bytes(page, D, kind)), dtype=torch.uint8, generator=g).to(dev)
    want, got = pool.clone(), pool.clone()
    small = 1024 // Hkv
    assert tokens_of(D, Hkv, T) > 1 == tokens_of(D, Hkv, small)
    for a in range(0, T, small):
        K.cb_write(kv[a:a + small], slots[a:a + small].contiguous(), CT, co, kind, want, page)
    if D == 128:
        K.cb_write3(kv, slots, CT, co, None, None, kind, got, page, split=False)
    else:
        K.cb_write(kv, slots, CT, co, kind, got, page)
    assert torch.equal(got, want), (kind, D, T, page, int((got != want).sum()))


@pytest.mark.parametrize("kind", ["konly", "konlya", "konlya2"])
@pytest.mark.parametrize("page", [16, 32])
@pytest.mark.parametrize("D,Hkv,T,steps", SHAPES)
def test_steps_write_the_bytes_of_small_calls(dev, kind, D, Hkv, T, steps, page):
    assert tokens_of(D, Hkv, T) == 16 * steps
    check(kind, D, Hkv, T, page)


# prompts of few pairs: half a step of 8 tokens a workgroup while that makes 256 workgroups at most, a whole step beyond; first
# and last of the range, rests of one token
@pytest.mark.parametrize("D,Hkv,T,half", [(128, 8, 129, True), (128, 8, 256, True), (128, 8, 257, False), (128, 1, 1031, True),
                                          (256, 4, 257, True), (256, 2, 1024, True), (256, 2, 1025, False)])
@pytest.mark.parametrize("kind,page", [("konly", 32), ("konlya2", 16)])
def test_half_steps_write_the_bytes_of_small_calls(dev, kind, page, D, Hkv, T, half):
    assert (tokens_of(D, Hkv, T) == 8) == half and tokens_of(D, Hkv, 1024 // Hkv) == 1
    check(kind, D, Hkv, T, page)


@pytest.mark.parametrize("env", [{"FLAGROT_W3": "2"}, {"FLAGROT_W3_KAPPA": "0.1"}], ids=["every token exact", "a tenth of the bound"])
def test_screen_at_its_ends(dev, env):
    """FLAGROT_W3=2: every token takes the exact path at the end, full lists of undecided tokens.  FLAGROT_W3_KAPPA=0.1: the
    estimates decide on a tenth of their proven bound, matrix pipe included, and no choice changes (measured: none down to a
    hundredth of it on these rows, the first at three thousandths).  Both are read once per process."""
    code = ("from tests.test_gpu_writer_steps import check\n"
            "check('konlya', 128, 8, 4000, 16); check('konlya2', 256, 4, 8201, 32)\nprint('same bytes')\n")
    r = subprocess.run([sys.executable, "-c", code], cwd=ROOT, env={**os.environ, **env}, capture_output=True, text=True,
                       timeout=100)
    assert r.returncode == 0 and "same bytes" in r.stdout, r.stdout + r.stderr

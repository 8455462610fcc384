"""Top-k selection of rows of more than 1024 blocks (scored by a launch over the whole
device, selected from the stored scores): the oracle's rule exactly on the kernel's own
scores at the edges of the keys held per thread, and the bits of the one-launch selector
for every key type, group size and query layout."""

import numpy as np
import pytest
import torch

import interattn_amd as ia
from oracle import select as S
from tests._util import announce

pytestmark = pytest.mark.gpu

HKV, D = 2, 64
# 4, 8, 16 and 32 keys per thread of 1024, and rows longer than that
EDGES = [1025, 4096, 4097, 8193, 16384, 16385, 32768, 32769]


def _keys(pattern, nb, q, gen, device):
    kb = torch.randn((HKV, nb, D), device=device, generator=gen)
    if pattern == "dup5":
        kb = kb[:, torch.randint(0, 5, (nb,), device=device, generator=gen)]
    elif pattern == "zero":
        kb.zero_()
    elif pattern == "crowd":  # 400 copies of each head's best row: a crowded threshold bucket
        best = (kb * q.view(HKV, -1, D).sum(1)[:, None]).sum(-1).argmax(-1)
        at = torch.randperm(nb, device=device, generator=gen)[:400]
        for h in range(HKV):
            kb[h, at] = kb[h, best[h]].clone()
    elif pattern == "inf":
        at = torch.randperm(nb, device=device, generator=gen)[:60]
        kb[:, at[:30]], kb[:, at[30:]] = 3e38, -3e38
    return kb


@pytest.mark.parametrize("pattern", ["random", "dup5", "zero", "crowd", "inf"])
@pytest.mark.parametrize("nb", EDGES)
def test_rule_exact_on_stored_scores(nb, pattern, device):
    announce(f"long selection {nb} {pattern}")
    gen = torch.Generator(device=device)
    gen.manual_seed(nb)
    q = torch.randn((1, 4 * HKV, D), device=device, generator=gen)
    if pattern == "inf":
        q = q.abs() + 0.1
    kb = _keys(pattern, nb, q[0], gen, device)[None].bfloat16()
    seq = torch.tensor([nb * 16 - 7], device=device, dtype=torch.int32)
    idx, n, sc = ia.select_blocks_topk(q.bfloat16(), kb, seq, 100, block_size=16, forced_first=2, forced_last=3,
                                       return_scores=True)
    for h in range(HKV):
        ref = S.select_topk(sc[0, h].cpu().numpy(), nb, 100, 2, 3, False)
        assert np.array_equal(idx[0, h, :int(n[0, h])].cpu().numpy(), ref)


@pytest.mark.parametrize("score", ["mean", "quest"])
@pytest.mark.parametrize("qdt,kdt", [("bf16", "bf16"), ("f32", "f32"), ("bf16", "f32")])
@pytest.mark.parametrize("g,d", [(1, 128), (2, 64), (4, 128), (8, 128), (8, 64)])
def test_bits_of_the_one_launch_selector(g, d, qdt, kdt, score, device):
    """The same 900 blocks through a 900-block table (one launch) and a 1500-block one
    (two launches), with aligned and unaligned query rows."""
    announce(f"long selection bits g{g} d{d} {qdt} {kdt} {score}")
    dt = {"bf16": torch.bfloat16, "f32": torch.float32}
    gen = torch.Generator(device=device)
    gen.manual_seed(g * d)
    hkv, lens = 3, [900 * 32, 411 * 32 - 5, 0]
    keys = [torch.randn((3, hkv, 1500, d), device=device, generator=gen).to(dt[kdt]) for _ in range(2)]
    keys = [torch.maximum(*keys), torch.minimum(*keys)]
    q = torch.randn((3, hkv * g, d), device=device, generator=gen).to(dt[qdt])
    odd = torch.empty((3, hkv * g, d + 3), device=device, dtype=dt[qdt])[:, :, 1:d + 1]
    odd.copy_(q)
    seq = torch.tensor(lens, device=device, dtype=torch.int32)
    kw = dict(block_size=32, forced_first=1, forced_last=2, score=score, return_scores=True)
    short, long = [tuple(k[:, :, :n].contiguous() for k in keys) for n in (900, 1500)]
    pick = (lambda k: k) if score == "quest" else (lambda k: k[0])
    ref = ia.select_blocks_topk(q, pick(short), seq, 50, **kw)
    for qq in (q, odd):
        got = ia.select_blocks_topk(qq, pick(long), seq, 50, **kw)
        assert torch.equal(ref[1], got[1])
        assert torch.equal(ref[2], got[2][:, :, :900]) and bool(torch.isinf(got[2][:, :, 900:]).all())
        for b in range(3):
            for h in range(hkv):
                m = int(ref[1][b, h])
                assert torch.equal(ref[0][b, h, :m], got[0][b, h, :m])

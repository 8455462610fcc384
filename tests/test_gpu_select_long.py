"""Top-k selection from tables of more than 1024 blocks (scored by a launch over the whole
device, selected from the stored scores): the oracle's rule exactly on the kernel's own
scores at the edges of the keys held per thread, and the bits of the one-launch selector
for every key type, group size and query layout; short rows of wide tables (the same
bits, and no work past a row's own blocks); both sides of the line between one launch and
two."""

import numpy as np
import pytest
import torch

import interattn_amd as ia
from interattn_amd import _native as N
from interattn_amd import ops
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


def _one_launch(q, kb, seq, k, block, ff, fl):
    """The C call without a workspace: one launch, tables of up to 8192 blocks."""
    keys, (b, hkv, nb_max, _), _, keep = ops._block_keys(kb, "mean")
    cap = k + ff + fl
    idx = torch.empty((b, hkv, cap), device=q.device, dtype=torch.int32)
    n_sel = torch.empty((b, hkv), device=q.device, dtype=torch.int32)
    N.check(N.lib().ia_select_topk(ops._decode_shape(q, hkv), q.data_ptr(), keys, seq.data_ptr(), block, nb_max, k,
                                   None, ff, fl, 0, idx.data_ptr(), cap, n_sel.data_ptr(), None, None, 0,
                                   ops._stream(q)))
    del keep
    return idx, n_sel


def _poisoned(b, hkv, nb_max, device):
    """A workspace whose score rows hold NaNs: (dict, the rows as int32 bits)."""
    n = N.lib().ia_select_topk_workspace_size(b, hkv, nb_max)
    buf = torch.full((n,), 0xff, device=device, dtype=torch.uint8)
    return {"topk_scratch": buf}, buf.view(torch.int32).view(b, hkv, nb_max)


def _same(a, b):
    """Equal counts and equal chosen blocks (entries past a row's count are not written)."""
    live = torch.arange(a[0].shape[-1], device=a[0].device) < a[1][..., None]
    return torch.equal(a[1], b[1]) and torch.equal(a[0][live], b[0][live])


@pytest.mark.parametrize("nb_max", [1025, 1500, 8192, 8193, 20000, 40000])
def test_short_rows_of_a_wide_table(nb_max, device):
    """Rows of every number of keys per thread in one table, with a workspace of NaNs: the
    narrow tables' selection, and no score stored past a row's own blocks."""
    announce(f"wide table {nb_max}")
    gen = torch.Generator(device=device)
    gen.manual_seed(nb_max)
    nbs = [min(n, nb_max) for n in (0, 1, 5, 127, 1024, 1025, 4097, 8200, 16385, 32769, nb_max)]
    b, block = len(nbs), 16
    kb = torch.randn((b, HKV, nb_max, D), device=device, generator=gen).bfloat16()
    q = torch.randn((b, 4 * HKV, D), device=device, generator=gen).bfloat16()
    seq = torch.tensor([max(n * block - 3, 0) for n in nbs], device=device, dtype=torch.int32)
    kw = dict(block_size=block, forced_first=1, forced_last=2)
    ws, rows = _poisoned(b, HKV, nb_max, device)
    got = ia.select_blocks_topk(q, kb, seq, 40, workspace=ws, **kw)
    for i, n in enumerate(nbs):
        assert bool((rows[i, :, n:] == -1).all()), (i, n)
        if n:  # the same row through a table of its own width
            own = ia.select_blocks_topk(q[i:i + 1], kb[i:i + 1, :, :n].contiguous(), seq[i:i + 1], 40, **kw)
            assert _same(own, (got[0][i:i + 1], got[1][i:i + 1])), (i, n)
        else:
            assert int(got[1][i].max()) == 0
    if nb_max <= 8192:
        assert _same(_one_launch(q, kb, seq, 40, block, 1, 2), got)


# rows below, at and past the CUs; tables on both sides of the line
@pytest.mark.parametrize("b,hkv,nb_max", [(1, 8, 1024), (1, 8, 1025), (16, 2, 1030), (32, 4, 4096), (32, 4, 4097),
                                          (32, 8, 8192), (32, 8, 8193), (64, 8, 1025), (64, 8, 4096), (64, 8, 4097)])
def test_line_between_one_launch_and_two(b, hkv, nb_max, device):
    announce(f"selection line: {b} x {hkv} rows, {nb_max} blocks")
    gen = torch.Generator(device=device)
    gen.manual_seed(b + nb_max)
    block = 32
    kb = torch.randn((b, hkv, nb_max, D), device=device, generator=gen, dtype=torch.bfloat16)
    q = torch.randn((b, hkv, D), device=device, generator=gen, dtype=torch.bfloat16)
    nbs = torch.randint(0, nb_max + 1, (b,), device=device, generator=gen)
    nbs[0] = nb_max
    seq = (nbs * block).to(torch.int32)
    ws, rows = _poisoned(b, hkv, nb_max, device)
    got = ia.select_blocks_topk(q, kb, seq, 30, block_size=block, forced_first=2, forced_last=1, workspace=ws)
    cus = torch.cuda.get_device_properties(device).multi_processor_count
    n = b * hkv
    two = nb_max > 8192 or (1024 < nb_max <= 4096 if n >= 2 * cus else nb_max > max(1024, 8192 * n // cus))
    assert bool((rows[0, 0] != -1).any()) == two
    full = ia.select_blocks_topk(q, kb, seq, 30, block_size=block, forced_first=2, forced_last=1, return_scores=True)
    assert _same(full, got)
    live = torch.arange(nb_max, device=device)[None, None] < nbs[:, None, None]
    assert torch.equal(torch.isfinite(full[2]), live.expand_as(full[2])) and bool((full[2][~live.expand_as(full[2])] < 0).all())
    if nb_max <= 8192:
        assert _same(_one_launch(q, kb, seq, 30, block, 2, 1), got)
    else:
        for i in (0, 5, b - 1):
            m = int(nbs[i])
            sel = S.select_topk(full[2][i, 0].cpu().numpy(), m, 30, 2, 1, False)
            assert np.array_equal(got[0][i, 0, :int(got[1][i, 0])].cpu().numpy(), sel)


def test_captured_call_follows_the_lengths(device):
    """A captured selection from a wide table, replayed while its rows grow, shrink and empty."""
    announce("wide table: captured call")
    gen = torch.Generator(device=device)
    gen.manual_seed(3)
    b, nb_max, block = 2, 5000, 16
    kb = torch.randn((b, HKV, nb_max, D), device=device, generator=gen).bfloat16()
    q = torch.randn((b, 4 * HKV, D), device=device, generator=gen).bfloat16()
    seq = torch.zeros((b,), device=device, dtype=torch.int32)
    kw = dict(block_size=block, forced_first=1, forced_last=2)
    ws = {}
    ia.select_blocks_topk(q, kb, seq, 40, workspace=ws, **kw)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        got = ia.select_blocks_topk(q, kb, seq, 40, workspace=ws, **kw)
    for lens in ((300, 80000), (80000, 17000), (0, 16), (65537, 16385)):
        seq.copy_(torch.tensor(lens, dtype=torch.int32))
        graph.replay()
        torch.cuda.synchronize()
        assert _same(ia.select_blocks_topk(q, kb, seq, 40, **kw), got), lens

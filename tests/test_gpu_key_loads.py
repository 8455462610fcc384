"""The one-launch top-k call on both sides of the line between whole-row and operand-layout
key loads: uniform k and per-sequence k choose the same blocks through the two instances
(short, ragged and partial subtiles), and both equal the two-step path bit for bit; the line
counts the blocks a row can choose, not the capacity of its index row."""

import math

import pytest
import torch

import interattn_amd as ia
from oracle.cases import make_case
from tests._util import announce, to_dev

pytestmark = pytest.mark.gpu

# query heads of 8 kv heads, page, block, lengths of 4 sequences
CASES = [(32, 16, 64, [1000, 64, 3333, 1]), (64, 32, 128, [300, 4133, 129, 17]), (8, 64, 64, [1250, 4096, 63, 65]),
         (16, 16, 64, [999, 33, 5000, 16])]
IDS = ["g4", "g8", "g1", "g2"]


def _setup(hq, page, block, lens, device):
    case = make_case(seed=7 + hq, batch=4, hq=hq, hkv=8, d=128, seq_lens=lens, page_size=page)
    dev = to_dev(case, device)
    nb_max = max(math.ceil(n / block) for n in lens)
    pool = (dev["pool_k"], dev["pool_v"], dev["block_table"], dev["seq_lens"])
    summ = ia.build_block_summaries(*pool, block, nb_max=nb_max, full=True)
    return dev["q"], pool, {"quest": (summ["k_max"], summ["k_min"]), "mean": summ["k_bar"]}, nb_max


@pytest.mark.parametrize("score", ["quest", "mean"])
@pytest.mark.parametrize("k", [8, 45])
@pytest.mark.parametrize("hq,page,block,lens", CASES, ids=IDS)
def test_both_key_loads_equal_two_step(hq, page, block, lens, k, score, device):
    announce(f"key loads: {hq} query heads, k {k}, {score}")
    q, pool, keys, nb_max = _setup(hq, page, block, lens, device)
    kw = dict(block_size=block, forced_first=1, forced_last=1, score=score)
    idx, n_sel = ia.select_blocks_topk(q, keys[score], pool[3], k, **kw)
    ref = ia.sparse_paged_decode(q, *pool, idx, n_sel, block_size=block)
    # 32 rows of 10 chosen blocks (operand-layout loads), of 33 to 47 (Quest: whole rows), and
    # with a k for each sequence (whole rows)
    per_seq = dict(kw, k_cap=k + 2, k_per_seq=torch.full((4,), k, device=device, dtype=torch.int32))
    for args in (kw, dict(kw, k_cap=512), per_seq):
        ws = {}
        for _ in range(2):
            assert torch.equal(ia.sparse_topk_decode(q, *pool, keys[score], k, workspace=ws, **args), ref)


@pytest.mark.parametrize("k,k_cap,in_k,whole", [(8, None, False, False), (8, 100, False, False),
                                                (8, 100, True, False), (45, None, False, True),
                                                (45, 512, True, True), (500, 20, False, False)])
def test_line_counts_the_blocks_a_row_can_choose(k, k_cap, in_k, whole, device):
    """Which instance runs, by its name: 32 rows of n 64-token blocks are 128 n subtiles, the
    line at 2.5 for each of 8 waves per CU."""
    announce(f"key loads line: k {k}, cap {k_cap}, in_k {in_k}")
    cus = torch.cuda.get_device_properties(device).multi_processor_count
    if not 2 * 128 * 10 < 5 * 8 * cus <= 2 * 128 * 45:
        pytest.skip("the sizes sit on both sides of the line of 256 CUs")
    q, pool, keys, _ = _setup(*CASES[0], device)
    kw = dict(block_size=64, forced_first=1, forced_last=1, forced_in_k=in_k, k_cap=k_cap, score="quest", workspace={})
    ia.sparse_topk_decode(q, *pool, keys["quest"], k, **kw)
    torch.cuda.synchronize()
    prof = torch.profiler.profile(activities=[torch.profiler.ProfilerActivity.CPU,
                                              torch.profiler.ProfilerActivity.CUDA])
    try:
        prof.start()
    except RuntimeError as e:
        pytest.skip(f"no profiler here: {e}")
    ia.sparse_topk_decode(q, *pool, keys["quest"], k, **kw)
    torch.cuda.synchronize()
    prof.stop()
    names = [e.key for e in prof.key_averages() if "paged_finalize" in e.key]
    if not names:
        pytest.skip("the profiler recorded no kernels")
    assert len(names) == 1 and ("true>" in names[0]) == whole, names

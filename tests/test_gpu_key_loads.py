"""The one-launch Quest call on both sides of the line between whole-row and
operand-layout key loads: a cap on the chosen blocks that puts the launch over it gives
the operand-layout instance short, ragged and partial subtiles too."""

import math

import pytest
import torch

import interattn_amd as ia
from oracle.cases import make_case
from tests._util import announce, to_dev

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("k_cap", [10, 100, 512], ids=["few", "rows", "operand"])
@pytest.mark.parametrize("hq,page,block,lens", [(32, 16, 64, [1000, 64, 3333, 1]), (64, 32, 128, [300, 4133, 129, 17]),
                                                (8, 64, 64, [1250, 4096, 63, 65]), (16, 16, 64, [999, 33, 5000, 16])],
                         ids=["g4", "g8", "g1", "g2"])
def test_both_key_loads_equal_two_step(hq, page, block, lens, k_cap, device):
    announce(f"key loads: {hq} query heads, cap {k_cap}")
    case = make_case(seed=7 + hq, batch=4, hq=hq, hkv=8, d=128, seq_lens=lens, page_size=page)
    dev = to_dev(case, device)
    # 4 x 8 rows of blocks of 64 or 128 tokens x 512 bytes of K and V: a cap of 10 is 10 to 20
    # MB (operand loads), 100 is 105 to 210 MB (whole rows), 512 above 512 MB (operand loads)
    nb_max = max(math.ceil(n / block) for n in lens)
    pool = (dev["pool_k"], dev["pool_v"], dev["block_table"], dev["seq_lens"])
    summ = ia.build_block_summaries(*pool, block, nb_max=nb_max, full=True)
    keys = (summ["k_max"], summ["k_min"])
    kw = dict(block_size=block, forced_first=1, forced_last=1, k_cap=k_cap, score="quest")
    idx, n_sel = ia.select_blocks_topk(dev["q"], keys, dev["seq_lens"], 8, **kw)
    ref = ia.sparse_paged_decode(dev["q"], *pool, idx, n_sel, block_size=block)
    ws = {}
    for _ in range(2):
        assert torch.equal(ia.sparse_topk_decode(dev["q"], *pool, keys, 8, workspace=ws, **kw), ref)

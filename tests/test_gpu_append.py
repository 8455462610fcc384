"""KV append, one workgroup per sequence: rows of every head at the sizes where the copy
takes part of a pass, one pass or several; unmapped and out-of-table positions untouched."""

import pytest
import torch

import interattn_amd as ia
from tests._util import announce

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float32], ids=["bf16", "f32"])
@pytest.mark.parametrize("hkv,d,page", [(1, 64, 16), (8, 128, 16), (7, 128, 32), (40, 128, 16)])
def test_append_rows_and_lengths(hkv, d, page, dt, device):
    announce(f"append hkv {hkv} d {d} {dt}")
    gen = torch.Generator(device=device)
    gen.manual_seed(hkv)
    lens = [0, page - 1, page, 3 * page, 2 * page + 5, 4 * page, -1]  # the last three: unmapped, past the table, none
    b, n_pages = len(lens), 4 * len(lens)
    pk, pv = (torch.randn((n_pages, hkv, page, d), device=device, generator=gen).to(dt) for _ in range(2))
    table = torch.randperm(n_pages, device=device, generator=gen).to(torch.int32).view(b, 4)
    table[4, 2] = -1
    new = torch.randn((2, b, hkv, d), device=device, generator=gen).to(dt)
    ref_k, ref_v, want = pk.clone(), pv.clone(), list(lens)
    for i in range(4):
        at = int(table[i, lens[i] // page])
        ref_k[at, :, lens[i] % page], ref_v[at, :, lens[i] % page] = new[0, i], new[1, i]
        want[i] += 1
    seq = torch.tensor(lens, device=device, dtype=torch.int32)
    ia.append_kv(pk, pv, table, seq, new[0], new[1])
    assert seq.tolist() == want
    assert torch.equal(pk, ref_k) and torch.equal(pv, ref_v)

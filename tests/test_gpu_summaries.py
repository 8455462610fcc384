"""Block summaries where the launch gives a wave several blocks, pages are missing or
outputs are not 16-byte aligned: each equals the same blocks summarised one per wave, or
into aligned arrays, bit for bit (a block's sums run in one order whatever wave takes it)."""

import pytest
import torch

import interattn_amd as ia
from tests._util import announce

pytestmark = pytest.mark.gpu

# dtype, block, lengths (one full, one ending inside a subtile of its last block)
CASES = [("bf16", 16, [26000, 25011]), ("bf16", 48, [40000, 39023]), ("f32", 16, [13000, 12345]),
         ("fp8", 64, [50000, 49999]), ("bf16", 1040, [9000, 1041])]


def _pool(dt, lens, device, hkv=8, d=64, page=16):
    gen = torch.Generator(device=device)
    gen.manual_seed(len(dt) + lens[1])
    need = [-(-n // page) for n in lens]
    n_pages = sum(need)
    shape = (n_pages, hkv, page, d)
    k, v = (torch.empty(shape, device=device, dtype=torch.float32).normal_(generator=gen) for _ in range(2))
    scales = None
    if dt == "fp8":
        scales = tuple(x.abs().amax(dim=(2, 3)) / 448.0 for x in (k, v))
        k, v = ((x / s[:, :, None, None]).to(torch.float8_e4m3fn) for x, s in zip((k, v), scales))
    elif dt == "bf16":
        k, v = k.bfloat16(), v.bfloat16()
    perm = torch.randperm(n_pages, device=device, generator=gen).to(torch.int32)
    table = torch.full((len(lens), max(need)), -1, device=device, dtype=torch.int32)
    table[0, :need[0]] = perm[:need[0]]
    table[1, :need[1]] = perm[need[0]:]
    table[0, 5], table[1, 7] = -1, n_pages  # unmapped pages count no tokens
    return k, v, scales, table


@pytest.mark.parametrize("full", [True, False], ids=["full", "keys"])
@pytest.mark.parametrize("c", CASES, ids=[f"{c[0]}_b{c[1]}" for c in CASES])
def test_wave_split_does_not_change_bits(c, full, device):
    dt, block, lens = c
    announce(f"summaries {dt} block {block} full {full}")
    k, v, scales, table = _pool(dt, lens, device)
    seq = torch.tensor(lens, device=device, dtype=torch.int32)
    nb_max = max(-(-n // block) for n in lens) + 1
    kw = dict(nb_max=nb_max, full=full, k_bar_dtype=torch.float32, v_bar_dtype=torch.float32)
    got = ia.build_block_summaries(k, v, table, seq, block, scales=scales, **kw)
    for b in range(2):
        for h in range(8):
            sc = None if scales is None else tuple(s[:, h:h + 1].contiguous() for s in scales)
            one = ia.build_block_summaries(k[:, h:h + 1], v[:, h:h + 1], table[b:b + 1], seq[b:b + 1], block,
                                           scales=sc, **kw)
            for key, x in one.items():
                y = got[key][b] if key == "block_valid_counts" else got[key][b, h]
                assert torch.equal(x.reshape(y.shape), y), (key, b, h)


def test_unaligned_outputs(device):
    announce("summaries into unaligned arrays")
    k, v, _, table = _pool("bf16", [1000, 333], device)
    old, new = (torch.tensor(x, device=device, dtype=torch.int32) for x in ([990, 320], [1000, 333]))
    ref = ia.build_block_summaries(k, v, table, new, 32, nb_max=33, full=True)
    got = ia.build_block_summaries(k, v, table, old, 32, nb_max=33, full=True)
    for key in ("k_bar", "v_bar", "k_max", "k_min"):
        flat = torch.empty(got[key].numel() + 1, device=device, dtype=got[key].dtype)
        flat[1:] = got[key].flatten()
        got[key] = flat[1:].view(got[key].shape)
    ia.update_block_summaries(got, k, v, table, old, new, 32, max_new_tokens=16)
    for key, x in ref.items():
        assert torch.equal(x, got[key]), key

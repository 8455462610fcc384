"""The one-launch eps-rule and fixed-mask calls with GQA groups of 8: against the
multi-launch path on the same inputs (selection equal away from eps, outputs within the
rounding of two orders of the same sums), at the edges of an item's blocks; the hand-off
fallback bit for bit; what does not fit stays on the multi-launch path."""

import numpy as np
import pytest
import torch

from interattn_amd import _native as N
from interattn_amd import condition_block as cb
from tests._util import announce

pytestmark = pytest.mark.gpu

# kv heads, head_dim, block, prompt, suffix, dtype, mixed summaries, k_bar dtype.  Prompts:
# one block; one item; items of 31-33 blocks; a ragged last block; more than one statistics step
CASES = [(8, 128, 64, 40, 1, "bf16", True, "bf16"), (2, 128, 16, 16 * 33, 5, "bf16", False, "f32"),
         (8, 128, 64, 20011, 100, "bf16", False, "f32"), (8, 128, 32, 32 * 1025, 0, "bf16", True, "bf16"),
         (1, 128, 16, 70001, 300, "bf16", True, "f32"), (4, 64, 64, 9000, 17, "f32", False, "f32"),
         (2, 64, 32, 5000, 3, "bf16", True, "bf16")]


def _inputs(c, device):
    hkv, d, block, p, s, dt, mixed, kbd = c
    gen = torch.Generator(device=device)
    gen.manual_seed(p + s)
    t = torch.bfloat16 if dt == "bf16" else torch.float32
    rnd = lambda *shape: torch.randn(shape, device=device, generator=gen)  # noqa: E731
    k = rnd(hkv, p, d) + 0.5 * rnd(hkv, 1, d)
    k[:, torch.randint(0, p, (max(1, p // 500),), device=device, generator=gen)] *= 4.0
    x = dict(k=k.to(t), v=rnd(hkv, p, d).to(t), q=rnd(hkv, 8, 1, d).to(t), ks=rnd(hkv, s, d).to(t),
             vs=rnd(hkv, s, d).to(t), len=torch.full((1,), s, device=device, dtype=torch.int32))
    x["prefix"] = cb._build_prompt_blocks(x["k"], x["v"], block, mixed=mixed,
                                          k_bar_dtype=torch.bfloat16 if kbd == "bf16" else torch.float32)
    return x


def _call(x, block, p, eps, ws):
    out = cb._condition_block_decode_output(
        q_grouped=x["q"], prompt_prefix=x["prefix"], k_suffix=x["ks"], v_suffix=x["vs"], suffix_len_dev=x["len"],
        block_size=block, eps=eps, prompt_len=p, attention_dtype=torch.float32, workspace=ws, collect_stats=True)[0]
    return out.clone(), ws["selected_rows"].clone()


def _fused(ws):
    return any(isinstance(k, tuple) and k[0] == "condition_fused_scratch" for k in ws)


def _eps(x):
    """An eps in the widest gap of the conditions' upper half (so both orders of the sums
    select the same blocks), from the standalone selection by bisection."""
    lo, hi = -9.0, 3.0
    nb = x["prefix"]["block_valid_counts"].numel()
    for _ in range(30):
        mid = 0.5 * (lo + hi)
        share = float(cb._select_prompt_blocks_triton(x["q"], x["prefix"], 10.0 ** mid)[0].float().mean())
        if share > (0.05 if nb > 40 else 0.5):
            lo = mid
        else:
            hi = mid
    return 10.0 ** hi


@pytest.mark.parametrize("c", CASES, ids=[f"h{c[0]}d{c[1]}b{c[2]}p{c[3]}_{c[5]}" for c in CASES])
def test_one_launch_equals_multi_launch(c, device, monkeypatch):
    hkv, d, block, p, s, dt, mixed, kbd = c
    announce(f"group of 8: {c}")
    x = _inputs(c, device)
    tol = 2e-2 if dt == "bf16" else 1e-4
    for eps in (0.0, _eps(x), 1e30):
        got = {}
        for one in ("1", "0"):
            monkeypatch.setenv("INTERATTN_CONDITION_ONE_LAUNCH", one)
            ws = {}
            got[one] = _call(x, block, p, eps, ws)
            assert _fused(ws) == (one == "1")
        differ = int((got["1"][1] != got["0"][1]).sum())
        assert differ == 0 or (0.0 < eps < 1e30 and differ <= 8), (eps, differ)  # one block at eps: its 8 rows
        if differ == 0:
            np.testing.assert_allclose(got["1"][0].cpu().numpy(), got["0"][0].cpu().numpy(), atol=tol, rtol=0)
    mask = torch.zeros((hkv, x["prefix"]["block_valid_counts"].numel()), device=device, dtype=torch.bool)
    mask[:, ::5] = True
    out = []
    for one in ("1", "0"):
        monkeypatch.setenv("INTERATTN_CONDITION_ONE_LAUNCH", one)
        out.append(cb.fixed_mask_hybrid_attention(
            q_grouped=x["q"], prompt_prefix=x["prefix"], selected=mask, k_suffix=x["ks"], v_suffix=x["vs"],
            block_size=block, output_dtype=torch.float32, workspace={}).cpu().numpy())
    np.testing.assert_allclose(out[0], out[1], atol=tol, rtol=0)


def test_handoff_fallback_and_replays_are_exact(device, monkeypatch):
    monkeypatch.setenv("INTERATTN_CONDITION_ONE_LAUNCH", "1")
    c = CASES[2]
    announce("group of 8: hand-off fallback, repeated calls on one workspace")
    x = _inputs(c, device)
    eps, ws = _eps(x), {}
    ref = _call(x, c[2], c[3], eps, ws)
    prev = N.lib().ia_set_wait_limit(0)  # every item computes every partial itself
    try:
        alone = _call(x, c[2], c[3], eps, {})
    finally:
        N.lib().ia_set_wait_limit(prev)
    for got in (alone, _call(x, c[2], c[3], eps, ws), _call(x, c[2], c[3], eps, ws)):
        assert torch.equal(ref[0], got[0]) and torch.equal(ref[1], got[1])


def test_fp32_head_dim_128_keeps_the_multi_launch_path(device, monkeypatch):
    monkeypatch.setenv("INTERATTN_CONDITION_ONE_LAUNCH", "1")
    announce("group of 8: fp32 caches at head_dim 128")
    x = _inputs((1, 128, 64, 3000, 5, "f32", False, "f32"), device)
    ws = {}
    _call(x, 64, 3000, 0.01, ws)
    assert not _fused(ws)

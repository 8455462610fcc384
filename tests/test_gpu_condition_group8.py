"""The one-launch eps-rule and fixed-mask calls with GQA groups of 8: against the
multi-launch path on the same inputs (the same selection, eps in a gap of the conditions;
outputs within the rounding of two splits of the same sums, in proportion to the outputs),
at the edges of an item's blocks; the hand-off fallback bit for bit; what does not fit stays
on the multi-launch path; the entry points for groups of up to 4 equal this one and refuse
groups of 8."""

import numpy as np
import pytest
import torch

from interattn_amd import _native as N
from interattn_amd import condition_block as cb
from tests._util import announce
from tests.test_gpu_condition import _np, _oracle_stats, _prefix_np

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
    """An eps that selects about 5% of the blocks (half of a few), in the middle of the
    widest relative gap there between the conditions' 64-bit values.  Float32 logits of up to
    ~20 leave a condition ~1e-5 of relative rounding, so either order of the row's sums
    selects the same blocks."""
    q = _np(x["q"].float())[:, :, 0]
    mean = _oracle_stats(q.reshape(-1, q.shape[-1]), _prefix_np(x["prefix"]), 8, False)[1]
    v = np.sort(mean[mean > 0])[::-1]
    n = (0.05 if x["prefix"]["block_valid_counts"].numel() > 40 else 0.5) * len(v)
    lo = max(int(0.5 * n), 1)
    hi = min(max(int(1.5 * n), lo + 1), len(v) - 1)
    i = lo + int(np.argmax(v[lo - 1:hi - 1] / v[lo:hi])) if hi > lo else lo
    assert v[i - 1] / v[i] > 1.0002, "no gap wide enough"
    return float(np.sqrt(v[i - 1] * v[i]))


def _check(got, ref, dt):
    """Two splits of the same sums.  bf16 caches: every softmax weight is rounded to bf16
    against its item's own maximum, a relative error of at most 2^-9 and ~0.42 x 2^-9 rms, so
    independent roundings on both sides leave ~0.42 sqrt(2) 2^-9 = 1.2e-3 of the output's
    2-norm whatever cancels in the sum; float32 caches keep float32 sums (a few 1e-7).  Bounds:
    ~3.5 of those rms, and 4 times that on single values (13 sigma).  An item's partial that is
    lost or counted twice moves the output by ~1 / sqrt(items) > 0.1."""
    got, ref = _np(got).astype(np.float64), _np(ref).astype(np.float64)
    rel = np.linalg.norm(got - ref) / np.linalg.norm(ref)
    rms = np.sqrt(np.mean(ref ** 2))
    bound = 2.0 ** -8 if dt == "bf16" else 2e-6
    assert rel <= bound, (rel, bound)
    assert np.abs(got - ref).max() <= 4 * bound * rms, (np.abs(got - ref).max() / rms, bound)


@pytest.mark.parametrize("c", CASES, ids=[f"h{c[0]}d{c[1]}b{c[2]}p{c[3]}_{c[5]}" for c in CASES])
def test_one_launch_equals_multi_launch(c, device, monkeypatch):
    hkv, d, block, p, s, dt, mixed, kbd = c
    announce(f"group of 8: {c}")
    x = _inputs(c, device)
    for eps in (0.0, _eps(x), 1e30):
        got = {}
        for one in ("1", "0"):
            monkeypatch.setenv("INTERATTN_CONDITION_ONE_LAUNCH", one)
            ws = {}
            got[one] = _call(x, block, p, eps, ws)
            assert _fused(ws) == (one == "1")
        assert torch.equal(got["1"][1], got["0"][1]), eps
        assert bool(got["0"][1].any()) == (eps < 1e30)
        _check(got["1"][0], got["0"][0], dt)
    mask = torch.zeros((hkv, x["prefix"]["block_valid_counts"].numel()), device=device, dtype=torch.bool)
    mask[:, ::5] = True
    out = []
    for one in ("1", "0"):
        monkeypatch.setenv("INTERATTN_CONDITION_ONE_LAUNCH", one)
        out.append(cb.fixed_mask_hybrid_attention(
            q_grouped=x["q"], prompt_prefix=x["prefix"], selected=mask, k_suffix=x["ks"], v_suffix=x["vs"],
            block_size=block, output_dtype=torch.float32, workspace={}))
    _check(out[0], out[1], dt)


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


@pytest.mark.parametrize("group", [1, 2, 4, 8])
def test_entry_points_for_groups_of_up_to_four(group, device):
    """``ia_condition_decode_fused`` and ``ia_fixed_mask_decode_fused`` through the C ABI: the
    bits of ``ia_condition_one_launch`` for groups of up to 4, a refusal for groups of 8."""
    announce(f"one-launch entry points, group of {group}")
    hkv, d, block, p, s = 2, 128, 64, 5000, 9
    x = _inputs((hkv, d, block, p, s, "bf16", True, "bf16"), device)
    q, sh = cb._grouped_shape(x["q"][:, :group].contiguous())
    sm, keep, nb = cb._summaries_desc(x["prefix"], hkv, d)
    kv = cb._kv_desc(x["prefix"]["k_block_attn"], x["prefix"]["v_block_attn"], block)
    sfx, keep_s = cb._suffix_desc(x["ks"], x["vs"], x["len"], torch.bfloat16)
    lib = N.lib()
    n = lib.ia_condition_decode_fused_workspace_size(1, hkv, group, d)
    stream = torch.cuda.current_stream().cuda_stream
    mask = torch.zeros((hkv, nb), device=device, dtype=torch.uint8)
    mask[:, ::7] = 1
    eps, scale = 0.02, d ** -0.5

    def run(call):
        out = torch.empty((hkv * group, d), device=device, dtype=torch.float32)
        sel = torch.zeros((hkv * group, nb), device=device, dtype=torch.uint8)
        ws = torch.zeros((n,), device=device, dtype=torch.uint8)
        rc = call(out.data_ptr(), sel.data_ptr(), ws.data_ptr())
        torch.cuda.synchronize()
        return rc, out, sel

    new = [run(lambda o, sl, w, m=m: lib.ia_condition_one_launch(
        sh, q.data_ptr(), sm, m, kv, sfx, eps, 0, sl, scale, o, N.IA_F32, w, n, stream)) for m in (None, mask.data_ptr())]
    old = [run(lambda o, sl, w: lib.ia_condition_decode_fused(sh, q.data_ptr(), sm, kv, sfx, eps, 0, sl, scale, o,
                                                              N.IA_F32, w, n, stream)),
           run(lambda o, sl, w: lib.ia_fixed_mask_decode_fused(sh, q.data_ptr(), sm, mask.data_ptr(), kv, sfx, scale, o,
                                                               N.IA_F32, w, n, stream))]
    assert lib.ia_condition_one_launch_items(sh, sm, N.IA_BF16, sfx.cap) > 0 and all(r[0] == N.IA_OK for r in new)
    assert (lib.ia_condition_decode_fused_items(sh, sm, N.IA_BF16, sfx.cap) > 0) == (group <= 4)
    for a, b in zip(old, new):
        if group > 4:
            assert a[0] == N.IA_ERR_UNSUPPORTED
        else:
            assert a[0] == N.IA_OK and torch.equal(a[1], b[1]) and torch.equal(a[2], b[2])
    assert bool(new[0][2].any()) and not bool(new[1][2].any())  # (a mask's call writes no selection)
    del keep, keep_s

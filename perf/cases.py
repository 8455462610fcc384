"""Workloads of the decode-attention library, as a serving program runs them.

A case is one call (or one decode step) through the package's public entry points.
Kinds:

  topk       ``ia.sparse_topk_decode``: one top-k layer call over a paged K/V pool
             (block scores, selection, attention over the chosen blocks)
  dense      ``ia.paged_decode``: the dense paged fallback
  summaries  ``ia.build_block_summaries``: the block summaries of freshly prefilled
             sequences
  serve      one serving decode step of one layer: new lengths, ``ia.append_kv``,
             ``ia.update_block_summaries``, ``ia.sparse_topk_decode``
  cond       ``condition_block._condition_block_decode_output``: the reference's
             eps-rule layer call over a prompt and its exact suffix (batch 1)
  fixed      ``condition_block.fixed_mask_hybrid_attention``: the same with a caller's
             block mask

Values are those the path meets: unit-variance queries and values, keys with a scale
per (kv head, channel) as rotary keys have; pages in random order; fp8 pages scaled by
their largest magnitude.
"""

import math
import random

import torch

import interattn_amd as ia
from interattn_amd import condition_block as cb

DTYPES = {"bf16": torch.bfloat16, "f32": torch.float32, "fp8": torch.float8_e4m3fn}
BYTES = {"bf16": 2, "f32": 4, "fp8": 1}
DEV = "cuda"


# ------------------------------------------------------------------ the cases

def listed():
    llama = {"hq": 32, "hkv": 8, "d": 128, "page": 16}
    return [
        # single-user decode at 32K: latency, one layer of a Llama-geometry model
        dict(llama, name="topk 1x32k", kind="topk", batch=1, lo=32768, hi=32768, block=64, k=64, ff=1, fl=2,
             kv="bf16", score="mean", per_seq_k=False, layout="split", len_seed=0),
        # a ragged batch, k in proportion to each length
        dict(llama, name="topk 16x8k-64k", kind="topk", batch=16, lo=8192, hi=65536, block=64, k=16, ff=0, fl=0,
             kv="bf16", score="mean", per_seq_k=True, layout="paired", len_seed=1236),
        # long-context batch, bf16: the headline layer call
        dict(llama, name="topk 16x128k", kind="topk", batch=16, lo=131072, hi=131072, block=128, k=64, ff=0, fl=0,
             kv="bf16", score="mean", per_seq_k=False, layout="paired", len_seed=0),
        # the same with quantised pages
        dict(llama, name="topk fp8 16x128k", kind="topk", batch=16, lo=131072, hi=131072, block=128, k=64, ff=0,
             fl=0, kv="fp8", score="mean", per_seq_k=False, layout="paired", len_seed=0),
        # Quest's page bound on small pages, groups of 8 query heads, odd lengths
        dict(name="topk quest g8 4x30k-60k", kind="topk", batch=4, hq=64, hkv=8, d=128, page=32, lo=30011, hi=60013,
             block=32, k=96, ff=1, fl=1, kv="bf16", score="quest", per_seq_k=False, layout="split", len_seed=5),
        # one very long context: more blocks than the one-launch call takes
        dict(llama, name="topk 1x1m", kind="topk", batch=1, lo=1000003, hi=1000003, block=64, k=256, ff=1, fl=4,
             kv="bf16", score="mean", per_seq_k=False, layout="split", len_seed=0),
        # the dense fallback layers of a moderate ragged batch
        dict(llama, name="dense 8x2k-16k", kind="dense", batch=8, lo=2000, hi=16384, kv="bf16", layout="split",
             len_seed=3),
        # summaries of a batch that has just been prefilled
        dict(llama, name="summaries 8x40k-64k", kind="summaries", batch=8, lo=40001, hi=65536, block=64, full=True,
             kv="bf16", layout="split", len_seed=4),
        # a decode step of a chat-length serving batch
        dict(llama, name="serve 32x1k-4k", kind="serve", batch=32, lo=1000, hi=4000, block=32, k=16, ff=1, fl=1,
             kv="bf16", score="mean", layout="split", len_seed=6),
        # the eps rule at 128K, mixed summaries (the reference's production setting)
        dict(name="cond 1x128k", kind="cond", hkv=8, g=4, d=128, block=64, seq=131072, suffix=1, kv="bf16",
             mixed=True, kbar="bf16", frac=0.0095, mass=False),
        # the eps rule with float32 summaries, groups of 8, an odd prompt, a growing suffix
        dict(name="cond g8 1x20k", kind="cond", hkv=8, g=8, d=128, block=64, seq=20011, suffix=100, kv="bf16",
             mixed=False, kbar="f32", frac=0.04, mass=False),
        # a caller's block mask (selection reused from another step), runs of neighbours
        dict(name="fixed 1x64k", kind="fixed", hkv=8, g=4, d=128, block=64, seq=65536, suffix=17, kv="bf16",
             mixed=True, kbar="bf16", frac=0.0155),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["topk", "topk", "topk", "topk", "dense", "summaries", "serve", "cond", "cond", "fixed"])
    g = rng.choice([1, 2, 4, 4, 4, 8])
    hkv = rng.choice([2, 4, 8, 8])
    d = rng.choice([64, 128, 128])
    page = rng.choice([16, 16, 32, 64])
    block = rng.choice([16, 32, 64, 64, 128])
    layout = rng.choice(["split", "paired"])
    len_seed = rng.randrange(1 << 20)
    if kind in ("cond", "fixed"):
        c = dict(kind=kind, hkv=hkv, g=g, d=d, block=block, seq=_log(rng, 3000, 131072), suffix=_log(rng, 1, 600),
                 kv=rng.choice(["bf16", "bf16", "f32"]), mixed=rng.random() < 0.6, kbar="f32",
                 frac=rng.choice([0.01, 0.03, 0.1]))
        if c["mixed"] and rng.random() < 0.7:
            c["kbar"] = "bf16"
        if kind == "cond":
            c["mass"] = rng.random() < 0.2
        return c
    base = dict(kind=kind, hq=g * hkv, hkv=hkv, d=d, page=page, layout=layout, len_seed=len_seed)
    if kind == "topk":
        batch = _log(rng, 1, 16)
        hi = _log(rng, 2500, 131072)
        lo = hi if rng.random() < 0.4 else max(hi // rng.choice([2, 4, 8]), 100)
        kv = rng.choice(["bf16", "bf16", "bf16", "fp8", "f32"])
        if kv == "f32":  # a state of float32 pools stays as small as the bf16 one
            lo, hi = (lo + 1) // 2, (hi + 1) // 2
        return dict(base, batch=batch, lo=lo, hi=hi, block=block, k=_log(rng, 8, 128), ff=rng.choice([0, 1]),
                    fl=rng.choice([0, 1, 2]), kv=kv, score=rng.choice(["mean", "mean", "quest"]),
                    per_seq_k=rng.random() < 0.3)
    if kind == "dense":
        batch = _log(rng, 1, 16)
        hi = _log(rng, 500, 32768)
        return dict(base, batch=batch, lo=max(hi // rng.choice([1, 2, 8]), 1), hi=hi,
                    kv=rng.choice(["bf16", "bf16", "fp8"]))
    if kind == "summaries":
        batch = _log(rng, 1, 8)
        hi = _log(rng, 4000, 65536)
        return dict(base, batch=batch, lo=max(hi // rng.choice([1, 2, 4]), 1), hi=hi, block=block,
                    full=rng.random() < 0.6, kv=rng.choice(["bf16", "bf16", "fp8"]))
    hi = _log(rng, 800, 8000)
    return dict(base, batch=_log(rng, 4, 32), lo=hi // 4, hi=hi, block=block, k=_log(rng, 8, 32), ff=1,
                fl=rng.choice([1, 2]), kv="bf16", score="mean")


# ------------------------------------------------------------------ inputs

def _lens(c):
    r = random.Random(c["len_seed"])
    return [r.randint(c["lo"], c["hi"]) for _ in range(c["batch"])]


def _ks(c):
    """k per sequence: a sixteenth of its blocks where k follows the length, else k."""
    return [max(c["k"], -(-n // c["block"]) // 16) if c["per_seq_k"] else c["k"] for n in _lens(c)]


def _gen(seed):
    g = torch.Generator(device=DEV)
    g.manual_seed(seed)
    return g


def _normal(gen, shape, dtype):
    return torch.empty(shape, device=DEV, dtype=dtype).normal_(generator=gen)


def _pool(c, gen, lens):
    """The paged pool: K and V views [n_pages, Hkv, page, D], scales, block table."""
    hkv, page, d = c["hkv"], c["page"], c["d"]
    need = [-(-n // page) for n in lens]
    n_pages = sum(need) + 8
    outlier = (0.5 * _normal(gen, (hkv, 1, d), torch.float32)).exp()
    if c["layout"] == "paired":
        buf = torch.empty((n_pages, hkv, 2, page, d), device=DEV, dtype=DTYPES[c["kv"]])
        k, v = buf[:, :, 0], buf[:, :, 1]
    else:
        k = torch.empty((n_pages, hkv, page, d), device=DEV, dtype=DTYPES[c["kv"]])
        v = torch.empty_like(k)
    scales = None
    ks, vs = [], []
    step = max(1, (1 << 28) // (hkv * page * d))
    for i in range(0, n_pages, step):
        n = min(step, n_pages - i)
        draw_t = torch.float32 if c["kv"] == "f32" else torch.bfloat16
        for pool, sc, mul in ((k, ks, outlier), (v, vs, None)):
            x = _normal(gen, (n, hkv, page, d), draw_t)
            if mul is not None:
                x.mul_(mul.to(draw_t))
            if c["kv"] == "fp8":
                s = x.abs().amax(dim=(2, 3)).float().clamp_min(1e-12) / 448.0
                sc.append(s)
                x = (x.float() / s[:, :, None, None])
            pool[i:i + n].copy_(x)
    perm = torch.randperm(n_pages, device=DEV, generator=gen).to(torch.int32)
    table = torch.full((len(lens), max(need)), -1, device=DEV, dtype=torch.int32)
    off = 0
    for b, n in enumerate(need):
        table[b, :n] = perm[off:off + n]
        off += n
    if c["kv"] == "fp8":
        scales = (torch.cat(ks).contiguous(), torch.cat(vs).contiguous())
    return k, v, scales, table


def _rows(pool, scale, table_row, n, dtype):
    """[Hkv, n, D]: the first n tokens of one sequence, dequantised, in ``dtype``."""
    page = pool.shape[2]
    pages = table_row[:-(-n // page)].long()
    x = pool[pages].to(torch.float32).to(dtype)
    if scale is not None:
        x = x * scale[pages][:, :, None, None].to(dtype)
    return x.transpose(0, 1).reshape(pool.shape[1], -1, pool.shape[3])[:, :n]


def _blocks(x, block, fill):
    """[Hkv, n, D] -> [Hkv, nb, block, D], the tail filled."""
    n = x.shape[1]
    nb = -(-n // block)
    return torch.nn.functional.pad(x, (0, 0, 0, nb * block - n), value=fill).view(x.shape[0], nb, block, x.shape[2])


def _block_keys(c, pool_k, scales, table, lens):
    """What a top-k program keeps per block: the mean key, or Quest's key extrema."""
    nb_max = max(-(-n // c["block"]) for n in lens)
    dt = torch.float32 if c["kv"] == "f32" else torch.bfloat16
    n_out = 2 if c["score"] == "quest" else 1
    out = [torch.zeros((len(lens), c["hkv"], nb_max, c["d"]), device=DEV, dtype=dt) for _ in range(n_out)]
    for b, n in enumerate(lens):
        x = _rows(pool_k, None if scales is None else scales[0], table[b], n, torch.float32)
        nb = -(-n // c["block"])
        if n_out == 2:
            out[0][b, :, :nb] = _blocks(x, c["block"], -math.inf).amax(2).to(dt)
            out[1][b, :, :nb] = _blocks(x, c["block"], math.inf).amin(2).to(dt)
        else:
            cnt = torch.full((nb, 1), c["block"], device=DEV, dtype=torch.float32)
            cnt[-1] = n - (nb - 1) * c["block"]
            out[0][b, :, :nb] = (_blocks(x, c["block"], 0.0).sum(2) / cnt).to(dt)
    return tuple(out) if n_out == 2 else out[0]


def _q_dtype(c):
    return torch.float32 if c["kv"] == "f32" else torch.bfloat16


def _paged_inputs(c, seed):
    gen = _gen(seed)
    lens = _lens(c)
    s = {"case": c, "lens": lens, "ws": {}}
    grown = [n + 1 for n in lens] if c["kind"] == "serve" else lens
    s["k"], s["v"], s["scales"], s["table"] = _pool(c, gen, grown)
    s["q"] = _normal(gen, (c["batch"], c["hq"], c["d"]), _q_dtype(c))
    s["seq"] = torch.tensor(lens, device=DEV, dtype=torch.int32)
    s["max_len"] = max(lens)
    if c["kind"] == "topk":
        s["keys"] = _block_keys(c, s["k"], s["scales"], s["table"], lens)
        ks = _ks(c)
        s["k_cap"] = max(ks) + c["ff"] + c["fl"]
        s["kvec"] = torch.tensor(ks, device=DEV, dtype=torch.int32) if c["per_seq_k"] else None
    elif c["kind"] == "serve":
        s["k_new"] = _normal(gen, (c["batch"], c["hkv"], c["d"]), DTYPES[c["kv"]])
        s["v_new"] = _normal(gen, (c["batch"], c["hkv"], c["d"]), DTYPES[c["kv"]])
    return s


def _prompt_inputs(c, seed):
    gen = _gen(seed)
    hkv, g, d, p, n = c["hkv"], c["g"], c["d"], c["seq"], c["suffix"]
    dt = DTYPES[c["kv"]]
    # a few heavy keys and a bias per head spread the condition over several decades
    k = _normal(gen, (hkv, p, d), torch.float32)
    heavy = torch.rand((1, p, 1), device=DEV, generator=gen) < 0.002
    k = (torch.where(heavy, 4.0 * k, k) + 0.5 * _normal(gen, (hkv, 1, d), torch.float32)).to(dt)
    s = {"case": c, "k": k, "v": _normal(gen, (hkv, p, d), dt), "q": _normal(gen, (hkv, g, 1, d), dt),
         "ks": _normal(gen, (hkv, n, d), dt), "vs": _normal(gen, (hkv, n, d), dt), "ws": {}}
    s["len"] = torch.full((1,), n, device=DEV, dtype=torch.int32)
    if c["kind"] == "fixed":  # runs of about four neighbouring blocks
        nb = -(-p // c["block"])
        start = torch.rand((hkv, nb), device=DEV, generator=gen) < c["frac"] / 4
        m = start.clone()
        for j in range(1, 4):
            m[:, j:] |= start[:, :nb - j]
        m[:, 0] = True
        s["mask"] = m
    return s


def _condition(q, k_bar, k_max, k_min, counts, v_norm, mass):
    """The eps rule's group-mean condition [Hkv, nb] and the logits z [Hkv, G, nb], in 64 bits."""
    hkv, g, _, d = q.shape
    q = q[:, :, 0].double()
    inv = d ** -0.5
    cnt = counts.double()
    mean, zs = [], []
    for h in range(hkv):
        kb, hi, lo = (x[h].double().t().contiguous() for x in (k_bar, k_max, k_min))
        s = torch.matmul(q[h], kb) * inv
        qp, qn = q[h].clamp_min(0), q[h].clamp_max(0)
        up = (torch.matmul(qp, hi) + torch.matmul(qn, lo)) * inv
        dn = (torch.matmul(qp, lo) + torch.matmul(qn, hi)) * inv
        dl = torch.maximum((up - s).abs(), (dn - s).abs())
        z = s + cnt.log()
        b = v_norm[h].double()
        zl = torch.log_softmax(z, -1)
        if mass:
            t1 = 2 * b.max() * torch.softmax(z + dl, -1)
        else:
            zc = z + dl + torch.log1p(torch.exp(-2 * dl)) - math.log(2.0)
            lc = torch.logsumexp(zc, -1, keepdim=True)
            t1 = 2 * b.max() * (torch.exp(zc - lc) - torch.exp(z - lc))
        mean.append((t1 + 2 * b * torch.exp(zl) * torch.tanh(0.5 * dl)).mean(0))
        zs.append(z)
    return torch.stack(mean), torch.stack(zs)


def _eps_at(mean, frac):
    """An eps between two condition values that selects about ``frac`` of the blocks."""
    v = torch.sort(mean.flatten(), descending=True).values
    i = min(max(int(round(frac * v.numel())), 1), v.numel() - 1)
    return float((v[i - 1] * v[i]).sqrt())


# ------------------------------------------------------------------ prepare and run

def prepare(case, seed):
    c = case
    if c["kind"] in ("cond", "fixed"):
        s = _prompt_inputs(c, seed)
        if c["mixed"]:
            s["prefix"] = cb._build_prompt_blocks(s["k"], s["v"], c["block"], mixed=True,
                                                  k_bar_dtype=DTYPES[c["kbar"]])
        else:
            s["prefix"] = cb._build_prompt_blocks(s["k"], s["v"], c["block"])
        if c["kind"] == "cond":
            p = s["prefix"]
            mean, _ = _condition(s["q"], p["k_bar"], p["k_max"], p["k_min"], p["block_valid_counts"],
                                 p["v_norm_max"], c["mass"])
            s["eps"] = _eps_at(mean, c["frac"])
        return s
    s = _paged_inputs(c, seed)
    if c["kind"] == "topk" and c["kv"] == "fp8":
        s["scales"] = s["scales"] + (ia.sequence_scales(s["scales"], s["table"]),)
    if c["kind"] == "serve":
        nb_max = max(-(-(n + 1) // c["block"]) for n in s["lens"])
        s["old"] = s["seq"].clone()
        s["sum"] = ia.build_block_summaries(s["k"], s["v"], s["table"], s["old"], c["block"], nb_max=nb_max)
    return s


def run(state):
    s = state
    c = s["case"]
    kind = c["kind"]
    if kind == "topk":
        return ia.sparse_topk_decode(s["q"], s["k"], s["v"], s["table"], s["seq"], s["keys"], c["k"],
                                     block_size=c["block"], forced_first=c["ff"], forced_last=c["fl"],
                                     k_cap=s["k_cap"], k_per_seq=s["kvec"], scales=s["scales"], score=c["score"],
                                     workspace=s["ws"])
    if kind == "dense":
        return ia.paged_decode(s["q"], s["k"], s["v"], s["table"], s["seq"], max_seq_len=s["max_len"],
                               scales=s["scales"], workspace=s["ws"])
    if kind == "summaries":
        return ia.build_block_summaries(s["k"], s["v"], s["table"], s["seq"], c["block"],
                                        nb_max=-(-s["max_len"] // c["block"]), full=c["full"], scales=s["scales"])
    if kind == "serve":
        # the scheduler writes the step's lengths, then the layer appends, refreshes and attends
        s["seq"].copy_(s["old"])
        ia.append_kv(s["k"], s["v"], s["table"], s["seq"], s["k_new"], s["v_new"])
        ia.update_block_summaries(s["sum"], s["k"], s["v"], s["table"], s["old"], s["seq"], c["block"],
                                  max_new_tokens=1)
        out = ia.sparse_topk_decode(s["q"], s["k"], s["v"], s["table"], s["seq"], s["sum"]["k_bar"], c["k"],
                                    block_size=c["block"], forced_first=c["ff"], forced_last=c["fl"],
                                    workspace=s["ws"])
        return {"out": out, "seq": s["seq"], "k_bar": s["sum"]["k_bar"], "counts": s["sum"]["block_valid_counts"],
                "pool_k": s["k"], "pool_v": s["v"]}
    if kind == "cond":
        return cb._condition_block_decode_output(
            q_grouped=s["q"], prompt_prefix=s["prefix"], k_suffix=s["ks"], v_suffix=s["vs"], suffix_len_dev=s["len"],
            block_size=c["block"], eps=s["eps"], prompt_len=c["seq"], attention_dtype=DTYPES[c["kv"]],
            workspace=s["ws"], term1_mass_exp=c["mass"], collect_stats=False)[0]
    return cb.fixed_mask_hybrid_attention(
        q_grouped=s["q"], prompt_prefix=s["prefix"], selected=s["mask"], k_suffix=s["ks"], v_suffix=s["vs"],
        block_size=c["block"], output_dtype=DTYPES[c["kv"]], workspace=s["ws"])


# ------------------------------------------------------------------ compulsory work

def work(case):
    c = case
    if c["kind"] in ("cond", "fixed"):
        nb = -(-c["seq"] // c["block"])
        sb = 4 if not c["mixed"] else 2
        kb = 2 if c["kbar"] == "bf16" else 4
        bb = BYTES[c["kv"]] if c["mixed"] else 4
        es = BYTES[c["kv"]]
        sel = c["frac"] * c["seq"] + c["suffix"]
        rows = (kb + 2 * bb) if c["kind"] == "cond" else kb
        byts = c["hkv"] * (nb * c["d"] * (rows + (1 - c["frac"]) * sb) + 2 * sel * c["d"] * es +
                           2 * c["g"] * c["d"] * es + 4 * nb)
        flops = 2.0 * c["hkv"] * c["g"] * c["d"] * ((4 if c["kind"] == "cond" else 2) * nb + 2 * sel)
        return {"bytes": byts, "flops": flops}
    lens = _lens(c)
    g = c["hq"] // c["hkv"]
    es, d, hkv = BYTES[c["kv"]], c["d"], c["hkv"]
    qb = 4 if c["kv"] == "f32" else 2
    qo = 2.0 * c["batch"] * c["hq"] * d * qb
    scales = 8.0 / c["page"] if c["kv"] == "fp8" else 0.0  # bytes a token and head
    if c["kind"] == "summaries":
        toks = sum(lens)
        nb = sum(-(-n // c["block"]) for n in lens)
        out = hkv * nb * (d * 2 * (4 if c["full"] else 1) + (4 if c["full"] else 0))
        reads = 2 if c["full"] else 1
        return {"bytes": toks * hkv * (reads * d * es + scales) + out, "flops": float(toks * hkv * d * 5)}
    if c["kind"] == "dense":
        toks = sum(lens)
        return {"bytes": qo + toks * hkv * (2 * d * es + scales), "flops": 4.0 * toks * c["hq"] * d}
    byts, flops = qo, 0.0
    key_bytes = qb * (2 if c["score"] == "quest" else 1)
    for n, k in zip(lens, _ks(c) if c["kind"] == "topk" else [c["k"]] * len(lens)):
        nb = -(-n // c["block"])
        toks = min(n, min(nb, k + c["ff"] + c["fl"]) * c["block"])
        byts += hkv * (nb * d * key_bytes + toks * (2 * d * es + scales))
        flops += hkv * (2.0 * nb * d + 4.0 * toks * g * d)
    if c["kind"] == "serve":
        byts += 2 * c["batch"] * hkv * d * es * (2 + c["block"] / 2.0)
    return {"bytes": byts, "flops": flops}


# ------------------------------------------------------------------ tolerances

def tolerance(case):
    """bf16 and fp8 caches round the softmax weights and the output to bf16 (2^-9 each,
    relative), so another order of the same sums moves an output by a rounding or two;
    float32 caches keep float32 sums.  Block extrema are copies; block means are float32
    sums rounded to their storage type."""
    if case["kind"] == "summaries":
        return {"rel": 2e-3, "max": 2e-2}
    if case["kv"] == "f32":
        return {"rel": 2e-5, "max": 2e-4}
    return {"rel": 1e-2, "max": 6e-2}


# ------------------------------------------------------------------ 64-bit results

def _attend(q, k, v, bias=None):
    """softmax(q k^T / sqrt(D) + bias) v of one head, 64 bits: q [G, D], k, v [T, D]."""
    lg = torch.matmul(q, k.t().contiguous()) * q.shape[-1] ** -0.5
    if bias is not None:
        lg = lg + bias
    return torch.matmul(torch.softmax(lg, -1), v)


def _topk_exact(c, s, pool_k, pool_v, lens, keys, ks):
    g = c["hq"] // c["hkv"]
    out = torch.zeros((c["batch"], c["hq"], c["d"]), device=DEV, dtype=torch.float64)
    ksc, vsc = (None, None) if s["scales"] is None else s["scales"][:2]
    for b, n in enumerate(lens):
        nb = -(-n // c["block"])
        for h in range(c["hkv"]):
            q = s["q"][b, h * g:(h + 1) * g].double()
            if c["score"] == "quest":
                hi, lo = (x[b, h, :nb].double() for x in keys)
                sc = torch.mv(hi, q.clamp_min(0).sum(0)) + torch.mv(lo, q.clamp_max(0).sum(0))
            else:
                sc = torch.mv(keys[b, h, :nb].double(), q.sum(0))
            forced = torch.zeros(nb, device=DEV, dtype=torch.bool)
            forced[:c["ff"]] = True
            if c["fl"]:
                forced[max(nb - c["fl"], 0):] = True
            order = torch.sort(sc.masked_fill(forced, -math.inf), descending=True, stable=True).indices
            take = min(ks[b], nb - int(forced.sum()))
            blk = torch.cat([torch.nonzero(forced).flatten(), order[:take]])
            tok = (blk[:, None] * c["block"] + torch.arange(c["block"], device=DEV)[None]).flatten()
            tok = tok[tok < n]
            pages = s["table"][b][tok // c["page"]].long()
            kk = pool_k[pages, h, tok % c["page"]].float().double()
            vv = pool_v[pages, h, tok % c["page"]].float().double()
            if ksc is not None:
                kk = kk * ksc[pages, h].double()[:, None]
                vv = vv * vsc[pages, h].double()[:, None]
            out[b, h * g:(h + 1) * g] = _attend(q, kk, vv)
    return out


def _mean_rows(x, n, block):
    """Block means of [Hkv, n, D] and the valid tokens per block."""
    nb = -(-n // block)
    cnt = torch.full((nb,), block, device=x.device, dtype=torch.float64)
    cnt[-1] = n - (nb - 1) * block
    return _blocks(x, block, 0.0).sum(2) / cnt[None, :, None], cnt


def _summaries_exact(c, s):
    lens = s["lens"]
    nb_max = -(-max(lens) // c["block"])
    shape = (c["batch"], c["hkv"], nb_max, c["d"])
    out = {"k_bar": torch.zeros(shape, device=DEV, dtype=torch.float64),
           "block_valid_counts": torch.zeros((c["batch"], nb_max), device=DEV, dtype=torch.int32)}
    if c["full"]:
        out["v_bar"] = torch.zeros(shape, device=DEV, dtype=torch.float64)
        out["k_max"] = torch.full(shape, -math.inf, device=DEV, dtype=torch.float64)
        out["k_min"] = torch.full(shape, math.inf, device=DEV, dtype=torch.float64)
        out["v_norm_max"] = torch.full(shape[:3], -math.inf, device=DEV, dtype=torch.float64)
    ksc, vsc = (None, None) if s["scales"] is None else s["scales"]
    for b, n in enumerate(lens):
        nb = -(-n // c["block"])
        x = _rows(s["k"], ksc, s["table"][b], n, torch.float64)
        mean, cnt = _mean_rows(x, n, c["block"])
        out["k_bar"][b, :, :nb] = mean
        out["block_valid_counts"][b, :nb] = cnt.to(torch.int32)
        if c["full"]:
            out["k_max"][b, :, :nb] = _blocks(x, c["block"], -math.inf).amax(2)
            out["k_min"][b, :, :nb] = _blocks(x, c["block"], math.inf).amin(2)
            y = _rows(s["v"], vsc, s["table"][b], n, torch.float64)
            out["v_bar"][b, :, :nb] = _mean_rows(y, n, c["block"])[0]
            out["v_norm_max"][b, :, :nb] = _blocks(y.square().sum(-1, keepdim=True).sqrt(), c["block"], 0.0).amax((2, 3))
    if c["full"]:
        out["v_norm_all"] = out["v_norm_max"].amax(-1)
    return out


def _prompt_exact(c, s):
    dt = DTYPES[c["kv"]]
    kb_t, vb_t, bd_t = (DTYPES[c["kbar"]], torch.bfloat16, dt) if c["mixed"] else (torch.float32,) * 3
    p, block, d = c["seq"], c["block"], c["d"]
    k64, v64 = s["k"].double(), s["v"].double()
    k_bar, cnt = _mean_rows(k64, p, block)
    k_bar = k_bar.to(kb_t)
    v_bar = _mean_rows(v64, p, block)[0].to(vb_t)
    if c["kind"] == "cond":
        k_max = _blocks(k64, block, -math.inf).amax(2).to(bd_t)
        k_min = _blocks(k64, block, math.inf).amin(2).to(bd_t)
        v_norm = _blocks(v64.square().sum(-1, keepdim=True).sqrt(), block, 0.0).amax((2, 3)).float()
        mean, z = _condition(s["q"], k_bar, k_max, k_min, cnt, v_norm, c["mass"])
        sel = mean > _eps_at(mean, c["frac"])
    else:
        sel = s["mask"]
        kb = k_bar.to(torch.bfloat16) if c["kv"] == "bf16" else k_bar
        z = torch.stack([torch.matmul(s["q"][h, :, 0].double(), kb[h].double().t().contiguous()) * d ** -0.5
                         for h in range(c["hkv"])]) + cnt.log()
    out = torch.zeros((c["hkv"], c["g"], 1, d), device=DEV, dtype=torch.float64)
    for h in range(c["hkv"]):
        q = s["q"][h, :, 0].double()
        tok = sel[h].repeat_interleave(block)[:p]
        kk = torch.cat([k64[h][tok], s["ks"][h].double()])
        vv = torch.cat([v64[h][tok], s["vs"][h].double()])
        lg = torch.cat([torch.matmul(q, kk.t().contiguous()) * d ** -0.5, z[h][:, ~sel[h]]], -1)
        out[h, :, 0] = torch.matmul(torch.softmax(lg, -1), torch.cat([vv, v_bar[h][~sel[h]].double()]))
    return out


def exact(case, seed):
    c = case
    if c["kind"] in ("cond", "fixed"):
        return _prompt_exact(c, _prompt_inputs(c, seed))
    s = _paged_inputs(c, seed)
    lens = s["lens"]
    if c["kind"] == "topk":
        return _topk_exact(c, s, s["k"], s["v"], lens, s["keys"], _ks(c))
    if c["kind"] == "summaries":
        return _summaries_exact(c, s)
    if c["kind"] == "dense":
        g = c["hq"] // c["hkv"]
        out = torch.zeros((c["batch"], c["hq"], c["d"]), device=DEV, dtype=torch.float64)
        ksc, vsc = (None, None) if s["scales"] is None else s["scales"]
        for b, n in enumerate(lens):
            x = _rows(s["k"], ksc, s["table"][b], n, torch.float64)
            y = _rows(s["v"], vsc, s["table"][b], n, torch.float64)
            for h in range(c["hkv"]):
                out[b, h * g:(h + 1) * g] = _attend(s["q"][b, h * g:(h + 1) * g].double(), x[h].contiguous(),
                                                    y[h].contiguous())
        return out
    # serve: the new token is written, its block's mean refreshed, then the layer call
    grown = [n + 1 for n in lens]
    nb_max = max(-(-n // c["block"]) for n in grown)
    k_bar = torch.zeros((c["batch"], c["hkv"], nb_max, c["d"]), device=DEV, dtype=torch.float64)
    counts = torch.zeros((c["batch"], nb_max), device=DEV, dtype=torch.int32)
    for b, n in enumerate(lens):
        at = int(s["table"][b, n // c["page"]])
        s["k"][at, :, n % c["page"]] = s["k_new"][b]
        s["v"][at, :, n % c["page"]] = s["v_new"][b]
        mean, cnt = _mean_rows(_rows(s["k"], None, s["table"][b], n + 1, torch.float64), n + 1, c["block"])
        k_bar[b, :, :mean.shape[1]] = mean
        counts[b, :mean.shape[1]] = cnt.to(torch.int32)
    keys = k_bar.to(torch.bfloat16)
    out = _topk_exact(c, s, s["k"], s["v"], grown, keys, [c["k"]] * len(lens))
    return {"out": out, "seq": torch.tensor(grown, dtype=torch.int32), "k_bar": k_bar, "counts": counts,
            "pool_k": s["k"], "pool_v": s["v"]}

"""Performance cases of the attention path: what a serving program calls, per layer.

Every case is one layer's attention of one step over paged caches: the step's
new rows are written through the slot mapping, then its query rows attend over
block tables. The kinds follow the operators of ``ironpangu_amd.ops``:

  gqa_step     write + ragged GQA decode, bf16 caches (one call)
  gqa_c8       quantizing write + GQA decode over int8 caches
  gqa_prefill  write + packed varlen prefill, with or without decode rows
  mla_step     fused latent-row writer + MLA decode, bf16 or packed C8 rows
  mla_rows     latent-row writer + MLA attention of packed query rows: bf16
               windows with learned sinks, or C8 rows over index lists
  mla_rowq     MLA attention over row-quantized (int8 / int4) latent rows
  gated        q/k producer + gated attention of the session ABI's Qwen shape

Lengths are the quantiles of a uniform or log-uniform distribution over
[lo, hi], so a case's work is a function of the case alone; their order, the
block tables and all values come from the seed. Caches hold N(0, 1) (GQA) or
N(0, 0.5) (MLA) values, the programs' own distributions after normalization.
The calls keep their block tables, lengths, workspace and output buffer, as a
serving loop does.
"""
from __future__ import annotations

import math

import numpy as np
import torch

from ironpangu_amd import ops

LATENT, ROPE, WIDE = 512, 64, 576
MLA_SCALE = 1.0 / math.sqrt(192.0)
EPS = 1e-5


# ---------------------------------------------------------------- the cases

def listed():
    return [
        # A small interactive batch: launches and latency, not bandwidth.
        dict(name="gqa_step_8", kind="gqa_step", seqs=8, lo=16, hi=512, dist="uniform",
             q_heads=16, kv_heads=2, head_dim=128, block=128),
        # Continuous batching at scale: ragged contexts, bandwidth-bound decode.
        dict(name="gqa_step_256", kind="gqa_step", seqs=256, lo=128, hi=32768, dist="log",
             q_heads=16, kv_heads=2, head_dim=128, block=128),
        # The same service over the quantized cache.
        dict(name="gqa_c8_256", kind="gqa_c8", seqs=256, lo=1024, hi=16384, dist="uniform",
             q_heads=16, kv_heads=2, head_dim=128, block=128),
        # A scheduler step that mixes prompt chunks with decode rows.
        dict(name="gqa_mixed_200", kind="gqa_prefill", chunks=8, c_lo=64, c_hi=2048, p_lo=0,
             p_hi=8192, decodes=192, d_lo=256, d_hi=16384, q_heads=16, kv_heads=2, head_dim=128,
             block=128),
        # Fresh prompts of odd lengths, no cached context: short causal prefill.
        dict(name="gqa_prompts_3", kind="gqa_prefill", chunks=3, c_lo=187, c_hi=1777, p_lo=0,
             p_hi=0, decodes=0, d_lo=1, d_hi=1, q_heads=16, kv_heads=2, head_dim=128, block=128),
        # MLA decode over long contexts, bf16 latent rows: the largest read.
        dict(name="mla_step_bf16_128", kind="mla_step", c8=False, seqs=128, lo=1024, hi=65536,
             dist="log", heads=16, block=64),
        # The same service over packed C8 rows.
        dict(name="mla_step_c8_128", kind="mla_step", c8=True, seqs=128, lo=1024, hi=65536,
             dist="log", heads=16, block=64),
        # The same contexts over row-quantized int8 rows.
        dict(name="mla_rowq8_128", kind="mla_rowq", bits=8, seqs=128, count=1, lo=1024, hi=65536,
             dist="log", heads=16, block=64, window=0, sinks=0),
        # Decode rows of a sliding-window layer with learned sinks.
        dict(name="mla_window_128", kind="mla_rows", topk=0, seqs=128, c_lo=1, c_hi=1, p_lo=4096,
             p_hi=65536, heads=16, block=16, window=2048, sinks=128),
        # Prompt chunks of a sliding-window layer with learned sinks.
        dict(name="mla_window_chunks_3", kind="mla_rows", topk=0, seqs=3, c_lo=101, c_hi=401,
             p_lo=0, p_hi=8192, heads=16, block=16, window=2048, sinks=128),
        # Decode rows of a sparse layer: top-k candidates, learned sinks, C8 rows.
        dict(name="mla_sparse_128", kind="mla_rows", topk=2048, seqs=128, c_lo=1, c_hi=1,
             p_lo=4096, p_hi=65536, heads=16, block=64, window=0, sinks=128),
        # The session ABI's layer: per-position row table and mask.
        dict(name="gated_64", kind="gated", batch=64, context=32768, lo=128, hi=32768),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    case = _draw(rng)
    if case["kind"] in ("mla_step", "mla_rowq"):  # at most 1.9 M cached keys, as the largest listed case
        while int(_sizes(case)[1].sum()) > 1_900_000:
            case.update(lo=max(case.get("count", 1), case["lo"] * 3 // 4), hi=case["hi"] * 3 // 4)
    return case


def _draw(rng):
    kind = rng.choice(["gqa_step", "gqa_step", "gqa_c8", "gqa_prefill", "gqa_prefill", "mla_step",
                       "mla_step", "mla_rows", "mla_rows", "mla_rows", "mla_rowq", "gated"])
    if kind in ("gqa_step", "gqa_c8"):
        q_heads, kv_heads, head_dim = rng.choice([(16, 2, 128), (16, 2, 128), (8, 2, 256),
                                                  (8, 1, 64), (16, 16, 128)])
        row = 2 * kv_heads * head_dim * (2 if kind == "gqa_step" else 1)
        seqs, hi = _log(rng, 1, 256), _log(rng, 48, 32768)
        hi = max(48, min(hi, int(1.8e9 / row / seqs)))
        return dict(kind=kind, seqs=seqs, lo=_log(rng, 16, hi), hi=hi,
                    dist=rng.choice(["uniform", "log"]), q_heads=q_heads, kv_heads=kv_heads,
                    head_dim=head_dim,
                    block=rng.choice([16, 32, 64, 128] if kind == "gqa_step" else [32, 64, 128]))
    if kind == "gqa_prefill":
        q_heads, kv_heads, head_dim = rng.choice([(16, 2, 128), (16, 2, 128), (8, 2, 256), (8, 1, 64)])
        decodes = rng.choice([0, _log(rng, 1, 192)])
        return dict(kind=kind, chunks=rng.randint(1, 8), c_lo=_log(rng, 2, 256),
                    c_hi=_log(rng, 256, 2048), p_lo=0, p_hi=rng.choice([0, _log(rng, 64, 8192)]),
                    decodes=decodes, d_lo=1 + rng.randint(0, 255), d_hi=_log(rng, 256, 16384),
                    q_heads=q_heads, kv_heads=kv_heads, head_dim=head_dim,
                    block=rng.choice([32, 64, 128]))
    if kind == "mla_step":
        c8, hi = rng.random() < 0.5, _log(rng, 64, 65536)
        return dict(kind=kind, c8=c8, seqs=_log(rng, 1, 128), lo=_log(rng, 32, hi), hi=hi,
                    dist=rng.choice(["uniform", "log"]) if hi < 32768 else "log",
                    heads=rng.choice([6, 16, 16]), block=rng.choice([32, 64, 128]))
    if kind == "mla_rows":
        topk = rng.choice([0, 0, 512, 2048])
        chunked = rng.random() < 0.6
        heads = rng.choice([6, 16, 16])
        sinks = rng.choice([0, 128, 128])
        if chunked:
            c_lo = _log(rng, 2, 301)
            c_hi = c_lo + _log(rng, 1, 800 if topk == 0 else 200)
            seqs = rng.randint(1, 3)
            if sinks:  # at most 750 rows of a layer with sinks per call
                c_lo = min(c_lo, 750 // seqs)
                c_hi = min(c_hi, 1500 // seqs - c_lo)
        else:
            c_lo = c_hi = 1
            seqs = _log(rng, 1, 128)
        return dict(kind=kind, topk=topk, seqs=seqs, c_lo=c_lo, c_hi=c_hi, p_lo=0 if chunked else 64,
                    p_hi=_log(rng, 65, 8192 if chunked else 65536), heads=heads,
                    block=rng.choice([32, 64, 128] if topk else [16, 16, 32, 64]),
                    window=0 if topk else rng.choice([512, 2048]), sinks=sinks)
    if kind == "mla_rowq":
        hi = _log(rng, 64, 32768)
        count = rng.choice([1, 1, rng.randint(2, 100)])
        seqs = _log(rng, 1, 128) if count == 1 else rng.randint(1, 3)
        return dict(kind=kind, bits=rng.choice([8, 8, 4]), seqs=seqs, count=count,
                    lo=max(count, _log(rng, 32, hi)), hi=max(count, hi), dist="log",
                    heads=rng.choice([6, 16, 16]), block=rng.choice([16, 32, 64]),
                    window=rng.choice([0, 512, 2048]) if count == 1 else rng.choice([512, 2048]),
                    sinks=rng.choice([0, 128]))
    hi = _log(rng, 128, 32768)
    return dict(kind="gated", batch=_log(rng, 1, 64), context=hi + rng.randint(0, 77),
                lo=_log(rng, 17, hi), hi=hi)


# ---------------------------------------------------------------- sizes of a case

def _quantiles(n, lo, hi, dist):
    """n lengths: the quantiles of the distribution over [lo, hi]."""
    if n == 0:
        return np.zeros(0, np.int64)
    u = (np.arange(n) + 0.5) / n
    lo, hi = max(0, min(lo, hi)), max(lo, hi)
    x = lo + (hi - lo) * u if dist == "uniform" or lo == 0 else lo * (hi / lo) ** u
    return np.rint(x).astype(np.int64)


def _sizes(case):
    """(query rows, cached keys after the step's writes) of every sequence."""
    k = case["kind"]
    if k in ("gqa_step", "gqa_c8", "mla_step"):
        kv = _quantiles(case["seqs"], case["lo"], case["hi"], case["dist"])
        return np.ones_like(kv), np.maximum(kv, 1)
    if k == "mla_rowq":
        kv = _quantiles(case["seqs"], case["lo"], case["hi"], case["dist"])
        return np.full_like(kv, case["count"]), np.maximum(kv, case["count"])
    if k == "mla_rows":
        n = case["seqs"]
        rows = np.maximum(_quantiles(n, case["c_lo"], case["c_hi"], "uniform"), 1)
        prior = _quantiles(n, case["p_lo"], case["p_hi"], "uniform")[::-1]
        return rows, rows + prior
    n = case["chunks"]
    rows = np.maximum(_quantiles(n, case["c_lo"], case["c_hi"], "uniform"), 1)
    prior = _quantiles(n, case["p_lo"], case["p_hi"], "uniform")[(np.arange(n) * 3 + 1) % n]
    dec = np.maximum(_quantiles(case["decodes"], case["d_lo"], case["d_hi"], "uniform"), 1)
    return (np.concatenate([rows, np.ones_like(dec)]), np.concatenate([rows + prior, dec]))


def _live(case):
    """Live positions of every gated request."""
    return np.minimum(_quantiles(case["batch"], case["lo"], case["hi"], "log"), case["context"])


def _visible(case):
    """(row, key) pairs attended, and cached keys read at least once."""
    rows, kv = _sizes(case)
    window, topk = case.get("window", 0), case.get("topk", 0)
    cap = topk or window or (1 << 40)
    pairs = keys = 0
    for c, n in zip(rows.tolist(), kv.tolist()):
        causal = np.arange(n - c + 1, n + 1)
        pairs += int(np.minimum(causal, cap).sum())
        keys += min(n, c * topk) if topk else min(n, (window or n) + c - 1)
    return pairs, keys


def work(case):
    k = case["kind"]
    if k == "gated":
        live, b = int(_live(case).sum()), case["batch"]
        return {"bytes": live * 2048 + b * case["context"] * 4 + live * 8 + b * (9 * 1024 + 4096 + 4096),
                "flops": 4 * 8 * 256 * live}
    rows, kv = _sizes(case)
    pairs, keys = _visible(case)
    n = int(rows.sum())
    if k.startswith("gqa"):
        hq, hkv, d = case["q_heads"], case["kv_heads"], case["head_dim"]
        tok = 2 * hkv * (d + 4) if k == "gqa_c8" else 2 * hkv * d * 2
        return {"bytes": keys * tok + n * (2 * hq * d * 2 + 2 * hkv * d * 2 + tok + 8),
                "flops": 4 * hq * d * pairs}
    h = case["heads"]
    if k == "mla_rowq":
        row, new = WIDE * case["bits"] // 8 + 4, 0
    else:
        row = 656 if case.get("c8") or case.get("topk") else 1152
        new = n * (1152 + 256 + row)
    sinks = case.get("sinks", 0)
    byts = keys * row + n * h * (WIDE + LATENT) * 2 + new + sinks * (WIDE + LATENT) * 2
    return {"bytes": byts + n * case.get("topk", 0) * 4,
            "flops": 2 * h * (WIDE + LATENT) * (pairs + n * sinks)}


def tolerance(case):
    # bf16 probabilities and bf16 outputs with fp32 sums.
    return {"rel": 0.01, "max": 0.08}


# ---------------------------------------------------------------- inputs

def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed))


def _randn(gen, shape, std=1.0, dtype=torch.bfloat16):
    return torch.randn(shape, generator=gen, device="cuda", dtype=dtype).mul_(std)


def _codes(gen, shape, top=127):
    """Integer codes of quantized normal rows (scale = row max / top, about 3.3 sigma)."""
    x = torch.randn(shape, generator=gen, device="cuda", dtype=torch.bfloat16)
    return x.mul_(top / 3.3).round_().clamp_(-top, top).to(torch.int8)


def _dev(a, dtype):
    return torch.from_numpy(np.ascontiguousarray(a)).to("cuda", dtype)


def _paging(seed, kv, block):
    """Block tables over a random permutation of the pool, and the pool's blocks."""
    rng = np.random.default_rng(seed)
    need = (kv + block - 1) // block
    pool = int(need.sum()) + 16
    perm = rng.permutation(pool)
    table = np.zeros((len(kv), int(need.max())), np.int64)
    at = 0
    for i, b in enumerate(need):
        table[i, :b] = perm[at:at + b]
        at += int(b)
    return table, pool


def _order(seed, rows, kv):
    o = np.random.default_rng(seed + 1).permutation(len(kv))
    return rows[o], kv[o]


def _new_slots(table, rows, kv, block):
    """Physical token row of every new row, the last `rows` positions of each sequence."""
    pos = np.concatenate([np.arange(n - c, n) for c, n in zip(rows, kv)])
    seq = np.repeat(np.arange(len(kv)), rows)
    return table[seq, pos // block] * block + pos % block


def prepare(case, seed):
    s = {"case": case, "gen": _gen(seed)}
    return (_prepare_gated if case["kind"] == "gated" else
            _prepare_gqa if case["kind"].startswith("gqa") else _prepare_mla)(case, seed, s)


def _prepare_paged(case, seed, s):
    rows, kv = _sizes(case)
    if case["kind"] != "gqa_prefill":  # chunks stay first in a mixed batch
        rows, kv = _order(seed, rows, kv)
    block = case["block"]
    table, pool = _paging(seed, kv, block)
    cu = np.concatenate([[0], np.cumsum(rows)])
    s.update(rows=rows, kv=kv, table=table, pool=pool, n=int(rows.sum()),
             max_context=int(kv.max()), tables=_dev(table, torch.int32),
             kv_lens=_dev(kv, torch.int32), cu=_dev(cu, torch.int32),
             slots=_dev(_new_slots(table, rows, kv, block), torch.int64))


def _prepare_gqa(case, seed, s):
    _prepare_paged(case, seed, s)
    g, n, pool, block = s["gen"], s["n"], s["pool"], case["block"]
    hq, hkv, d = case["q_heads"], case["kv_heads"], case["head_dim"]
    s["q"] = _randn(g, (n, hq, d))
    s["k_new"], s["v_new"] = _randn(g, (n, hkv, d)), _randn(g, (n, hkv, d))
    if case["kind"] == "gqa_c8":
        for c in "kv":
            s[c + "_cache"] = _codes(g, (pool, block, hkv, d))
            s[c + "_scale"] = torch.rand((pool, block, hkv), generator=g, device="cuda").mul_(0.01).add_(0.02)
    else:
        s["k_cache"], s["v_cache"] = (_randn(g, (pool, block, hkv, d)) for _ in "kv")
    s["out"] = torch.empty_like(s["q"])
    if case["kind"] == "gqa_prefill":
        s["workspace"] = ops.prefill_workspace(len(s["kv"]), n, hq, d, s["max_context"])
    else:
        s["workspace"] = ops.decode_workspace(n, hq, d, s["max_context"])
    return s


def _prepare_mla(case, seed, s):
    _prepare_paged(case, seed, s)
    g, n, pool, block, h = s["gen"], s["n"], s["pool"], case["block"], case["heads"]
    s["q"] = _randn(g, (n, h, WIDE), 0.5)
    if case["kind"] == "mla_rowq":
        codes = _codes(g, (pool * block, WIDE), 127 if case["bits"] == 8 else 7)
        if case["bits"] == 4:
            lo, hi = codes[:, 0::2].view(torch.uint8) & 15, codes[:, 1::2].view(torch.uint8)
            codes = lo | (hi << 4)
        s["cache"] = codes.view(torch.uint8).reshape(pool, block, -1).contiguous()
        s["row_scales"] = torch.rand(pool * block, generator=g, device="cuda").mul_(0.5).add_(1.0).mul_(
            0.5 * 3.3 / (127 if case["bits"] == 8 else 7))
    else:
        if case.get("c8") or case.get("topk"):
            codes = _codes(g, (pool * block, LATENT)).view(torch.uint8)
            rope = _randn(g, (pool * block, ROPE), 0.5).view(torch.uint8)
            scale = torch.rand((pool * block, 4), generator=g, device="cuda").mul_(0.004).add_(0.011)
            s["cache"] = torch.cat([codes, rope, scale.view(torch.uint8)], 1).reshape(pool, block, 656)
        else:
            s["cache"] = _randn(g, (pool, block, WIDE), 0.5)
        s["x_new"] = _randn(g, (n, WIDE))
        s["gamma"] = _randn(g, (LATENT,), 0.05).add_(0.5)
        angle = torch.rand((n, ROPE // 2), generator=g, device="cuda").mul_(2 * math.pi).repeat(1, 2)
        s["cos"], s["sin"] = angle.cos().to(torch.bfloat16), angle.sin().to(torch.bfloat16)
    sinks, topk = case.get("sinks", 0), case.get("topk", 0)
    if sinks:
        s["sink_k"], s["sink_v"] = _randn(g, (sinks, WIDE), 0.5), _randn(g, (sinks, LATENT), 0.5)
    if topk:
        # Each row's candidates: distinct causal positions in random order, -1 padding.
        causal = torch.from_numpy(np.concatenate(
            [np.arange(n - c + 1, n + 1) for c, n in zip(s["rows"], s["kv"])])).cuda()
        idx = torch.full((n, topk), -1, dtype=torch.int32, device="cuda")
        for a in range(0, n, 64):
            c = causal[a:a + 64, None]
            key = torch.rand((c.shape[0], int(c.max())), generator=g, device="cuda")
            key.masked_fill_(torch.arange(key.shape[1], device="cuda")[None] >= c, 2.0)
            k = min(topk, key.shape[1])
            v, i = key.topk(k, dim=1, largest=False)
            idx[a:a + 64, :k] = torch.where(v < 1.5, i, -1).to(torch.int32)
        s["indices"] = idx
    s["out"] = torch.empty((n, h, LATENT), dtype=torch.bfloat16, device="cuda")
    if case["kind"] == "mla_step":
        s["workspace"] = ops.mla_workspace(n, h, s["max_context"], block)
    else:
        size = ops.lib().ifattn_mla_attention_workspace_size(n, h, s["max_context"],
                                                             case.get("window", 0), topk, sinks, block)
        s["workspace"] = torch.empty(max(int(size), 16), dtype=torch.uint8, device="cuda")
    return s


def _prepare_gated(case, seed, s):
    g, b, context = s["gen"], case["batch"], case["context"]
    live = np.random.default_rng(seed).permutation(_live(case))
    slots = min(1 << 20, int(live.sum()) + 1024)
    perm = torch.randperm(slots, generator=g, device="cuda")[:int(live.sum())]
    at = np.concatenate([[0], np.cumsum(live)])
    table = torch.zeros((b, context), dtype=torch.int64, device="cuda")
    mask = torch.full((b, context), -math.inf, device="cuda")
    for i, n in enumerate(live.tolist()):
        table[i, :n] = perm[at[i]:at[i + 1]]
        mask[i, :n] = 0.0
    s.update(live=live, table=table, mask=mask,
             append=table[torch.arange(b, device="cuda"), _dev(live - 1, torch.int64)].contiguous(),
             positions=_dev(live - 1, torch.int64),
             packed_q=_randn(g, (b, 8, 512)), k=_randn(g, (b, 2, 256)), v=_randn(g, (b, 512)),
             q_gamma=torch.randn(256, generator=g, device="cuda").mul_(0.05).add_(1.0),
             k_gamma=torch.randn(256, generator=g, device="cuda").mul_(0.05).add_(1.0),
             keys=_randn(g, (slots, 512)), values=_randn(g, (slots, 512)),
             out=torch.empty((b, 8, 256), dtype=torch.bfloat16, device="cuda"))
    size = ops.lib().ifattn_gated_paged_attention_workspace_size(b, context)
    s["workspace"] = torch.empty(max(int(size), 16), dtype=torch.uint8, device="cuda")
    return s


# ---------------------------------------------------------------- one pass

def run(s):
    """One layer's attention of one step; returns its outputs and updated caches."""
    case = s["case"]
    kind, out, ws = case["kind"], s["out"], s["workspace"]
    if kind == "gqa_step":
        ops.paged_decode_step(s["q"], s["k_new"], s["v_new"], s["k_cache"], s["v_cache"], s["slots"],
                              s["tables"], s["kv_lens"], s["max_context"], out=out, workspace=ws)
        return out, s["k_cache"], s["v_cache"]
    if kind == "gqa_c8":
        ops.kv_cache_write_c8(s["k_new"], s["v_new"], s["k_cache"], s["v_cache"], s["k_scale"],
                              s["v_scale"], s["slots"])
        ops.paged_decode(s["q"], s["k_cache"], s["v_cache"], s["tables"], s["kv_lens"],
                         s["max_context"], out=out, workspace=ws, k_scale=s["k_scale"],
                         v_scale=s["v_scale"])
        return out, s["k_cache"], s["v_cache"], s["k_scale"], s["v_scale"]
    if kind == "gqa_prefill":
        ops.kv_cache_write(s["k_new"], s["v_new"], s["k_cache"], s["v_cache"], s["slots"])
        ops.varlen_prefill(s["q"], s["k_cache"], s["v_cache"], s["tables"], s["cu"], s["kv_lens"],
                           int(s["rows"].max()), s["max_context"], out=out, workspace=ws)
        return out, s["k_cache"], s["v_cache"]
    if kind == "mla_step":
        ops.mla_decode_step(s["q"], s["x_new"], s["gamma"], s["cos"], s["sin"], s["cache"], s["tables"],
                            s["kv_lens"], s["max_context"], eps=EPS, out=out, workspace=ws)
        return out, s["cache"]
    if kind == "mla_rows":
        ops.mla_norm_rope_cache_write(s["x_new"], s["gamma"], s["cos"], s["sin"], s["cache"], s["slots"],
                                      eps=EPS)
        ops.mla_attention(s["q"], s["cache"], s["tables"], s["kv_lens"], s["max_context"],
                          cu_seqlens=s["cu"], indices=s.get("indices"), window=case["window"],
                          sink_keys=s.get("sink_k"), sink_values=s.get("sink_v"), out=out, workspace=ws)
        return out, s["cache"]
    if kind == "mla_rowq":
        ops.mla_attention(s["q"], s["cache"], s["tables"], s["kv_lens"], s["max_context"],
                          cu_seqlens=s["cu"], window=case["window"], sink_keys=s.get("sink_k"),
                          sink_values=s.get("sink_v"), out=out, workspace=ws,
                          row_scales=s["row_scales"], bits=case["bits"])
        return out
    q, k, gate = ops.qk_norm_rope_gate(s["packed_q"], s["k"], s["q_gamma"], s["k_gamma"], s["positions"])
    ops.gated_paged_attention(q, k.view(-1, 512), s["v"], gate, s["keys"], s["values"], s["append"],
                              s["table"], s["mask"], out=out, workspace=ws)
    return out, q, k, gate, s["keys"], s["values"]


# ---------------------------------------------------------------- in 64 bits

def _attend(q, k, v, scale, mask=None):
    """Softmax attention of q [.., rows, d] over k [.., keys, d], v [.., keys, dv], float64."""
    x = torch.matmul(q, k.transpose(-1, -2).contiguous()) * scale
    if mask is not None:
        x = x.masked_fill(~mask, -math.inf)
    return torch.matmul(torch.softmax(x, dim=-1), v)


def exact(case, seed):
    s = prepare(case, seed)
    if case["kind"] == "gated":
        return _exact_gated(case, s)
    return _exact_gqa(case, s) if case["kind"].startswith("gqa") else _exact_mla(case, s)


def _rows_of(s, i, lo, hi):
    """Physical token rows of positions [lo, hi) of sequence i."""
    pos = np.arange(lo, hi)
    block = s["case"]["block"]
    return _dev(s["table"][i, pos // block] * block + pos % block, torch.int64)


def _quantized(x):
    """Symmetric int8 codes times scale along the last axis, float64."""
    x = x.float()
    scale = x.abs().amax(-1, keepdim=True) / 127
    codes = torch.where(scale > 0, (x / scale).round().clamp(-127, 127), torch.zeros_like(x))
    return codes.double() * scale.double()


def _exact_gqa(case, s):
    hq, hkv, d = case["q_heads"], case["kv_heads"], case["head_dim"]
    c8, group = case["kind"] == "gqa_c8", hq // hkv
    flat = {c: s[c + "_cache"].view(-1, hkv, d) for c in "kv"}
    out = torch.empty(s["q"].shape, dtype=torch.float64, device="cuda")
    at = 0
    for i, (c, n) in enumerate(zip(s["rows"].tolist(), s["kv"].tolist())):
        phys = _rows_of(s, i, 0, n)
        kv = []
        for name in "kv":
            x = flat[name][phys].double()
            if c8:
                x *= s[name + "_scale"].view(-1, hkv)[phys].double()[..., None]
            new = s[name + "_new"][at:at + c]
            x[n - c:] = _quantized(new) if c8 else new.double()
            kv.append(x.transpose(0, 1).contiguous())  # [hkv, n, d]
        for a in range(0, c, 256):
            b = min(c, a + 256)
            q = s["q"][at + a:at + b].double().view(b - a, hkv, group, d).permute(1, 0, 2, 3)
            seen = torch.arange(n, device="cuda")[None] <= torch.arange(n - c + a, n - c + b, device="cuda")[:, None]
            seen = seen[:, None].expand(-1, group, -1).reshape(-1, n)
            o = _attend(q.reshape(hkv, -1, d), kv[0], kv[1], 1 / math.sqrt(d), seen if c > 1 else None)
            out[at + a:at + b] = o.view(hkv, b - a, group, d).permute(1, 0, 2, 3).reshape(b - a, hq, d)
        at += c
    return (out,) + (None,) * (4 if c8 else 2)


def _new_rows(case, s):
    """The latent rows the writer stores, as the cache holds them, float64."""
    x = s["x_new"].double()
    y = x[:, :LATENT]
    y = y / torch.sqrt(y.square().mean(-1, keepdim=True) + EPS) * s["gamma"].double()
    r = x[:, LATENT:]
    r = r * s["cos"].double() + torch.cat([-r[:, 32:], r[:, :32]], 1) * s["sin"].double()
    y = (_quantized(y.view(-1, 4, 128)).view(-1, LATENT) if s["cache"].dtype == torch.uint8
         else y.to(torch.bfloat16).double())
    return torch.cat([y, r.to(torch.bfloat16).double()], 1)


def _latent(case, s, phys):
    """Cached latent rows [keys, 576] in float64."""
    flat = s["cache"].view(-1, s["cache"].shape[2])[phys]
    if case["kind"] == "mla_rowq":
        if case["bits"] == 4:
            both = torch.stack([flat & 15, flat >> 4], -1).view(flat.shape[0], WIDE).to(torch.int16)
            codes = (both ^ 8) - 8
        else:
            codes = flat.view(torch.int8)
        # The attention's keys are the bf16 values of the dequantized cache.
        return (codes.float() * s["row_scales"][phys][:, None]).to(torch.bfloat16).double()
    if flat.dtype != torch.uint8:
        return flat.double()
    codes = flat[:, :LATENT].contiguous().view(torch.int8).double().view(-1, 4, 128)
    scale = flat[:, 640:].contiguous().view(torch.float32).double()
    rope = flat[:, LATENT:640].contiguous().view(torch.bfloat16).double()
    return torch.cat([(codes * scale[..., None]).view(-1, LATENT), rope], 1)


def _exact_mla(case, s):
    h = case["heads"]
    out = torch.empty(s["out"].shape, dtype=torch.float64, device="cuda")
    new = _new_rows(case, s) if "x_new" in s else None
    sinks = case.get("sinks", 0)
    sk, sv = (s["sink_k"].double(), s["sink_v"].double()) if sinks else (None, None)
    window, at = case.get("window", 0), 0
    for i, (c, n) in enumerate(zip(s["rows"].tolist(), s["kv"].tolist())):
        first = max(0, n - c + 1 - window) if window else 0
        rows = _latent(case, s, _rows_of(s, i, first, n))
        if new is not None:
            rows[n - c - first:] = new[at:at + c]
        for a in range(0, c, 64):
            b = min(c, a + 64)
            q = s["q"][at + a:at + b].double()
            if "indices" in s:
                for t in range(a, b):
                    pick = s["indices"][at + t].long()
                    k = rows[pick[pick >= 0]]
                    v = k[:, :LATENT]
                    if sinks:
                        k, v = torch.cat([sk, k]), torch.cat([sv, v])
                    out[at + t] = _attend(q[t - a], k, v, MLA_SCALE)
                continue
            hi = n - c + b
            lo = max(0, n - c + a + 1 - window) if window else 0
            k = rows[lo - first:hi - first]
            v = k[:, :LATENT]
            pos = torch.arange(lo, hi, device="cuda")[None]
            row = torch.arange(n - c + a, n - c + b, device="cuda")[:, None]
            seen = (pos <= row) & (pos > row - window) if window else pos <= row
            if sinks:
                k, v = torch.cat([sk, k]), torch.cat([sv, v])
                seen = torch.cat([torch.ones((b - a, sinks), dtype=torch.bool, device="cuda"), seen], 1)
            seen = seen[:, None].expand(-1, h, -1).reshape(-1, k.shape[0])
            out[at + a:at + b] = _attend(q.reshape(-1, WIDE), k, v, MLA_SCALE, seen).view(b - a, h, LATENT)
        at += c
    return out if case["kind"] == "mla_rowq" else (out, None)


def _exact_gated(case, s):
    def normed(x, gamma):
        x = x.double()
        y = x / torch.sqrt(x.square().mean(-1, keepdim=True) + 1e-6) * gamma.double()
        f = 1.0 / 1e7 ** (torch.arange(32, device="cuda", dtype=torch.float64) / 32)
        ang = s["positions"].double()[:, None, None] * f
        # The rotation's cos and sin are bf16 by definition of the operator.
        c, sn = ang.float().cos().to(torch.bfloat16).double(), ang.float().sin().to(torch.bfloat16).double()
        a, b = y[..., :32], y[..., 32:64]
        return torch.cat([a * c - b * sn, b * c + a * sn, y[..., 64:]], -1)

    q = normed(s["packed_q"][..., :256], s["q_gamma"])
    k = normed(s["k"], s["k_gamma"])
    gate = torch.sigmoid(s["packed_q"][..., 256:].double())
    out = torch.empty(s["out"].shape, dtype=torch.float64, device="cuda")
    for i, n in enumerate(s["live"].tolist()):
        phys = s["table"][i, :n]
        kk, vv = (s[x][phys].double().view(n, 2, 256).transpose(0, 1).contiguous() for x in ("keys", "values"))
        kk[:, n - 1], vv[:, n - 1] = k[i], s["v"][i].double().view(2, 256)
        out[i] = _attend(q[i].view(2, 4, 256), kk, vv, 1 / 16).reshape(8, 256)
    return out * gate, q, k, gate, None, None

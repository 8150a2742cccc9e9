"""The attention work that a serving program asks of this library.

Each case is one step of one transformer layer (or the attention of that
step) as a serving loop issues it: single-token decode of one sequence and of
batches, chunked prefill, steps that mix both, whole layer passes (head norm +
RoPE + cache write, attention, o_proj) and the block-sparse decode.  Shapes
are those of the repository's tests and benchmark: 16 q / 8 kv heads x 256,
16 q / 2 kv heads x 512, windows of 1024 on page rings, 64-token pages, o_proj
to 2816 columns, and the 64 q / 4 kv x 128 block-sparse layer.

Fields of a case:
  op      "attention": the attention over a cache that already holds the
          step's tokens; "layer": append, attention and o_proj;
          "sparse": lightning indexer and block-sparse attention
  heads   "256" (16 q / 8 kv) or "512" (16 q / 2 kv)
  kv      "bf16" or "bq" (int8 codes with f32 scales)
  window  0 for full attention, else the sliding window
  seqs, new, lo, hi
          seqs sequences feed `new` tokens each on contexts of U[lo, hi]
          tokens (their lengths come from `lens`, a seed of the case)
  extra   further sequences that feed one token each in the same step
  cap     the worker capacity that the plan splits for (the benchmark's
          choice for the kind of step)
"""
import math
import random

import numpy as np
import torch

from inferno_amd import attention as A
from inferno_amd.kv import FULL, SLIDING, AttentionPlan, KVRunTable

PAGE = 64
HIDDEN = 2816  # o_proj output columns
SHAPES = {"256": (16, 8, 256, 128, 128), "512": (16, 2, 512, 64, 256)}  # nq, nkv, d, rope half, pair stride
S_NQ, S_NKV, S_D, S_IH, S_BLOCK, S_TOPK = 64, 4, 128, 4, 128, 16


def _case(name, op, **kw):
    c = {"op": op, "heads": "256", "kv": "bf16", "window": 0, "seqs": 1, "new": 1, "lo": 0, "hi": 0,
         "extra": 0, "cap": 16, "lens": 1}
    c.update(kw)
    if name:
        c["name"] = name
    return c


def listed():
    return [
        # One user's next token, the latency of one layer: norm + RoPE + cache
        # write, attention over 4k tokens, o_proj.
        _case("layer_decode", "layer", seqs=1, lo=4095, hi=4095, cap=128),
        # The batched decode step of a busy server at mixed context lengths.
        _case("decode_batch", "attention", seqs=64, lo=512, hi=32768, cap=512, lens=2),
        # The same server's sliding-window layers: short ranges, many sequences.
        _case("decode_sliding", "attention", seqs=64, lo=512, hi=32768, window=1024, cap=256, lens=3),
        # A larger batch over the quantized cache.
        _case("decode_bq", "attention", kv="bq", seqs=128, lo=1024, hi=65536, cap=2048, lens=5),
        # The full-attention layers with 2 kv heads x 512.
        _case("decode_full_layer", "attention", heads="512", seqs=64, lo=512, hi=32768, cap=512, lens=7),
        # One chunk of one long prompt (an odd number of tokens), as a scheduler
        # that bounds a step's tokens feeds it.
        _case("prefill_chunk", "attention", seqs=1, new=500, lo=7013, hi=7013, lens=11),
        # Eight prompts' chunks at once on prefixes of any length: the largest.
        _case("prefill_batch", "attention", seqs=8, new=2048, lo=0, hi=16384, lens=4),
        # The same chunk width on the sliding layers, quantized cache.
        _case("prefill_sliding_bq", "attention", kv="bq", window=1024, seqs=8, new=2048, lo=0, hi=16384, lens=6),
        # Two prompts at the 512-dim full-attention layers.
        _case("prefill_full_layer", "attention", heads="512", seqs=2, new=1500, lo=1000, hi=8000, lens=12),
        # Continuous batching: 32 sequences decode while one prompt's chunk is
        # prefilled in the same step.
        _case("mixed_step", "attention", seqs=1, new=512, lo=3000, hi=3000, extra=32, lens=13),
        # A whole sliding layer for a fresh 2,000-token prompt.
        _case("layer_prompt", "layer", window=1024, seqs=1, new=2000, lo=0, hi=0, lens=14),
        # Block-sparse decode of a batch at long contexts.
        _case("sparse_decode", "sparse", heads="128", seqs=64, lo=1024, hi=131071, lens=9),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    lens = rng.randrange(1 << 30)
    kind = rng.choice(["layer_decode", "decode", "decode", "chunk", "chunk", "mixed", "layer_prompt", "sparse"])
    if kind == "layer_decode":
        n = _log(rng, 1, 32)
        lo = _log(rng, 64, 8192)
        return _case(None, "layer", seqs=n, lo=lo, hi=lo + rng.randrange(1, 4096), cap=128 if n == 1 else 512,
                     window=rng.choice([0, 1024]), lens=lens)
    if kind == "decode":
        heads, kv, window = rng.choice([("256", "bf16", 0), ("256", "bf16", 1024), ("256", "bq", 0),
                                        ("512", "bf16", 0), ("512", "bq", 0), ("256", "bq", 1024)])
        n = _log(rng, 2, 100)
        lo = _log(rng, 100, 8000)
        cap = 256 if window else 2048 if kv == "bq" else 512
        return _case(None, "attention", heads=heads, kv=kv, window=window, seqs=n, lo=lo,
                     hi=lo + _log(rng, 10, 24000), cap=cap, lens=lens)
    if kind == "chunk":
        heads, kv, window = rng.choice([("256", "bf16", 0), ("256", "bf16", 1024), ("256", "bq", 0),
                                        ("512", "bf16", 0), ("512", "bq", 0), ("256", "bq", 1024)])
        n = rng.choice([1, 1, 1, 2, 4])
        lo = rng.choice([0, _log(rng, 50, 12000)])
        return _case(None, "attention", heads=heads, kv=kv, window=window, seqs=n, new=_log(rng, 17, 2048),
                     lo=lo, hi=lo + rng.randrange(0, 3000), lens=lens)
    if kind == "mixed":
        window = rng.choice([0, 0, 1024])
        lo = _log(rng, 50, 6000)
        return _case(None, "attention", heads=rng.choice(["256", "512"]) if not window else "256", window=window,
                     seqs=1, new=_log(rng, 32, 1024), lo=lo, hi=lo + 100, extra=_log(rng, 4, 64), lens=lens)
    if kind == "layer_prompt":
        heads, window = rng.choice([("256", 1024), ("256", 1024), ("512", 0)])
        return _case(None, "layer", heads=heads, window=window, seqs=rng.choice([1, 2]), new=_log(rng, 17, 3000),
                     lo=0, hi=rng.choice([0, 700]), lens=lens)
    return _case(None, "sparse", heads="128", seqs=_log(rng, 1, 64), lo=_log(rng, 1024, 30000),
                 hi=rng.randrange(30000, 131071), lens=lens)


# ---- the step's sequences -------------------------------------------------------


def _runs(case):
    """(position of the first new token, new tokens) of each sequence, in step order."""
    rng = random.Random(case["lens"])
    runs = [(rng.randint(case["lo"], case["hi"]), 1) for _ in range(case["extra"])]
    runs += [(rng.randint(case["lo"], case["hi"]), case["new"]) for _ in range(case["seqs"])]
    return runs


def _ring(case):
    """Pages of a sequence's ring (a power of two that holds the window and the step)."""
    need = case["window"] + case["new"]
    pages = 1
    while pages * PAGE < need:
        pages *= 2
    return pages


def _table(case, page, seed):
    runs = _runs(case)
    need = [_ring(case) if case["window"] else (p + n + page - 1) // page for p, n in runs]
    pool = sum(need)
    perm = np.random.default_rng(seed).permutation(pool).tolist()
    table, tok, at = KVRunTable(), 0, 0
    for (p, n), k in zip(runs, need):
        table.begin_run(tok, p)
        for x in perm[at:at + k]:
            table.add_base_row(x * page)
        tok, at = tok + n, at + k
    return table, tok, pool * page


def _normal(n, gen, scale=1.0):
    return torch.randn(n, generator=gen, device="cuda", dtype=torch.bfloat16).mul_(scale)


def _codes(n, gen):
    """Codes of rotated N(0, 1) rows: their absmax over a few hundred values is about 3."""
    out = torch.empty(n, dtype=torch.int8, device="cuda")
    for a in range(0, n, 1 << 28):
        b = min(n, a + (1 << 28))
        out[a:b] = torch.randn(b - a, generator=gen, device="cuda", dtype=torch.bfloat16).mul_(127 / 3).round_().clamp_(
            -127, 127).to(torch.int8)
    return out


def prepare(case, seed):
    gen = torch.Generator(device="cuda")
    gen.manual_seed(seed)
    if case["op"] == "sparse":
        return _prepare_sparse(case, seed, gen)
    nq, nkv, d, half, pair = SHAPES[case["heads"]]
    kvs = nkv * d
    table, n, rows = _table(case, PAGE, seed)
    bq = case["kv"] == "bq"
    window = case["window"]
    plan = AttentionPlan(table, n, kind=SLIDING if window else FULL, window=window,
                         cache_size=_ring(case) * PAGE if window else PAGE, page_len=PAGE, cache_rows=rows,
                         cap=case["cap"], kv_row_bytes=kvs * (1 if bq else 2))
    s = {"case": case, "plan": plan, "n": n, "table": table}
    s["partials"], s["stride"] = A.partials_buffer(plan, nq, d)
    s["out"] = torch.empty(n, nq, d, dtype=torch.bfloat16, device="cuda")
    if bq:
        s["k"], s["v"] = _codes(rows * kvs, gen), _codes(rows * kvs, gen)
        s["ks"], s["vs"] = (torch.rand(rows * nkv, generator=gen, device="cuda") * 0.8 + 2.6 for _ in "kv")
        s["q"] = _codes(n * nq * d, gen)
        s["qb"] = s["q"].view(-1, d).sum(1, dtype=torch.int32).mul(128).float()
        s["fq"] = torch.rand(n * nq, generator=gen, device="cuda") * 0.8 + 2.6
        s["o_i8"] = torch.empty(n, nq, d, dtype=torch.int8, device="cuda")
        s["o_sa"] = torch.empty(n, nq, dtype=torch.float32, device="cuda")
        return s
    s["k"], s["v"] = _normal(rows * kvs, gen).view(rows, kvs), _normal(rows * kvs, gen).view(rows, kvs)
    s["q"] = _normal(n * nq * d, gen)
    if case["op"] == "layer":
        s["q_step"] = torch.empty_like(s["q"])
        s["k_src"], s["v_src"] = _normal(n * kvs, gen), _normal(n * kvs, gen)
        s["q_gain"], s["k_gain"] = (_normal(d, gen, 0.1) + 1 for _ in "qk")
        top = max(p + m for p, m in _runs(case))
        inv = 10000.0 ** (-torch.arange(half, device="cuda", dtype=torch.float64) / half)
        ang = torch.arange(top, device="cuda", dtype=torch.float64)[:, None] * inv
        s["cos"], s["sin"] = ang.cos().float().contiguous(), ang.sin().float().contiguous()
        s["w"] = _normal(HIDDEN * nq * d, gen, 1 / math.sqrt(nq * d)).view(HIDDEN, nq * d)
        s["proj"] = torch.empty(n, HIDDEN, dtype=torch.bfloat16, device="cuda")
        s["ws"] = A.gemm_cols_workspace(HIDDEN, nq * d, n)
    return s


def _prepare_sparse(case, seed, gen):
    table, n, rows = _table(case, S_BLOCK, seed)
    plan = AttentionPlan(table, n, kind=FULL, window=0, cache_size=S_BLOCK, page_len=S_BLOCK, cache_rows=rows,
                         cap=16, kv_row_bytes=S_NKV * S_D * 2)
    return {"case": case, "plan": plan, "n": n, "table": table,
            "index_k": _normal(rows * S_D, gen).view(rows, S_D),
            "index_q": _normal(n * S_IH * S_D, gen),
            "k": _normal(rows * S_NKV * S_D, gen).view(rows, -1),
            "v": _normal(rows * S_NKV * S_D, gen).view(rows, -1),
            "q": _normal(n * S_NQ * S_D, gen, 1 / math.sqrt(S_D)),
            "scores": A.index_scores_buffer(plan, S_IH, S_BLOCK),
            "idx": torch.empty(n, S_IH, S_TOPK, dtype=torch.int32, device="cuda"),
            "out": torch.empty(n, S_NQ, S_D, dtype=torch.bfloat16, device="cuda")}


def run(s):
    case, plan = s["case"], s["plan"]
    if case["op"] == "sparse":
        A.dispatch_lightning_indexer(plan, s["index_q"], s["index_k"], s["idx"], s["scores"])
        A.dispatch_block_sparse_attention(plan, s["q"], s["k"], s["v"], s["idx"], s["out"])
        return {"blocks": s["idx"], "out": s["out"]}
    nq, nkv, d, half, pair = SHAPES[case["heads"]]
    kvs = nkv * d
    if case["kv"] == "bq":
        A.bq_attention(plan, s["q"], s["qb"], s["fq"], s["k"], s["ks"], s["v"], s["vs"], s["out"], s["partials"],
                       s["stride"], num_q=nq, num_kv=nkv, head_dim=d, kv_stride=kvs, o_i8=s["o_i8"], o_sa=s["o_sa"])
        return {"out": s["out"], "codes": s["o_i8"], "scales": s["o_sa"]}
    if case["op"] == "attention":
        A.attention_bf16(plan, s["q"], s["k"], s["v"], s["out"], s["partials"], s["stride"], num_q=nq, num_kv=nkv,
                         head_dim=d, kv_stride=kvs)
        return {"out": s["out"]}
    # The append rotates q in place: a fresh q, as the projection before it writes one.
    q = s["q_step"].copy_(s["q"])
    A.dispatch_rms_norm_rope_cache_write(plan, q, s["k_src"], s["v_src"], s["k"], s["v"], s["q_gain"], s["k_gain"],
                                         s["cos"], s["sin"], num_q=nq, num_kv=nkv, half=half, pair_stride=pair,
                                         head_dim=d, sqrt_n=math.sqrt(d), n_eps=d * 1e-6)
    A.attention_bf16(plan, q, s["k"], s["v"], s["out"], s["partials"], s["stride"], num_q=nq, num_kv=nkv,
                     head_dim=d, kv_stride=kvs)
    A.dispatch_gemm_cols(s["out"], s["w"], s["proj"], rows=HIDDEN, cols=nq * d, seq_len=s["n"], workspace=s["ws"])
    return {"q": q, "k": s["k"], "v": s["v"], "out": s["out"], "proj": s["proj"]}


# ---- what a pass cannot do without ----------------------------------------------


def work(case):
    runs = _runs(case)
    n = sum(m for _, m in runs)
    if case["op"] == "sparse":
        kept = sum(min(S_TOPK * S_BLOCK, p + 1) for p, _ in runs)
        by = sum(p + 1 for p, _ in runs) * S_D * 2 + n * (S_IH + 2 * S_NQ) * S_D * 2 + kept * S_NKV * S_D * 4 + n * S_IH * S_TOPK * 4
        fl = sum(p + 1 for p, _ in runs) * 2 * S_IH * S_D + kept * 4 * S_NQ * S_D
        return {"bytes": by, "flops": fl}
    nq, nkv, d, half, _ = SHAPES[case["heads"]]
    kvs, w = nkv * d, case["window"]
    keys = pairs = 0
    for p, m in runs:
        keys += min(p + m, w + m - 1) if w else p + m
        if w:
            pairs += sum(min(t + 1, w) for t in range(p, p + m))
        else:
            pairs += m * p + m * (m + 1) // 2
    fl = 4 * d * nq * pairs
    if case["kv"] == "bq":
        return {"bytes": keys * (2 * kvs + 8 * nkv) + n * nq * (4 * d + 12), "flops": fl}
    if case["op"] == "attention":
        return {"bytes": keys * 4 * kvs + n * nq * d * 4, "flops": fl}
    # q, k and v in; q, the two cache rows, the attention and the projection out; the older keys; the weight
    by = n * (6 * nq * d + 8 * kvs + 2 * HIDDEN) + (keys - n if not w else max(0, keys - n)) * 4 * kvs + HIDDEN * nq * d * 2
    return {"bytes": by, "flops": fl + 2 * n * HIDDEN * nq * d}


def tolerance(case):
    # Outputs are bf16 (0.0015 from the 64-bit result, as their rounding gives):
    # another order of the f32 sums moves some of them to the neighbouring bf16
    # value, 2^-8 of the value, and a weight at a step of the biased exponential
    # by 0.7 %.  The int8 codes of those outputs move with them; block numbers
    # do not.
    tol = {"rel": 0.006, "max": 0.08, "differ": 0.0}
    if case["kv"] == "bq":
        tol["differ"] = 0.005
    return tol


# ---- the same in 64 bits ---------------------------------------------------------
# The attention that this library computes is a walk over tiles of 16 keys from
# each range's first key.  m is the running maximum after a tile, a key's weight
# fexp(score - m), and every tile scales what came before by fexp(m_old - m);
# fexp is a biased exponential (fexp(0) is not 1), so the walk is part of the
# result.  Ranges of one token that were split are joined by fexp(m_i - max m).

_EXP_A, _EXP_BIAS = 12102203.16156148, 1059208216.0
_EXP_P = (1.6501418352127075, -0.37554836273193359, 0.38696467876434326)


def _fexp(x):
    t = (float(np.float32(_EXP_A)) * x + _EXP_BIAS).clamp_min_(0.0) / 8388608.0
    e = t.floor()
    f = t - e
    return torch.exp2(e - 127.0) * (1.0 + f) * (_EXP_P[0] + f * (_EXP_P[1] + f * _EXP_P[2])) * (t > 0)


def _walk(s, live):
    """Weights [rows, keys] of the walk over scores s [rows, keys] from the first column, the keys with
    live[rows, keys] counted, and the last running maximum [rows]."""
    r, n = s.shape
    pad = -n % 16
    if pad:
        s = torch.nn.functional.pad(s, (0, pad))
        live = torch.nn.functional.pad(live, (0, pad))
    s = torch.where(live, s, torch.full_like(s, -1e30)).view(r, -1, 16)
    m = s.amax(2).cummax(1).values
    before = torch.cat([torch.full_like(m[:, :1], -1e30), m[:, :-1]], 1)
    corr = _fexp((before - m).clamp_min(-87.0))
    corr = torch.where(live.view(r, -1, 16).any(2), corr, torch.ones_like(corr))
    after = torch.cat([corr[:, 1:], torch.ones_like(corr[:, :1])], 1).flip(1).cumprod(1).flip(1)
    w = _fexp((s - m[:, :, None]).clamp_min(-87.0)) * after[:, :, None]
    w = torch.where(live.view(r, -1, 16), w, torch.zeros_like(w))
    return w.view(r, -1)[:, :n], m[:, -1]


def _splits(lens, cap, row_bytes):
    """The ranges [(a, b), ...] that a decode step's plan cuts each sequence's keys into."""
    def cut(n, k):
        per = -(-n // k)
        return [(min(i * per, n), min((i + 1) * per, n)) for i in range(k)]

    if len(lens) == 1:
        nbytes, k = lens[0] * row_bytes, cap
        if cap > 1 and nbytes < 1 << 20:
            k = 1
            while (k + 1) ** 2 <= nbytes // 2280 and k < cap:
                k += 1
        return [cut(lens[0], min(k, cap, lens[0]))]
    count, left = [1] * len(lens), cap - len(lens)
    while left > 0:
        best = None
        for i, n in enumerate(lens):
            if count[i] < -(-n // 16) and (best is None or n * count[best] > lens[best] * count[i]):
                best = i
        if best is None:
            break
        count[best] += 1
        left -= 1
    return [cut(n, k) for n, k in zip(lens, count)]


def _bf16(x):
    return x.to(torch.bfloat16).double()


def _slots(s, run, first, last, page):
    case, t = s["case"], s["table"]
    _, _, off, count = t.runs[run]
    rows = torch.tensor(t.base_rows[off:off + count], device="cuda", dtype=torch.int64)
    p = torch.arange(first, last, device="cuda")
    at = p // page
    return rows[at % count if case["window"] else at] + p % page


def _attend(s, q, k_rows, v_rows, score, nq, nkv, d):
    """Attention of the step in 64 bits, [n, nq, d].  k_rows(slots, head) and v_rows(...) give the 64-bit
    rows of a kv head, score(tokens, head, slots, raw) what a raw dot product counts."""
    case = s["case"]
    gqa, w = nq // nkv, case["window"]
    runs = _runs(case)
    out = torch.zeros(s["n"], nq, d, dtype=torch.float64, device="cuda")
    decode = all(m == 1 for _, m in runs) and (len(runs) == 1 or len(runs) < case["cap"])
    if decode:
        width = nkv * d * (1 if case["kv"] == "bq" else 2)
        lens = [min(p + 1, w) if w else p + 1 for p, _ in runs]
        parts = _splits(lens, case["cap"], width)
        for i, (p, _) in enumerate(runs):
            slots = _slots(s, i, p + 1 - lens[i], p + 1, PAGE)
            for g in range(nkv):
                k, v = k_rows(slots, g), v_rows(slots, g)
                raw = q[i, g * gqa:(g + 1) * gqa] @ k.T
                sc = score(torch.tensor([i], device="cuda"), g, slots, raw)
                acc, ls, ms = [], [], []
                for a, b in parts[i]:
                    if a >= b:
                        continue
                    wt, m = _walk(sc[:, a:b], torch.ones_like(sc[:, a:b], dtype=torch.bool))
                    acc.append(wt @ v[a:b])
                    ls.append(wt.sum(1))
                    ms.append(m)
                m = torch.stack(ms)
                c = _fexp((m - m.amax(0)).clamp_min(-87.0))
                o = (torch.stack(acc) * c[:, :, None]).sum(0) / (torch.stack(ls) * c).sum(0)[:, None]
                out[i, g * gqa:(g + 1) * gqa] = o
        return out
    t0 = 0
    for i, (p0, m) in enumerate(runs):
        for a in range(0, m, 256):
            b = min(m, a + 256)
            first = max(0, p0 + a - w + 1) if w else 0
            slots = _slots(s, i, first, p0 + b, PAGE)
            pos = torch.arange(p0 + a, p0 + b, device="cuda").repeat_interleave(gqa)
            tok = torch.arange(t0 + a, t0 + b, device="cuda")
            lo = (pos - w + 1).clamp_min(0) - first if w else torch.zeros_like(pos)
            # columns of a row: keys from the row's own first key
            cols = min(w, slots.numel()) if w else slots.numel()
            at = lo[:, None] + torch.arange(cols, device="cuda")
            live = at <= (pos - first)[:, None]
            at = at.clamp_max(slots.numel() - 1)
            for g in range(nkv):
                k, v = k_rows(slots, g), v_rows(slots, g)
                raw = q[t0 + a:t0 + b, g * gqa:(g + 1) * gqa].reshape(-1, d) @ k.T
                sc = score(tok, g, slots, raw)
                wt, _ = _walk(sc.gather(1, at) if w else sc, live)
                if w:
                    wt = torch.zeros_like(sc).scatter_add_(1, at, wt)
                o = (wt @ v) / wt.sum(1, keepdim=True)
                out[t0 + a:t0 + b, g * gqa:(g + 1) * gqa] = o.view(b - a, gqa, d)
        t0 += m
    return out


def exact(case, seed):
    s = prepare(case, seed)
    if case["op"] == "sparse":
        return _exact_sparse(s)
    nq, nkv, d, half, pair = SHAPES[case["heads"]]
    n = s["n"]
    if case["kv"] == "bq":
        k, v = s["k"].view(-1, nkv, d), s["v"].view(-1, nkv, d)
        ks, vs = s["ks"].view(-1, nkv).double(), s["vs"].view(-1, nkv).double()
        fq, off = s["fq"].view(n, nq).double(), s["q"].view(n, nq, d).double().sum(2) * 128 - s["qb"].view(n, nq).double()
        gqa = nq // nkv

        def score(tok, g, slots, raw):
            f, o = (x[tok, g * gqa:(g + 1) * gqa].reshape(-1, 1) for x in (fq, off))
            return (raw + o) * f * ks[slots, g] / 127.0 ** 2

        out = _attend(s, s["q"].view(n, nq, d).double(), lambda sl, g: k[sl, g].double(),
                      lambda sl, g: v[sl, g].double() * vs[sl, g][:, None] / 127.0, score, nq, nkv, d)
        return {"out": out, "codes": None, "scales": out.abs().amax(2)}
    q = s["q"].view(n, nq, d).double()
    k, v = s["k"].view(-1, nkv, d), s["v"].view(-1, nkv, d)
    res = {}
    if case["op"] == "layer":
        runs = _runs(case)
        pos = torch.cat([torch.arange(p, p + m, device="cuda") for p, m in runs])
        slots = torch.cat([_slots(s, i, p, p + m, PAGE) for i, (p, m) in enumerate(runs)])
        cos, sin = s["cos"][pos].double()[:, None], s["sin"][pos].double()[:, None]

        def norm(x, gain):
            x = x * (math.sqrt(d) / (x.square().sum(2, keepdim=True) + d * 1e-6).sqrt())
            return _bf16(x * gain.double() if gain is not None else x)

        def rope(x):
            a, b = x[..., :half], x[..., pair:pair + half]
            y = x.clone()
            y[..., :half], y[..., pair:pair + half] = a * cos - b * sin, b * cos + a * sin
            return _bf16(y)

        q = rope(norm(q, s["q_gain"]))
        k, v = k.double(), v.double()
        k[slots] = rope(norm(s["k_src"].view(n, nkv, d).double(), s["k_gain"]))
        v[slots] = norm(s["v_src"].view(n, nkv, d).double(), None)
        res = {"q": q.flatten(), "k": k.view(-1, nkv * d), "v": v.view(-1, nkv * d)}
    out = _attend(s, q, lambda sl, g: k[sl, g].double(), lambda sl, g: v[sl, g].double(),
                  lambda tok, g, sl, raw: raw, nq, nkv, d)
    res["out"] = out
    if case["op"] == "layer":
        res["proj"] = _bf16(out).view(n, nq * d) @ s["w"].double().T
    return res


def _exact_sparse(s):
    case = s["case"]
    n = s["n"]
    iq = s["index_q"].view(n, S_IH, S_D).double()
    q = s["q"].view(n, S_NQ, S_D).double()
    k, v = s["k"].view(-1, S_NKV, S_D), s["v"].view(-1, S_NKV, S_D)
    gqa = S_NQ // S_NKV
    out = torch.zeros(n, S_NQ, S_D, dtype=torch.float64, device="cuda")
    for i, (p, _) in enumerate(_runs(case)):
        slots = _slots(s, i, 0, p + 1, S_BLOCK)
        sc = iq[i] @ s["index_k"][slots].double().T
        blocks = p // S_BLOCK + 1
        sc = torch.nn.functional.pad(sc, (0, blocks * S_BLOCK - p - 1), value=-1e300).view(S_IH, blocks, S_BLOCK).amax(2)
        sc[:, -1] = 1e300  # the block that holds the token is always kept
        top = sc.topk(min(S_TOPK, blocks), 1).indices.sort(1).values
        for g in range(S_NKV):
            p_at = (top[g][:, None] * S_BLOCK + torch.arange(S_BLOCK, device="cuda")).flatten()
            p_at = p_at[p_at <= p]
            sl = slots[p_at]
            w, _ = _walk(q[i, g * gqa:(g + 1) * gqa] @ k[sl, g].double().T,
                         torch.ones(gqa, p_at.numel(), dtype=torch.bool, device="cuda"))
            out[i, g * gqa:(g + 1) * gqa] = (w @ v[sl, g].double()) / w.sum(1, keepdim=True)
    return {"blocks": None, "out": out}

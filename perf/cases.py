"""The work that users of this package have it do, as cases that can be timed and compared.

Every case goes through public entry points and stands for one call site of a serving engine:

* ``layer``   one decode layer's attention: the paged KV append and the mixed draft/verify attention;
* ``refresh`` a refresh layer: full attention with page scores (or the first/last logits dump) and the
              page selection from them;
* ``prefill`` one layer of prompt chunks: the append of the chunk and the paged prefill attention;
* ``rope``    one layer's q/k RMSNorm, rotary permute, RoPE and K/V append of a token batch;
* ``sample``  token picks from logits: top-k candidates, temperature + softmax + top-p, one draw a row;
* ``verify``  speculative verification: the target's candidates from its logits, then the chain rule;
* ``step``    a whole decode step of a Qwen3-shape model, planned on the host and replayed as a HIP graph.

``rows_seed`` fixes a case's row lengths; values, page orders and selections come from the seed that
``prepare`` gets. Sizes are the benchmark's and the tests' (16-token pages, head_dim 128, bf16).
"""

from __future__ import annotations

import math

import numpy as np
import torch

from aspire_amd.attention import kv_ops  # noqa: F401  (registers mylib::update_kv_padded)
from aspire_amd.attention.holistic_wrapper import HolisticAttentionWrapper, build_holistic_dump_jit_args
from aspire_amd.attention.prefill import BatchPrefillWithPagedKVCacheWrapper
from aspire_amd.attention.rope import RopeConfig, qk_norm_rope_update_kv
from aspire_amd.backends.page_selector import KeyMeanPageSelector, PageSelectorFirstLastAvg
from aspire_amd.decode_step import DecodeWeights, MixedDecodeStep, ModelShape, alloc_kv_caches
from aspire_amd.engine.sampling import local_topk_candidates, verify_topk_speculation
from aspire_amd.logits_processor import build_logits_pipe
from aspire_amd.sampling import sampling_from_probs

PAGE, D, VOCAB = 16, 128, 151936
EPS, THETA = 1e-6, 1e6
LOG2E = 1.4426950408889634


# ------------------------------------------------------------------------------- the cases
def listed():
    return [
        # the smallest attention call: a 16/8-head layer, 4 rows of 4096 tokens, two drafting over 64
        # selected pages, two verifying 5 tokens; launches and host work count here
        {"name": "layer_small", "kind": "layer", "hq": 16, "hkv": 8, "batch": 4, "lo": 4096, "hi": 4096, "draft": 0.5,
         "q_lo": 5, "q_hi": 5, "budget": 64, "rows_seed": 0},
        # the ordinary mixed layer of the benchmark: 32 rows of 32768 tokens, half drafting over 128 pages
        {"name": "layer_mixed", "kind": "layer", "hq": 32, "hkv": 8, "batch": 32, "lo": 32768, "hi": 32768,
         "draft": 0.5, "q_lo": 4, "q_hi": 4, "budget": 128, "rows_seed": 0},
        # long contexts, ragged lengths and verify lengths (1, 2 and 3 row tiles in one launch)
        {"name": "layer_long", "kind": "layer", "hq": 32, "hkv": 8, "batch": 16, "lo": 65536, "hi": 131072,
         "draft": 0.5, "q_lo": 2, "q_hi": 9, "budget": 256, "rows_seed": 4000},
        # a refresh layer of drafting rows: full attention, per-head key-mean page scores, top-128 pages
        {"name": "refresh_keymean", "kind": "refresh", "selector": "keymean", "hq": 32, "hkv": 8, "batch": 64,
         "lo": 8192, "hi": 32768, "draft": 1.0, "q_lo": 2, "q_hi": 9, "budget": 128, "rows_seed": 1000},
        # a refresh layer with the first/last logits dump of a mixed batch and the selection over it
        {"name": "refresh_first_last", "kind": "refresh", "selector": "first_last", "hq": 32, "hkv": 8, "batch": 64,
         "lo": 8192, "hi": 32768, "draft": 0.5, "q_lo": 2, "q_hi": 9, "budget": 128, "rows_seed": 3000},
        # the largest prompt chunk an engine sends in one call
        {"name": "prefill_chunk", "kind": "prefill", "hq": 32, "hkv": 8, "rows": 1, "t_lo": 8192, "t_hi": 8192,
         "p_lo": 0, "p_hi": 0, "rows_seed": 0},
        # last chunks of several prompts: odd lengths over cached prefixes of odd lengths
        {"name": "prefill_ragged", "kind": "prefill", "hq": 32, "hkv": 8, "rows": 5, "t_lo": 17, "t_hi": 700,
         "p_lo": 300, "p_hi": 8192, "rows_seed": 1},
        # q/k preparation and append of a prompt chunk's tokens (decode-sized calls are in the steps)
        {"name": "rope_chunk", "kind": "rope", "hq": 32, "hkv": 8, "rows": 3, "tokens": 8192, "prefix": 5000,
         "rows_seed": 2},
        # token picks of a decode step of 64 requests: 208 rows of a 151936-entry vocabulary
        {"name": "sample_step", "kind": "sample", "rows": 208, "top_k": 50, "temperature": 0.8, "top_p": 0.9},
        # speculative verification of a small batch: 4 requests, 5 drafts each
        {"name": "verify_small", "kind": "verify", "requests": 4, "drafts": 5, "top_k": 50, "temperature": 0.8,
         "top_p": 0.9},
        # a small model's whole decode step, as latency-bound as serving gets
        {"name": "step_small", "kind": "step", "selector": "first_last", "layers": 8, "dim": 2048, "hq": 16, "hkv": 8,
         "inter": 6144, "batch": 4, "lo": 4096, "hi": 4096, "draft": 0.5, "q_lo": 5, "q_hi": 5, "budget": 64,
         "rows_seed": 0},
        # the benchmark's decode step (8 of its layers): 64 rows, 208 tokens, per-head draft lists
        {"name": "step_large", "kind": "step", "selector": "keymean", "layers": 8, "dim": 4096, "hq": 32, "hkv": 8,
         "inter": 12288, "batch": 64, "lo": 8192, "hi": 32768, "draft": 0.5, "q_lo": 2, "q_hi": 9, "budget": 128,
         "rows_seed": 3000},
    ]


HEADS = [(32, 8), (32, 8), (32, 8), (16, 8), (8, 8), (64, 8), (16, 4), (16, 2)]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["layer", "layer", "layer", "refresh", "prefill", "prefill", "rope", "sample", "verify", "step"])
    seed = rng.randrange(1 << 20)
    if kind in ("layer", "refresh"):
        hq, hkv = rng.choice(HEADS)
        most = max(2, min(9, 48 // (hq // hkv)))
        q_lo = rng.randint(2, most)
        hi = _log(rng, 300, 131072)
        batch = max(1, min(_log(rng, 1, 64), 1600000 // hi))
        c = {"kind": kind, "hq": hq, "hkv": hkv, "batch": batch, "lo": max(64, hi // rng.choice([1, 2, 4])), "hi": hi,
             "draft": rng.choice([0.0, 0.25, 0.5, 0.75, 1.0]), "q_lo": q_lo, "q_hi": rng.randint(q_lo, most),
             "budget": rng.randint(16, 256), "rows_seed": seed}
        if kind == "refresh":
            c["selector"] = rng.choice(["keymean", "first_last"])
            if c["selector"] == "first_last":   # the dump is of one engine's maximum length
                c["hi"] = min(c["hi"], 32768)
                c["lo"] = min(c["lo"], c["hi"])
        return c
    if kind == "prefill":
        hq, hkv = rng.choice([(32, 8), (32, 8), (16, 8), (8, 8), (64, 8), (64, 2)])
        rows = rng.randint(1, 8)
        t_hi = _log(rng, 16, 8192 // rows)
        p_hi = rng.choice([0, _log(rng, 16, 32768)])
        return {"kind": kind, "hq": hq, "hkv": hkv, "rows": rows, "t_lo": max(1, t_hi // rng.choice([1, 3])),
                "t_hi": t_hi, "p_lo": p_hi // rng.choice([1, 4]), "p_hi": p_hi, "rows_seed": seed}
    if kind == "rope":
        hq, hkv = rng.choice(HEADS)
        rows = rng.randint(1, 64)
        return {"kind": kind, "hq": hq, "hkv": hkv, "rows": rows, "tokens": max(rows, _log(rng, 1, 8192)),
                "prefix": _log(rng, 16, 16384), "rows_seed": seed}
    if kind == "sample":
        return {"kind": kind, "rows": _log(rng, 1, 256), "top_k": rng.choice([20, 50, 64, 100, 1024]),
                "temperature": round(rng.uniform(0.5, 1.3), 3), "top_p": round(rng.uniform(0.5, 0.99), 3)}
    if kind == "verify":
        return {"kind": kind, "requests": _log(rng, 1, 32), "drafts": rng.randint(1, 8),
                "top_k": rng.choice([20, 50, 64]), "temperature": round(rng.uniform(0.5, 1.3), 3),
                "top_p": round(rng.uniform(0.5, 0.99), 3)}
    dim, hq, hkv, inter = rng.choice([(2048, 16, 8, 6144), (4096, 32, 8, 12288)])
    hi = _log(rng, 1024, 32768)
    q_lo = rng.randint(2, 9)
    return {"kind": "step", "selector": rng.choice(["keymean", "first_last"]), "layers": rng.randint(3, 6), "dim": dim,
            "hq": hq, "hkv": hkv, "inter": inter, "batch": max(4, min(_log(rng, 4, 64), 1200000 // hi)),
            "lo": max(256, hi // rng.choice([1, 2, 4])), "hi": hi, "draft": rng.choice([0.25, 0.5, 0.75]),
            "q_lo": q_lo, "q_hi": rng.randint(q_lo, 9), "budget": rng.randint(64, 256), "rows_seed": seed}


# ------------------------------------------------------------------- what a case's rows look like
def _decode_rows(c):
    """(context after the append, new tokens, drafting) of each row, from the case alone."""
    r = np.random.default_rng(c["rows_seed"])
    ctx = r.integers(c["lo"], c["hi"] + 1, size=c["batch"]).astype(np.int64)
    dr = np.zeros(c["batch"], dtype=bool)
    dr[r.permutation(c["batch"])[: int(round(c["draft"] * c["batch"]))]] = True
    ql = np.where(dr, 1, r.integers(c["q_lo"], c["q_hi"] + 1, size=c["batch"])).astype(np.int64)
    return ctx, ql, dr


def _chunk_rows(c):
    """(length after the append, new tokens) of each row of a token batch."""
    r = np.random.default_rng(c["rows_seed"])
    if c["kind"] == "rope":
        cuts = np.sort(r.choice(np.arange(1, c["tokens"]), size=c["rows"] - 1, replace=False)) \
            if c["rows"] > 1 else np.zeros(0, np.int64)
        t = np.diff(np.concatenate([[0], cuts, [c["tokens"]]])).astype(np.int64)
        p = r.integers(0, c["prefix"] + 1, size=c["rows"]).astype(np.int64)
    else:
        t = r.integers(c["t_lo"], c["t_hi"] + 1, size=c["rows"]).astype(np.int64)
        p = r.integers(c["p_lo"], c["p_hi"] + 1, size=c["rows"]).astype(np.int64)
    return p + t, t


def _pages(n):
    return (np.asarray(n, dtype=np.int64) + PAGE - 1) // PAGE


def _ptr(n):
    return np.concatenate([[0], np.cumsum(n)]).astype(np.int32)


def _table(n_pages, seed):
    """[B, W] logical -> physical pages: a random order of a pool of just these pages."""
    perm = np.random.default_rng(seed + 77).permutation(int(n_pages.sum())).astype(np.int32)
    table = np.zeros((len(n_pages), int(n_pages.max())), dtype=np.int32)
    at = _ptr(n_pages)
    for b, n in enumerate(n_pages):
        table[b, :n] = perm[at[b]: at[b] + n]
    return table


def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(seed)


def _normal(shape, gen, std=1.0, mean=0.0):
    return torch.empty(shape, dtype=torch.bfloat16, device="cuda").normal_(mean, std, generator=gen)


def _cache(pool, hkv, gen):
    """Keys and values N(0, 1); every (page, kv head) shifts its keys by one scalar, so pages differ."""
    cache = _normal((pool, 2, PAGE, hkv, D), gen)
    cache[:, 0] += _normal((pool, 1, hkv, 1), gen, 0.5)
    return cache


def _dev(a, dtype=torch.int32):
    return torch.from_numpy(np.ascontiguousarray(a)).to("cuda", dtype)


def _decode_inputs(c, seed, whole):
    """A decode layer's inputs; ``whole``: every row reads all its pages (a refresh layer)."""
    ctx, ql, dr = _decode_rows(c)
    n_pages = _pages(ctx)
    table = _table(n_pages, seed)
    r = np.random.default_rng(seed)
    lists = []
    for b in range(c["batch"]):
        n = int(n_pages[b])
        if dr[b] and not whole:  # a selection that ends with the current page, in logical order
            k = min(c["budget"], n)
            lists.append(table[b, np.sort(np.concatenate([r.choice(n - 1, k - 1, replace=False), [n - 1]]))
                               if k > 1 else np.array([n - 1])])
        else:
            lists.append(table[b, :n])
    counts = np.array([len(x) for x in lists])
    gen, T = _gen(seed), int(ql.sum())
    return dict(ctx=ctx, ql=ql, dr=dr, n_pages=n_pages, table=table, lists=lists, counts=counts,
                last=(ctx - 1) % PAGE + 1, cache=_cache(int(n_pages.sum()), c["hkv"], gen),
                q=_normal((T, c["hq"], D), gen), k=_normal((T, c["hkv"], D), gen), v=_normal((T, c["hkv"], D), gen))


def _chunk_inputs(c, seed):
    ctx, t = _chunk_rows(c)
    n_pages = _pages(ctx)
    table = _table(n_pages, seed)
    gen, T = _gen(seed), int(t.sum())
    d = dict(ctx=ctx, ql=t, n_pages=n_pages, counts=n_pages, lists=[table[b, :n] for b, n in enumerate(n_pages)],
             last=(ctx - 1) % PAGE + 1, cache=_cache(int(n_pages.sum()), c["hkv"], gen))
    if c["kind"] == "rope":  # one projection's output, [q | k | v] a row
        qkv = _normal((T, (c["hq"] + 2 * c["hkv"]) * D), gen)
        a, b = c["hq"] * D, (c["hq"] + c["hkv"]) * D
        d.update(q=qkv[:, :a].view(T, c["hq"], D), k=qkv[:, a:b].view(T, c["hkv"], D),
                 v=qkv[:, b:].view(T, c["hkv"], D), qw=_normal(D, gen, 0.1, 1.0), kw=_normal(D, gen, 0.1, 1.0))
    else:
        d.update(q=_normal((T, c["hq"], D), gen), k=_normal((T, c["hkv"], D), gen), v=_normal((T, c["hkv"], D), gen))
    return d


def _index(d):
    """The device index arrays of a set of rows."""
    return dict(qo=_dev(_ptr(d["ql"])), kvp=_dev(_ptr(d["counts"])), idx=_dev(np.concatenate(d["lists"])),
                lpl=_dev(d["last"]))


def _logits(rows, seed):
    """Next-token logits: a broad normal body with a peaked head, as a language model's are."""
    gen = _gen(seed)
    x = torch.empty(rows, VOCAB, dtype=torch.float32, device="cuda").normal_(0.0, 2.0, generator=gen)
    top = torch.randint(0, VOCAB, (rows, 40), device="cuda", generator=gen)
    x.scatter_add_(1, top, torch.empty(rows, 40, device="cuda").exponential_(0.25, generator=gen))
    return x.to(torch.bfloat16), gen


def _verify_inputs(c, seed):
    R, n, K = c["requests"], c["drafts"], c["top_k"]
    logits, gen = _logits(R * (n + 1), seed)
    # the draft's candidates: the target's, with its logits moved a little (a draft that reads fewer pages)
    near = logits.view(R, n + 1, VOCAB)[:, :n].float()
    near = near + 0.5 * torch.empty(near.shape, device="cuda").normal_(generator=gen)
    val, ids = torch.topk(near, K, dim=-1)
    probs = torch.softmax(val / c["temperature"], dim=-1)
    pick = torch.multinomial(probs.view(-1, K), 1, generator=gen).view(R, n, 1)
    return dict(logits=logits.view(R, n + 1, VOCAB), draft_probs=probs, draft_ids=ids,
                draft_tokens=torch.gather(ids, 2, pick)[..., 0].to(torch.int32),
                counts=torch.randint(max(1, n - 2), n + 1, (R,), device="cuda", generator=gen, dtype=torch.int32),
                u=torch.rand(R, n + 1, device="cuda", generator=gen))


def _shape(c):
    return ModelShape(n_layer=c["layers"], dim=c["dim"], n_head=c["hq"], n_local_heads=c["hkv"],
                      intermediate_size=c["inter"], vocab_size=VOCAB, rope_base=THETA, norm_eps=EPS)


REFRESH_LAYER = 2


def _recent(selector):
    return 8 if selector == "first_last" else 1


# ---------------------------------------------------------------------------------- prepare, run
def prepare(case, seed):
    c, kind = case, case["kind"]
    if kind == "sample":
        logits, gen = _logits(c["rows"], seed)
        pipe, kw = build_logits_pipe(c["temperature"], c["top_p"])
        return dict(case=c, logits=logits, pipe=pipe, kw=kw, u=torch.rand(c["rows"], device="cuda", generator=gen))
    if kind == "verify":
        pipe, kw = build_logits_pipe(c["temperature"], c["top_p"])
        return dict(_verify_inputs(c, seed), case=c, pipe=pipe, kw=kw)
    if kind == "step":
        return _prepare_step(c, seed)
    d = _chunk_inputs(c, seed) if kind in ("prefill", "rope") else _decode_inputs(c, seed, kind == "refresh")
    d.update(_index(d), case=c)
    if kind == "rope":
        d.update(offsets=_dev(d["ctx"] - d["ql"]), rope=RopeConfig(rope_theta=THETA))
        return d
    d["out"] = torch.empty_like(d["q"])
    ws = torch.empty(1, device="cuda")
    if kind == "prefill":
        w = BatchPrefillWithPagedKVCacheWrapper(ws, "NHD")
    elif kind == "refresh" and c["selector"] == "first_last":
        w = HolisticAttentionWrapper(ws, "NHD", jit_args=build_holistic_dump_jit_args(
            torch.bfloat16, D, dump_kind="first_last_compact", dump_buffer_dtype=torch.float16))
    else:
        w = HolisticAttentionWrapper(ws, "NHD")
    w.plan(d["qo"], d["kvp"], d["idx"], d["lpl"], c["hq"], c["hkv"], D, PAGE, causal=True)
    d["wrapper"] = w
    if kind == "refresh":
        B, W = c["batch"], d["table"].shape[1]
        d.update(npg=_dev(d["n_pages"]), tab=_dev(d["table"]), stride=W * PAGE)
        if c["selector"] == "keymean":
            d["sel"] = KeyMeanPageSelector(B, c["hkv"], W, c["budget"], L=1, device="cuda")
            d["sel"].page_scores.zero_()
        else:
            d["dump"] = torch.full((B * c["hq"] * 2 * W * PAGE,), float("-inf"), dtype=torch.float16, device="cuda")
            d["sel"] = PageSelectorFirstLastAvg(
                max_batch_size=B, pages_per_slot=W, subset_cache_size=min(c["budget"], W), L=8, n_heads=c["hq"],
                page_size=PAGE, max_seq_length=W * PAGE, device="cuda", bsz=B, dec_len=int(d["ql"].max()), head_dim=D,
                kv_stride=W * PAGE)
    return d


def _prepare_step(c, seed):
    """The model, its caches and one captured step, after one eager step (as an engine warms up)."""
    ctx, ql, dr = _decode_rows(c)
    n_pages = _pages(ctx)
    shape = _shape(c)
    weights = DecodeWeights(shape, "cuda", seed=seed)
    caches = alloc_kv_caches(shape, int(n_pages.sum()), "cuda", seed=seed)
    step = MixedDecodeStep(weights, caches, ctx, ql, dr, torch.from_numpy(_table(n_pages, seed)), budget=c["budget"],
                           refresh_layer=REFRESH_LAYER, selector=c["selector"], seed=seed)
    step.forward()
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        step.forward()
    return dict(case=c, step=step, graph=graph)


def run(state):
    s, c = state, state["case"]
    kind = c["kind"]
    if kind == "step":
        step = s["step"]
        step.plan()
        s["graph"].replay()
        # the logits the ids are picked from, and what the next step selects its pages by
        return {"logits": step.logits, "scores": step.dump if c["selector"] == "first_last" else step.selector.page_scores}
    if kind == "sample":
        values, ids = local_topk_candidates(s["logits"], c["top_k"])
        probs = s["pipe"](values, **s["kw"])
        return {"values": values, "ids": ids, "probs": probs, "pick": sampling_from_probs(probs, uniforms=s["u"])}
    if kind == "verify":
        values, ids = local_topk_candidates(s["logits"], c["top_k"])
        probs = s["pipe"](values, **s["kw"])
        output, emitted = verify_topk_speculation(s["draft_probs"], s["draft_ids"], s["draft_tokens"], s["counts"],
                                                  probs, ids, uniforms=s["u"])
        return {"values": values, "ids": ids, "probs": probs, "output": output, "emitted": emitted}
    if kind == "rope":
        # q is rewritten in place, as the package does it: a repeated pass prepares the last one's q again
        qk_norm_rope_update_kv(s["q"], s["k"], s["v"], s["qw"], s["kw"], EPS, s["qo"], s["offsets"], s["cache"],
                               s["idx"], s["kvp"], s["lpl"], PAGE, config=s["rope"])
        return {"q": s["q"], "cache": s["cache"]}
    w = s["wrapper"]
    if kind == "refresh":
        if c["selector"] == "keymean":
            out, lse = w.run(s["q"], s["cache"], out=s["out"], return_lse=True, page_scores=s["sel"].page_scores)
            selected, counts = s["sel"].select(s["npg"], s["tab"])
            extra = s["sel"].page_scores
        else:
            out, lse = w.run(s["q"], s["cache"], s["dump"], c["hq"], s["stride"], out=s["out"], return_lse=True)
            selected, counts = s["sel"].select(s["dump"], lse, s["npg"], s["tab"], s["qo"])
            extra = s["dump"]
        return {"out": out, "lse": lse, "scores": extra, "selected": selected, "counts": counts}
    torch.ops.mylib.update_kv_padded(s["k"], s["v"], s["qo"], s["cache"], s["idx"], s["kvp"], s["lpl"], PAGE)
    out, lse = w.run(s["q"], s["cache"], out=s["out"], return_lse=True)
    return {"out": out, "lse": lse, "cache": s["cache"]}


# ------------------------------------------------------------------------------ work, tolerance
def work(case):
    c, kind = case, case["kind"]
    if kind in ("sample", "verify"):
        rows = c["rows"] if kind == "sample" else c["requests"] * (c["drafts"] + 1)
        more = 0 if kind == "sample" else c["requests"] * c["drafts"] * c["top_k"] * 12
        return {"bytes": rows * (VOCAB * 2 + c["top_k"] * (2 + 8 + 4) + 8) + more, "flops": 0}
    kv_row = c["hkv"] * D * 2 * 2  # one token's K and V
    if kind in ("prefill", "rope"):
        ctx, t = _chunk_rows(c)
        T = int(t.sum())
        io = T * c["hq"] * D * 2 * 2
        if kind == "rope":
            return {"bytes": io + T * kv_row * 2, "flops": 0}
        keys = sum(int(n) * (int(x) - int(n)) + int(n) * (int(n) + 1) // 2 for x, n in zip(ctx, t))
        # the new tokens' K and V are read once, written once; the prefix's are read
        return {"bytes": io + T * (c["hq"] * 4 + 2 * kv_row) + int((ctx - t).sum()) * kv_row + int(_pages(ctx).sum()) * 4,
                "flops": 4 * D * c["hq"] * keys}
    ctx, ql, dr = _decode_rows(c)
    n_pages, T = _pages(ctx), int(ql.sum())
    cnt = np.where(dr, np.minimum(c["budget"], n_pages), n_pages)
    part = (cnt - 1) * PAGE + (ctx - 1) % PAGE + 1
    if kind == "step":
        d, i = c["dim"], c["inter"]
        layer = (c["hq"] + 2 * c["hkv"]) * D * d + c["hq"] * D * d + 3 * i * d
        read = (c["layers"] - 1) * int(part.sum()) + int(ctx.sum())
        dump = int((np.where(ql > 1, 2, 1) * ctx).sum()) * c["hq"] * 2 * 2 if c["selector"] == "first_last" else 0
        return {"bytes": 2 * (c["layers"] * layer + VOCAB * d) + read * kv_row + c["layers"] * T * kv_row
                + T * (VOCAB + d) * 2 + dump,
                "flops": 2 * T * (c["layers"] * layer + VOCAB * d)
                + 4 * D * c["hq"] * ((c["layers"] - 1) * int((ql * part).sum()) + int((ql * ctx).sum()))}
    kv = ctx if kind == "refresh" else part
    nbytes = int(kv.sum()) * kv_row + T * c["hq"] * (D * 4 + 4) + int(_pages(kv).sum()) * 4
    if kind == "layer":
        nbytes += T * kv_row  # the appended rows are read from k / v and written to the cache
    elif c["selector"] == "first_last":
        nbytes += int((np.where(ql > 1, 2, 1) * ctx).sum()) * c["hq"] * 2 + c["batch"] * c["budget"] * 4
    else:
        nbytes += int((n_pages * (ql == 1)).sum()) * c["hkv"] * 4 + c["batch"] * c["hkv"] * c["budget"] * 4
    return {"bytes": nbytes, "flops": 4 * D * c["hq"] * int((ql * kv).sum())}


def tolerance(case):
    kind = case["kind"]
    if kind in ("sample", "verify"):
        # candidates are copied logits; probabilities are fp32 sums of fp32 exponentials
        return {"rel": 1e-5, "max": 1e-3, "differ": 0.005}
    if kind == "step":
        # bf16 roundings travel through every layer, and a page at the edge of a selection may change:
        # the same step with its products summed in another order is 0.008 to 0.013 off (largest 0.25)
        return {"rel": 3e-2, "max": 0.9}
    if kind == "rope":
        return {"rel": 4e-3, "max": 0.05}
    if kind == "refresh":
        # bf16 outputs; page lists shift where one page at the edge of a selection changes
        return {"rel": 8e-3, "max": 0.1, "differ": 0.005}
    return {"rel": 8e-3, "max": 0.1}


# ------------------------------------------------------------------------- the same in 64 bits
def _append64(d, k, v):
    """``cache`` with each row's new k / v at its last positions."""
    cache, at = d["cache"], 0
    for b, n in enumerate(d["ql"]):
        kv_len = (d["counts"][b] - 1) * PAGE + d["last"][b]
        pos = np.arange(kv_len - n, kv_len)
        page, slot = _dev(d["lists"][b][pos // PAGE], torch.int64), _dev(pos % PAGE, torch.int64)
        cache[page, 0, slot] = k[at: at + n].to(cache.dtype)
        cache[page, 1, slot] = v[at: at + n].to(cache.dtype)
        at += int(n)
    return cache


def _attend64(q, cache, pages, kv_len, heads, group, visit=None):
    """Causal attention of one row's q [n, hq, D] over the listed pages, for kv heads ``heads``:
    ([n, len(heads) * group, D], base-2 LSE). ``visit(kv head, raw logits [group, n, kv], keys)`` sees each."""
    n, outs, lses = q.shape[0], [], []
    pages = _dev(pages, torch.int64)
    for g in heads:
        k = cache[pages, 0, :, g].reshape(-1, D)[:kv_len].double()
        v = cache[pages, 1, :, g].reshape(-1, D)[:kv_len].double()
        qg = q[:, g * group: (g + 1) * group].double().transpose(0, 1)  # [group, n, D]
        parts, sums = [], []
        for i0 in range(0, n, 1024):
            x = qg[:, i0: i0 + 1024].reshape(-1, D) @ k.t()
            m = min(1024, n - i0)
            x = x.view(group, m, kv_len)
            if visit is not None:
                visit(g, x, k)
            x = x * (LOG2E / math.sqrt(D))
            see = torch.arange(i0, i0 + m, device="cuda")[:, None] + (kv_len - n) >= torch.arange(kv_len, device="cuda")
            x = x.masked_fill(~see, float("-inf"))
            top = x.amax(dim=-1, keepdim=True)
            p = torch.exp2(x - top)
            den = p.sum(dim=-1, keepdim=True)
            parts.append(((p.reshape(-1, kv_len) @ v).view(group, m, D) / den).transpose(0, 1))
            sums.append((top + torch.log2(den))[..., 0].transpose(0, 1))
        outs.append(torch.cat(parts))
        lses.append(torch.cat(sums))
    return torch.cat(outs, dim=1), torch.cat(lses, dim=1)


def _norm64(x, w):
    x = x.double()
    return x / torch.sqrt((x * x).mean(dim=-1, keepdim=True) + EPS) * w.double()


def _rope64(x, w, pos):
    """RMSNorm, the permute of the two halves into pairs, and the rotation of each pair."""
    x = _norm64(x, w)
    a, b = x[..., : D // 2], x[..., D // 2:]
    freq = (THETA ** (-2.0 * torch.arange(D // 2, device="cuda", dtype=torch.float64) / D)).float().double()
    ang = (pos.double()[:, None] * freq)[:, None]
    return torch.stack([a * ang.cos() - b * ang.sin(), b * ang.cos() + a * ang.sin()], dim=-1).flatten(-2)


def _pipe64(values, c):
    """softmax(values / temperature), cut to the smallest head that holds top_p, renormalised."""
    p = torch.softmax(values.double() / c["temperature"], dim=-1)
    srt = torch.sort(p, dim=-1, descending=True).values
    n = (torch.cumsum(srt, dim=-1) < c["top_p"]).sum(dim=-1, keepdim=True).clamp(max=p.shape[-1] - 1)
    p = torch.where(p >= torch.gather(srt, -1, n), p, torch.zeros_like(p))
    return p / p.sum(dim=-1, keepdim=True)


def exact(case, seed):
    c, kind = case, case["kind"]
    if kind == "sample":
        logits, _ = _logits(c["rows"], seed)
        values = torch.topk(logits.double(), c["top_k"], dim=-1).values
        return {"values": values, "ids": None, "probs": _pipe64(values, c), "pick": None}
    if kind == "verify":
        values = torch.topk(_verify_inputs(c, seed)["logits"].double(), c["top_k"], dim=-1).values
        return {"values": values, "ids": None, "probs": _pipe64(values, c), "output": None, "emitted": None}
    if kind == "step":
        return _exact_step(c, seed)
    d = _chunk_inputs(c, seed) if kind in ("prefill", "rope") else _decode_inputs(c, seed, kind == "refresh")
    if kind == "rope":
        pos = torch.cat([torch.arange(x - n, x) for x, n in zip(d["ctx"], d["ql"])]).to("cuda")
        q = _rope64(d["q"], d["qw"], pos)
        cache = {"cache": d["cache"].double(), **{k: d[k] for k in ("ql", "counts", "last", "lists")}}
        return {"q": q, "cache": _append64(cache, _rope64(d["k"], d["kw"], pos), d["v"].double())}
    group = c["hq"] // c["hkv"]
    if kind != "refresh":
        _append64(d, d["k"], d["v"])
    W = int(d["n_pages"].max())
    scores, dump = None, None
    if kind == "refresh" and c["selector"] == "keymean":
        scores = torch.zeros(c["batch"] * c["hkv"], W, dtype=torch.float64, device="cuda")
    elif kind == "refresh":
        dump = torch.full((c["batch"], c["hq"], 2, W * PAGE), float("-inf"), dtype=torch.float64, device="cuda")
    out, lse, at = torch.zeros(d["q"].shape, dtype=torch.float64, device="cuda"), [], 0
    for b, n in enumerate(d["ql"]):
        n, kv_len = int(n), int((d["counts"][b] - 1) * PAGE + d["last"][b])

        def visit(g, x, k):
            if dump is not None:
                heads = slice(g * group, (g + 1) * group)
                dump[b, heads, 0, :kv_len] = x[:, 0]
                if n > 1:
                    dump[b, heads, 1, :kv_len] = x[:, -1]
            elif n == 1:
                scores[b * c["hkv"] + g, : d["n_pages"][b]] = _key_mean64(x[:, 0], kv_len)

        out[at: at + n], l = _attend64(d["q"][at: at + n], d["cache"], d["lists"][b], kv_len, range(c["hkv"]), group,
                                       visit if kind == "refresh" else None)
        lse.append(l)
        at += n
    res = {"out": out, "lse": torch.cat(lse)}
    if kind != "refresh":
        return {**res, "cache": d["cache"]}
    return {**res, "scores": scores if scores is not None else dump.view(-1), "selected": None, "counts": None}


def _key_mean64(x, kv_len):
    """[group, kv] raw logits of one query -> each page's largest mean over the group's heads."""
    n = -(-kv_len // PAGE)
    x = torch.nn.functional.pad(x, (0, n * PAGE - kv_len)).view(x.shape[0], n, PAGE).sum(dim=-1)
    size = torch.full((n,), float(PAGE), dtype=torch.float64, device="cuda")
    size[-1] = kv_len - (n - 1) * PAGE
    return (x / size).amax(dim=0)


def _exact_step(c, seed):
    """The whole step in 64 bits: an eager one (its refresh layer chooses the pages) and the one that counts."""
    ctx, ql, dr = _decode_rows(c)
    n_pages, T = _pages(ctx), int(ql.sum())
    table = _table(n_pages, seed)
    hq, hkv, group, B, W = c["hq"], c["hkv"], c["hq"] // c["hkv"], c["batch"], table.shape[1]
    # the weights, keys and tokens of prepare(): random inputs by the same generators
    weights = DecodeWeights(_shape(c), "cuda", seed=seed)
    caches = alloc_kv_caches(_shape(c), int(n_pages.sum()), "cuda", seed=seed)
    tokens = torch.randint(0, VOCAB, (T,), generator=_gen(seed + 9), device="cuda")
    pos = torch.cat([torch.arange(x - n, x) for x, n in zip(ctx, ql)]).to("cuda")
    at, last = _ptr(ql), (ctx - 1) % PAGE + 1
    keep = np.where(dr, np.minimum(c["budget"], n_pages), n_pages)
    recent = _recent(c["selector"])
    logical = [[np.arange(n_pages[b] - keep[b], n_pages[b])] * hkv for b in range(B)]  # before any selection

    if c["selector"] == "first_last":
        scores = torch.full((B, hq, 2, W * PAGE), float("-inf"), dtype=torch.float64, device="cuda")
    else:
        scores = torch.zeros(B * hkv, W, dtype=torch.float64, device="cuda")

    def choose(b, page_scores):
        s = page_scores.clone()
        s[max(int(n_pages[b]) - recent, 0):] = float("inf")
        return torch.topk(s, int(keep[b])).indices.sort().values.cpu().numpy()

    def forward(lists, layers):
        """The last hidden state after ``layers`` layers, and the refresh layer's choice."""
        x, chosen = weights.tok_embeddings[tokens].double(), None
        for i in range(layers):
            lw = weights.layers[i]
            qkv = _norm64(x, lw["attention_norm"]) @ lw["wqkv"].double().t()
            q = _rope64(qkv[:, : hq * D].view(T, hq, D), lw["q_norm"], pos)
            k = _rope64(qkv[:, hq * D: (hq + hkv) * D].view(T, hkv, D), lw["k_norm"], pos)
            v = qkv[:, (hq + hkv) * D:].view(T, hkv, D)
            _append64(dict(cache=caches[i], ql=ql, counts=n_pages, last=last,
                           lists=[table[b, : n_pages[b]] for b in range(B)]), k, v)
            y = torch.zeros(T, hq, D, dtype=torch.float64, device="cuda")
            picked = [[None] * hkv for _ in range(B)]
            for b in range(B):
                rows, n = slice(int(at[b]), int(at[b + 1])), int(ql[b])
                whole = i == REFRESH_LAYER or not dr[b]
                row_max = [torch.zeros(int(ctx[b]), dtype=torch.float64, device="cuda") for _ in range(2)]
                raw = []

                def visit(g, z, _):
                    if c["selector"] == "first_last":
                        heads = slice(g * group, (g + 1) * group)
                        scores[b, heads, 0, : int(ctx[b])] = z[:, 0]
                        if n > 1:
                            scores[b, heads, 1, : int(ctx[b])] = z[:, -1]
                        raw.append(torch.stack([z[:, 0], z[:, -1]]))
                    elif n == 1:
                        scores[b * hkv + g, : n_pages[b]] = s = _key_mean64(z[:, 0], int(ctx[b]))
                        picked[b][g] = choose(b, s)

                for g in range(hkv):
                    pages = table[b, : n_pages[b]] if whole else table[b, lists[b][g]]
                    kv_len = (len(pages) - 1) * PAGE + int(last[b])
                    see = visit if i == REFRESH_LAYER else None
                    heads = slice(g * group, (g + 1) * group)
                    y[rows, heads], l = _attend64(q[rows], caches[i], pages, kv_len, [g], group, see)
                    if raw:  # the first/last queries' weights: the largest over heads, one row each
                        z, raw = raw[0], []
                        for slot, w in enumerate((l[0], l[-1])):
                            if slot == 0 or n > 1:
                                p = torch.exp2(z[slot] * (LOG2E / math.sqrt(D)) - w[:, None]).amax(dim=0)
                                row_max[slot] = torch.maximum(row_max[slot], p)
                if i == REFRESH_LAYER and c["selector"] == "first_last" and dr[b]:
                    s = torch.nn.functional.pad(row_max[0] + row_max[1], (0, int(n_pages[b]) * PAGE - int(ctx[b])))
                    s = s.view(-1, PAGE).sum(dim=-1) - 1e-7 * torch.arange(int(n_pages[b]), device="cuda")
                    picked[b] = [choose(b, s)] * hkv
            if i == REFRESH_LAYER:
                chosen = [picked[b] if dr[b] else lists[b] for b in range(B)]
                if c["selector"] == "keymean":
                    lists = chosen
            x = x + y.view(T, hq * D) @ lw["wo"].double().t()
            gate, up = (_norm64(x, lw["ffn_norm"]) @ lw["w13"].double().t()).chunk(2, dim=-1)
            x = x + (torch.nn.functional.silu(gate) * up) @ lw["w2"].double().t()
        return x, chosen

    if c["selector"] == "first_last":  # an empty dump selects the first pages and the recent ones
        logical = [[choose(b, -1e-7 * torch.arange(int(n_pages[b]), device="cuda", dtype=torch.float64))] * hkv
                   if dr[b] else logical[b] for b in range(B)]
    _, logical = forward(logical, REFRESH_LAYER + 1)
    x, _ = forward(logical, c["layers"])
    h, out = _norm64(x, weights.norm), torch.empty(T, VOCAB, dtype=torch.float64, device="cuda")
    for j in range(0, VOCAB, 16384):
        out[:, j: j + 16384] = h @ weights.output[j: j + 16384].double().t()
    return {"logits": out, "scores": scores.view(-1) if c["selector"] == "first_last" else scores}

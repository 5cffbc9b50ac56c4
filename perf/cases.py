"""The work that a serving program has this library do, as cases that can be timed and compared.

Four kinds of call, each through the entry point a program uses:

    attend   PagedAttention.forward_async    one layer's attention over the paged cache: decode
                                             (one row a sequence), verify (the drafts and one
                                             more), prefill (a prompt or a chunk of one)
    append   PagedKVCache.append_kv_async    one layer's new K/V rows into the paged cache
    accept   verify_drafts_async             acceptance sampling of a verify step
    sample   sample_tokens_async             plain-decode sampling with the logit processors

A case is a dict of plain values; `listed` gives the ones that are always measured, `draw` more of
the same ranges. Lengths and row counts follow from the case alone, the values and the order of
the sequences from the seed. Inputs are made on the GPU.
"""
import math

import numpy as np
import torch

import kyro_amd
from kyro_amd.sampling import Processors

_DTYPES = {"bf16": torch.bfloat16, "f32": torch.float32}


def _attend(name, batch, heads, kv_heads, dim, ctx, rows, dtype="bf16", block=16):
    """`ctx` and `rows` are (least, most) over the batch; a context length counts the new rows."""
    case = {"op": "attend", "batch": batch, "heads": heads, "kv_heads": kv_heads, "dim": dim, "block": block,
            "ctx_min": ctx[0], "ctx_max": ctx[1], "rows_min": rows[0], "rows_max": rows[1], "dtype": dtype}
    return dict(case, name=name) if name else case


def listed():
    return [
        # One conversation, one token: the call a single user waits for, all latency.
        _attend("decode_one", 1, 32, 8, 128, (1000, 1000), (1, 1)),
        # Continuous batching: one token for each of 48 sequences of very different ages.
        _attend("decode_ragged", 48, 32, 8, 128, (200, 6000), (1, 1)),
        # The Llama-3-8B verify step: 7 drafts and one more row for 64 sequences.
        _attend("verify_batch", 64, 32, 8, 128, (4096, 4096), (8, 8)),
        # A Llama-3-70B layer under mixed draft lengths: 0 to 8 drafts, short and long contexts.
        _attend("verify_mixed", 128, 64, 8, 128, (256, 8192), (1, 9)),
        # Four new prompts of 2048 tokens.
        _attend("prefill", 4, 32, 8, 128, (2048, 2048), (2048, 2048)),
        # Chunked prefill of a small model: the next 500 or so tokens of prompts under way.
        _attend("prefill_chunk", 6, 32, 8, 64, (700, 8000), (300, 512)),
        # The reference computes in f32, so its own caches are f32: a verify step on them.
        _attend("verify_f32", 32, 32, 8, 128, (500, 4000), (5, 5), dtype="f32"),
        # Decode of a small model with 64-wide heads on f32 caches.
        _attend("decode_f32_dim64", 16, 32, 8, 64, (300, 3000), (1, 1), dtype="f32"),
        # The new K/V of four 2048-token prompts into the cache.
        {"name": "append_prompts", "op": "append", "batch": 4, "kv_heads": 8, "dim": 128, "block": 16,
         "old_min": 0, "old_max": 0, "rows_min": 2048, "rows_max": 2048, "src": "bf16", "dtype": "bf16"},
        # Acceptance of the Llama-3-8B verify step, with the probabilities of the drafts.
        {"name": "accept_batch", "op": "accept", "batch": 64, "drafts_min": 7, "drafts_max": 7, "vocab": 128256,
         "temperature": 0.8, "greedy": 0.0, "target_sigma": 3.0, "noise_sigma": 1.0, "probs": True},
        # Acceptance of a small batch over a small vocabulary: launches count.
        {"name": "accept_small", "op": "accept", "batch": 8, "drafts_min": 4, "drafts_max": 4, "vocab": 32000,
         "temperature": 1.0, "greedy": 0.0, "target_sigma": 2.0, "noise_sigma": 0.5, "probs": False},
        # Sampling a decode batch with top-k, top-p, penalties, biases and a grammar mask.
        {"name": "sample_nucleus", "op": "sample", "batch": 64, "vocab": 128256, "temperature": 0.8, "sigma": 3.0,
         "top_k": 50, "top_p": 0.9, "processors": True},
    ]


# ------------------------------------------------------------------------------------ drawn cases

def _spread(rng, lo, hi):
    """An integer in [lo, hi], spread over its logarithm."""
    return int(min(hi, max(lo, round(math.exp(rng.uniform(math.log(lo), math.log(hi + 1)))))))


def _draw_attend(rng):
    mode = rng.choice(("decode", "decode", "verify", "verify", "prefill", "prefill"))
    dtype = rng.choice(("bf16", "bf16", "bf16", "f32"))
    dim = rng.choice((64, 80, 96, 128, 128, 128, 256) if dtype == "bf16" else (64, 80, 96, 128, 128))
    kv_heads = rng.choice((2, 4, 8, 8, 16, 32))
    group = rng.choice((1, 4, 7, 8) if kv_heads <= 8 else (1, 2))
    block = rng.choice((16, 16, 16, 32, 64))
    size = 2 if dtype == "bf16" else 4
    if mode == "prefill":
        batch = _spread(rng, 1, 8)
        most = _spread(rng, 64, 4096)
        rows = (max(1, most // rng.choice((1, 2, 7))), most)
        old = rng.choice((0, 0, _spread(rng, 1, 4096)))
        # At most the work of the largest listed prefill (f32 does a product in eight times the time).
        budget = (1.3e11 if dtype == "bf16" else 1.6e10) * (0.5 if dim > 128 else 1.0)
        while True:
            case = _attend(None, batch, kv_heads * group, kv_heads, dim, (rows[0] + old, rows[1] + old), rows, dtype, block)
            if work(case)["flops"] <= budget:
                return case
            if batch > 1:
                batch = (batch + 1) // 2
            elif rows[1] > 64 and rows[1] >= old:
                rows = (max(1, rows[0] // 2), rows[1] // 2 + 1)
            else:
                old //= 2
    batch = _spread(rng, 1, 128)
    rows = (1, 1) if mode == "decode" else rng.choice(((5, 5), (8, 8), (2, 9), (3, 3)))
    most = _spread(rng, 64, 16384)
    while True:  # at most the bytes of the largest listed verify step
        case = _attend(None, batch, kv_heads * group, kv_heads, dim, (max(rows[1], most // rng.choice((1, 3, 12))), most),
                       rows, dtype, block)
        if 2 * kv_heads * dim * size * sum(_lengths(case)[0]) <= 1.2e9:
            return case
        batch, most = max(1, batch * 2 // 3), max(64, most * 4 // 5)


def draw(rng):
    kind = rng.choice(("attend", "attend", "attend", "attend", "append", "accept", "sample"))
    if kind == "attend":
        return _draw_attend(rng)
    if kind == "append":
        prompts = rng.random() < 0.5
        most = _spread(rng, 64, 4096) if prompts else rng.choice((1, 5, 9))
        batch = _spread(rng, 1, 4) if prompts else _spread(rng, 1, 128)
        src = rng.choice(("bf16", "f32"))
        return {"op": "append", "batch": batch, "kv_heads": rng.choice((2, 8, 8, 32)), "dim": rng.choice((64, 80, 128, 128)),
                "block": rng.choice((16, 16, 32)), "old_min": 0, "old_max": 0 if prompts else _spread(rng, 16, 1024),
                "rows_min": max(1, most // 2), "rows_max": most, "src": src, "dtype": rng.choice(("bf16", src))}
    vocab = rng.choice((32000, 50257, 128256, _spread(rng, 1000, 150000)))
    temperature = round(rng.uniform(0.5, 1.2), 2)
    if kind == "accept":
        drafts = rng.choice((1, 3, 4, 5, 7, 8))
        batch = max(1, min(_spread(rng, 1, 96), int(1.1e8 / (vocab * (2 * drafts + 1)))))
        return {"op": "accept", "batch": batch, "drafts_min": rng.choice((drafts, 1)), "drafts_max": drafts, "vocab": vocab,
                "temperature": temperature, "greedy": rng.choice((0.0, 0.0, 0.5)), "target_sigma": 3.0,
                "noise_sigma": rng.choice((0.3, 1.0)), "probs": rng.random() < 0.5}
    top_k, top_p = rng.choice(((0, 1.0), (50, 1.0), (0, 0.9), (40, 0.95), (0, 0.95)))
    return {"op": "sample", "batch": _spread(rng, 1, 128), "vocab": vocab, "temperature": rng.choice((0.0, temperature, temperature)),
            "sigma": 3.0, "top_k": top_k, "top_p": top_p, "processors": rng.random() < 0.4}


# ------------------------------------------------------------------------------- sizes of a case

def _even(lo, hi, n):
    """n integers from hi down to lo, evenly spaced (hi alone for one)."""
    return [hi] if n == 1 else [int(round(hi - (hi - lo) * i / (n - 1))) for i in range(n)]


def _lengths(case):
    """(context lengths, new rows) of a batch's sequences, before the seed orders them."""
    n = case["batch"]
    step = next(s for s in (7, 5, 3, 1) if math.gcd(s, n) == 1)  # rows and lengths out of step
    if case["op"] == "attend":
        rows = _even(case["rows_min"], case["rows_max"], n)
        rows = [rows[i * step % n] for i in range(n)]
        return [max(c, r) for c, r in zip(_even(case["ctx_min"], case["ctx_max"], n), rows)], rows
    rows = _even(case["rows_min"], case["rows_max"], n)
    old = _even(case["old_min"], case["old_max"], n)
    return [o + rows[i * step % n] for i, o in enumerate(old)], [rows[i * step % n] for i in range(n)]


def _drafts(case):
    return _even(case["drafts_min"], case["drafts_max"], case["batch"])


def _greedy_rows(case):
    return int(round(case["greedy"] * case["batch"]))


def work(case):
    if case["op"] == "attend":
        size = 2 if case["dtype"] == "bf16" else 4
        ctx, rows = _lengths(case)
        per_row = case["heads"] * case["dim"]
        seen = sum(r * c - r * (r - 1) // 2 for c, r in zip(ctx, rows))  # causal pairs of a row and a token
        return {"bytes": 2 * sum(ctx) * case["kv_heads"] * case["dim"] * size + 2 * sum(rows) * per_row * size,
                "flops": 4 * seen * per_row}
    if case["op"] == "append":
        each = (2 if case["src"] == "bf16" else 4) + (2 if case["dtype"] == "bf16" else 4)
        return {"bytes": 2 * sum(_lengths(case)[1]) * case["kv_heads"] * case["dim"] * each, "flops": 0}
    if case["op"] == "accept":
        # Every sequence needs the rows of its first draft; which of the later ones it needs
        # depends on the values. About half of the drafts are accepted, so two positions stand for them.
        rows = sum(2 * min(2, k) + (k < 2) for k in _drafts(case))
        return {"bytes": 4 * rows * case["vocab"], "flops": 8 * rows * case["vocab"]}
    n = case["batch"] * case["vocab"]
    return {"bytes": 4 * n, "flops": 4 * n}


def tolerance(case):
    if case["op"] == "attend":
        # bf16: probabilities and outputs are rounded to 8 bits, about 2.5e-3 of the result in all.
        # f32: sums of thousands of products, 3e-7 to 8e-7.
        return {"rel": 1e-2, "max": 0.1} if case["dtype"] == "bf16" else {"rel": 5e-6, "max": 1e-4}
    if case["op"] == "append":
        return "exact"
    if case["op"] == "accept":
        # A draw or a decision within rounding of its boundary may fall on the other side.
        return {"rel": 2e-5, "max": 2e-4, "differ": 0.004}
    return {"differ": 0.01}


# ------------------------------------------------------------------------------------------ inputs

def _generator(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed))
    return g


def _randn(g, shape, dtype=torch.float32):
    return torch.randn(shape, generator=g, device="cuda", dtype=dtype)


def _paged(case, seed):
    """(context lengths, new rows, q_start_loc, block table, blocks) with the sequences and the
    pool's blocks in the seed's order."""
    rng = np.random.default_rng(int(seed))
    ctx, rows = (np.asarray(x, np.int64) for x in _lengths(case))
    order = rng.permutation(case["batch"])
    ctx, rows = ctx[order], rows[order]
    need = -(-ctx // case["block"])
    pool = int(need.sum())
    perm = rng.permutation(pool)
    table = np.zeros((case["batch"], int(need.max())), np.int64)
    at = 0
    for b, n in enumerate(need):
        table[b, :n] = perm[at:at + n]
        at += n
    start = np.zeros(case["batch"] + 1, np.int32)
    start[1:] = np.cumsum(rows)
    return ctx, rows, start, table, pool


def prepare(case, seed):
    g = _generator(seed)
    if case["op"] in ("attend", "append"):
        ctx, rows, start, table, pool = _paged(case, seed)
        state = {"case": case, "rows": int(rows.max()), "ctx": torch.from_numpy(ctx).cuda(),
                 "table": torch.from_numpy(table).cuda(),
                 # One row a sequence is the library's plain form: no q_start_loc.
                 "start": None if int(rows.max()) == 1 else torch.from_numpy(start).cuda()}
        total, dtype = int(rows.sum()), _DTYPES[case["dtype"]]
        cache = (pool, case["kv_heads"], case["block"], case["dim"])
        if case["op"] == "attend":
            return dict(state, attn=kyro_amd.PagedAttention(case["block"], case["heads"], case["dim"], case["kv_heads"]),
                        q=_randn(g, (total, case["heads"], case["dim"]), dtype), k=_randn(g, cache, dtype),
                        v=_randn(g, cache, dtype))
        new, src = (total, case["kv_heads"], case["dim"]), _DTYPES[case["src"]]
        return dict(state, cache=kyro_amd.PagedKVCache(case["block"], case["kv_heads"], case["dim"]),
                    key=_randn(g, new, src), value=_randn(g, new, src),
                    k=torch.zeros(cache, dtype=dtype, device="cuda"), v=torch.zeros(cache, dtype=dtype, device="cuda"))
    B, V = case["batch"], case["vocab"]
    if case["op"] == "accept":
        k = np.asarray(_drafts(case), np.int32)[np.random.default_rng(int(seed)).permutation(B)]
        kmax = case["drafts_max"]
        t = np.full(B, case["temperature"], np.float32)
        t[np.random.default_rng(int(seed) + 1).permutation(B)[:_greedy_rows(case)]] = 0.0
        t = torch.from_numpy(t).cuda()
        target = _randn(g, (B, kmax + 1, V)).mul_(case["target_sigma"])
        draft = target[:, :kmax] + _randn(g, (B, kmax, V)).mul_(case["noise_sigma"])
        # Drafts are drawn from the draft model at the same temperature (its maximum when greedy).
        noise = torch.empty(B, kmax, V, device="cuda").exponential_(generator=g).log_().neg_()
        tokens = (draft + noise * t.view(B, 1, 1)).argmax(-1).to(torch.int32)
        draws = torch.rand(B, kmax + 1, generator=g, device="cuda").clamp_(1e-6, 1 - 1e-6)
        return {"case": case, "args": (target, draft.contiguous(), tokens.contiguous(), torch.from_numpy(k).cuda(), t,
                                       draws[:, :kmax].contiguous(), draws[:, kmax].contiguous())}
    state = {"case": case, "logits": _randn(g, (B, V)).mul_(case["sigma"]),
             "t": torch.full((B,), case["temperature"], device="cuda"),
             "u": torch.rand(B, generator=g, device="cuda"), "top_k": None, "top_p": None, "processors": None}
    if case["top_k"]:
        state["top_k"] = torch.full((B,), case["top_k"], dtype=torch.int32, device="cuda")
    if case["top_p"] < 1.0:
        state["top_p"] = torch.full((B,), case["top_p"], device="cuda")
    if case["processors"]:
        rng = np.random.default_rng(int(seed))
        # A request's generated tokens with their penalties, a few biases, and for every fourth row
        # a grammar that allows half of the vocabulary.
        penalty = [{int(x): -float(rng.uniform(0.1, 2.0)) for x in rng.integers(0, V, 60)} for _ in range(B)]
        bias = [{int(x): float(rng.uniform(-5, 5)) for x in rng.integers(0, V, 8)} if b % 2 else None for b in range(B)]
        words = rng.integers(0, 1 << 32, size=(1, (V + 31) // 32), dtype=np.uint64).astype(np.uint32)
        if V % 32:
            words[:, -1] &= np.uint32((1 << (V % 32)) - 1)
        mask_row = np.where(np.arange(B) % 4 == 0, 0, -1)
        state["processors"] = Processors(B, V, torch.device("cuda", 0), bias=bias, penalty=penalty, masks=words,
                                         mask_row=mask_row)
    return state


def run(state):
    case = state["case"]
    if case["op"] == "attend":
        return state["attn"].forward_async(state["q"], state["k"], state["v"], state["table"], state["ctx"],
                                           q_start_loc=state["start"], max_q_len=state["rows"],
                                           out_dtype=_DTYPES[case["dtype"]])
    if case["op"] == "append":
        state["cache"].append_kv_async(state["key"], state["value"], state["k"], state["v"], state["table"], state["ctx"],
                                       q_start_loc=state["start"], max_q_len=state["rows"])
        return [state["k"], state["v"]]
    if case["op"] == "accept":
        got = kyro_amd.verify_drafts_async(*state["args"], return_probs=case["probs"])
        return {"accepted": got.accepted, "tokens": got.tokens, "p": got.p_draft, "q": got.q_draft}
    return kyro_amd.sample_tokens_async(state["logits"], state["t"], state["u"], top_p=state["top_p"], top_k=state["top_k"],
                                        processors=state["processors"])


# ---------------------------------------------------------------------------------- 64-bit results

def _exact_attend(state):
    case, out = state["case"], []
    H, Hkv, D = case["heads"], case["kv_heads"], case["dim"]
    starts = state["start"].tolist() if state["start"] is not None else list(range(case["batch"] + 1))
    for b, ctx in enumerate(state["ctx"].tolist()):
        q = state["q"][starts[b]:starts[b + 1]].double()
        n = q.shape[0]
        ids = state["table"][b, :-(-ctx // case["block"])]
        k, v = (state[x][ids].transpose(0, 1).reshape(Hkv, -1, D)[:, :ctx].double() for x in ("k", "v"))
        q = q.view(n, Hkv, H // Hkv, D).permute(1, 0, 2, 3).reshape(Hkv, -1, D)
        hidden = torch.arange(ctx, device="cuda").view(1, -1) > (ctx - n + torch.arange(n, device="cuda")).view(-1, 1)
        hidden = hidden.repeat_interleave(H // Hkv, 0)
        parts = []
        for h in range(Hkv):
            s = (q[h] @ k[h].t()) / math.sqrt(D)
            s.masked_fill_(hidden, -math.inf)
            parts.append(torch.softmax(s, -1) @ v[h])
        o = torch.stack(parts).view(Hkv, n, H // Hkv, D).permute(1, 0, 2, 3).reshape(n, H, D)
        out.append(o)
    return torch.cat(out)


def _exact_accept(state):
    target, draft, tokens, k, t, u, _ = state["args"]
    B, kmax = tokens.shape
    p = torch.full((B, kmax), math.nan, dtype=torch.float64)
    q, accepted = p.clone(), []
    for b in range(B):
        kb, T, stop = int(k[b]), float(t[b]), None
        for i in range(kb):
            x = int(tokens[b, i])
            if T > 0:
                p[b, i] = torch.softmax(target[b, i].double() / T, -1)[x]
                q[b, i] = torch.softmax(draft[b, i].double() / T, -1)[x]
                ok = float(u[b, i]) * float(q[b, i]) < float(p[b, i])
            else:
                ok = int(target[b, i].argmax()) == x
            if not ok:
                stop = i
                break
        accepted.append(kb if stop is None else stop)
    return {"accepted": torch.tensor(accepted, dtype=torch.int32), "tokens": None,
            "p": p if state["case"]["probs"] else None, "q": q if state["case"]["probs"] else None}


def exact(case, seed):
    if case["op"] == "attend":
        return _exact_attend(prepare(case, seed))
    if case["op"] == "accept":
        return _exact_accept(prepare(case, seed))
    return None

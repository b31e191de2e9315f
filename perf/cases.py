"""Performance cases of the framework's public entry points.

Each case is one call (or one short chain of calls) that a serving or training
program makes: sparse MLA decode, verification and prefill (``sparse_mla``), the
framework ops chained as one attention layer (``sparse_topk_indices`` ->
``sparse_flash_mla``), the top-k index selection alone, BNSD flash attention
(``attention_target``) and the single-tile attention (``simple_attention``).

``listed()`` gives the fixed cases, ``draw(rng)`` another one of the same
ranges, ``prepare`` the device tensors a program has in hand before the call,
``run`` the call, ``exact`` its result in float64 with plain torch.
"""

from __future__ import annotations

import math
import random

import torch

from ascendflow_amd.flash_attention import attention_target, simple_attention
from ascendflow_amd.sparse_attention import sparse_mla, sparse_topk_indices
from ascendflow_amd.sparse_attention import ops  # noqa: F401  (registers the torch ops)

PAGE = 128
WINDOW = 128
B16 = {"bf16": torch.bfloat16, "f16": torch.float16}


def listed():
    return [
        # One user's single-token decode step: the smallest call, launch and latency bound.
        _mla("mla_decode_1x1_4k", B=1, n=1, context=4096),
        # Batched decode with five draft tokens per request at 128K context.
        _mla("mla_decode_64x6_128k", B=64, n=6, context=131072),
        # One long prompt chunk: 8K query tokens against 32K of context.
        _mla("mla_prefill_8k_32k", B=1, n=8192, context=32768),
        # Chunked prefill of a few unequal requests on a small f16 model: 32 heads of 256 features, no compression.
        _mla("mla_chunk_3x470_f16", B=3, n=470, context=6000, H=32, D=256, R=1, dtype="f16", ragged=True),
        # A whole attention layer of a mixed decode batch through the framework ops: scores -> top-k -> attention + LSE.
        {**_mla("layer_24x3_h128", B=24, n=3, context=20000, H=128, ragged=True), "kind": "layer"},
        # Index selection of the batched decode above: 384 rows of 64K scores.
        _topk("topk_decode_64x6_64k", B=64, n=6, context=131072),
        # Index selection of a prompt chunk; the row length is odd, as context lengths are.
        _topk("topk_prefill_4k_16391", B=1, n=4096, context=32782),
        # Index selection of one request at 1M tokens of context with three draft tokens.
        _topk("topk_decode_1x4_512k", B=1, n=4, context=1048576),
        # Dense prefill of the published size.
        _fa("fa_prefill_8k_f16", B=1, HQ=32, HKV=32, Sq=8192, Sk=8192, dtype="f16", causal=False),
        # Causal training-style forward with grouped heads at an ordinary, odd length.
        _fa("fa_causal_2x1987_gqa", B=2, HQ=32, HKV=8, Sq=1987, Sk=1987, dtype="bf16", causal=True),
        # Dense decode: one query token per request against a 32K cache, grouped heads.
        _fa("fa_decode_8x32k_gqa", B=8, HQ=32, HKV=8, Sq=1, Sk=32768, dtype="bf16", causal=False),
        # Single-tile attention over many rows.
        {"name": "simple_32x8192", "kind": "simple", "H": 32, "S": 8192},
    ]


def _mla(name, *, B, n, context, H=64, D=512, R=2, topk=512, dtype="bf16", ragged=False, lse=False):
    return {"name": name, "kind": "mla", "B": B, "n": n, "context": context, "H": H, "D": D, "R": R, "topk": topk,
            "dtype": dtype, "ragged": ragged, "lse": lse}


def _topk(name, *, B, n, context, R=2, topk=512, ragged=False):
    return {"name": name, "kind": "topk", "B": B, "n": n, "context": context, "R": R, "topk": topk, "ragged": ragged}


def _fa(name, **sizes):
    return {"name": name, "kind": "fa", **sizes}


def _log_int(rng, low, high):
    return int(round(math.exp(rng.uniform(math.log(low), math.log(max(low, high))))))


def draw(rng):
    kind = rng.choice(["mla", "mla", "mla", "mla", "layer", "topk", "topk", "topk", "fa", "fa", "fa", "simple"])
    if kind == "simple":
        return {"kind": kind, "H": _log_int(rng, 1, 64), "S": 64 * _log_int(rng, 1, 128)}
    if kind == "fa":
        HQ, HKV = rng.choice([(32, 32), (32, 8), (32, 8), (16, 2), (8, 8), (28, 4), (64, 8)])
        decode = rng.random() < 0.4
        if decode:  # a few query rows against a cache
            Sq, Sk, causal = _log_int(rng, 1, 16), _log_int(rng, 500, 65536), False
        else:
            Sk, causal = _log_int(rng, 100, 8192), rng.random() < 0.6
            Sq = Sk if causal or rng.random() < 0.7 else _log_int(rng, 64, 8192)
        cost = HQ * max(Sq * Sk, Sk * 256)  # of one batch entry, against the largest listed case
        B = _log_int(rng, 1, max(1, min(32, int(32 * 8192 * 8192 / cost))))
        return {"kind": kind, "B": B, "HQ": HQ, "HKV": HKV, "Sq": Sq, "Sk": Sk, "dtype": rng.choice(["bf16", "f16"]),
                "causal": causal}
    B = _log_int(rng, 1, 64)
    n = _log_int(rng, 1, 8 if rng.random() < 0.5 else max(8, 6000 // B))
    case = {"kind": kind, "B": B, "n": n, "R": rng.choice([2, 2, 2, 1]), "topk": rng.choice([512, 512, 512, 256, 1024]),
            "ragged": rng.random() < 0.6}
    longest = min(131072, 4194304 // B)
    if kind == "topk":
        if B * n <= 16:  # few rows: up to the longest contexts served
            longest = 1048576
        longest = min(longest, max(1024, 2 ** 26 // (B * n)) * case["R"])
        case["context"] = max(2 * n, _log_int(rng, 1500, longest))
        return case
    H, D = rng.choice([(64, 512), (64, 512), (64, 512), (128, 512), (32, 256), (64, 128)])
    case["n"] = n = max(1, min(n, int(6.0e11 / (4 * H * D * (WINDOW + case["topk"]) * B * 1.5))))
    case["context"] = max(2 * n, _log_int(rng, 1500, longest))
    return {**case, "H": H, "D": D, "dtype": rng.choice(["bf16", "bf16", "f16"]), "lse": rng.random() < 0.3}


# ---- sizes of a sparse case ----------------------------------------------------


def _requests(case):
    """(query tokens, context) of each request; the same for every seed."""
    B, n, context = case["B"], case["n"], case["context"]
    if not case["ragged"]:
        return [n] * B, [context] * B
    rng = random.Random(B * 1000003 + n * 1009 + context)
    counts = [max(1, rng.randint(n // 2, n + n // 2)) for _ in range(B)]
    return counts, [max(c, rng.randint(context // 2, context)) for c in counts]


def _bounds(case):
    """Per token (on the host): its request, the causal end of its window and its compressed candidates."""
    counts, contexts = _requests(case)
    request, right = [], []
    for b, (c, s) in enumerate(zip(counts, contexts)):
        request += [b] * c
        right += range(s - c + 1, s + 1)
    return request, right, [r // case["R"] for r in right]


def _columns(case):
    return max(c // case["R"] for c in _requests(case)[1])


def _metadata(case, gen, device):
    counts, contexts = _requests(case)
    R = case["R"]
    i32 = dict(dtype=torch.int32, device=device)
    cu = [0]
    for c in counts:
        cu.append(cu[-1] + c)
    width = -(-max(contexts) // PAGE)
    blocks = len(counts) * width
    return {
        "cu_seqlens_q": torch.tensor(cu, **i32),
        "seqused_ori_kv": torch.tensor(contexts, **i32),
        "seqused_cmp_kv": torch.tensor([c // R for c in contexts], **i32),
        "cmp_residual_kv": torch.tensor([c % R for c in contexts], **i32),
        "ori_block_table": torch.randperm(blocks, generator=gen, device=device).to(torch.int32).view(len(counts), width),
        "cmp_block_table": torch.randperm(blocks, generator=gen, device=device).to(torch.int32).view(len(counts), width),
    }, width, blocks


def _scores(case, gen, device):
    """Index scores [T, C] f32: one per (token, compressed position), neighbouring tokens alike."""
    counts, _ = _requests(case)
    C = _columns(case)
    scores = torch.empty((sum(counts), C), dtype=torch.float32, device=device)
    first = 0
    for c in counts:
        shared = torch.randn((1, C), generator=gen, device=device)
        scores[first:first + c].normal_(generator=gen).mul_(0.6).add_(shared, alpha=0.8)
        first += c
    return scores


def _random_indices(case, gen, device):
    """Sorted random selections without repeats below each token's candidates, -1 after them."""
    topk, C = case["topk"], _columns(case)
    limit = torch.tensor(_bounds(case)[2], device=device).view(-1, 1)
    out = torch.full((limit.shape[0], 1, topk), -1, dtype=torch.int32, device=device)
    position = torch.arange(C, device=device)
    k = min(topk, C)
    step = max(1, 2 ** 26 // C)
    for t in range(0, limit.shape[0], step):
        lim = limit[t:t + step]
        keys = torch.rand((lim.shape[0], C), generator=gen, device=device).masked_fill_(position >= lim, -1.0)
        value, index = keys.topk(k, dim=1)
        index = index.masked_fill(value < 0, C).sort(dim=1).values  # unused ones to the end
        out[t:t + step, 0, :k] = index.masked_fill(index == C, -1).to(torch.int32)
    return out


def prepare(case, seed):
    device = torch.device("cuda")
    gen = torch.Generator(device=device)
    gen.manual_seed(seed)
    kind = case["kind"]

    def normal(shape, dtype):
        return torch.randn(shape, generator=gen, device=device, dtype=dtype)

    if kind == "simple":
        H, S = case["H"], case["S"]
        q, k, v = (normal((H, rows, 128), torch.float16) for rows in (S, 128, 128))
        return {"kind": kind, "args": (q, k, v, torch.empty_like(q)), "kw": {"S": S, "H": H}}
    if kind == "fa":
        B, HQ, HKV, Sq, Sk = (case[x] for x in ("B", "HQ", "HKV", "Sq", "Sk"))
        b16 = B16[case["dtype"]]
        q, k, v = (normal(shape, b16) for shape in ((B, HQ, Sq, 128), (B, HKV, Sk, 128), (B, HKV, Sk, 128)))
        return {"kind": kind, "args": (q, k, v, torch.empty_like(q), Sq, Sk),
                "kw": dict(B=B, HQ=HQ, HKV=HKV, D=128, DTYPE=case["dtype"], SCALE=128 ** -0.5, CAUSAL=case["causal"])}

    meta, width, blocks = _metadata(case, gen, device)
    R, topk = case["R"], case["topk"]
    T = sum(_requests(case)[0])
    state = {"kind": kind, "meta": meta, "R": R, "topk": topk}
    if kind in ("topk", "layer"):
        state["scores"] = _scores(case, gen, device)
    if kind == "topk":
        state["out"] = torch.empty((T, 1, topk), dtype=torch.int32, device=device)
        return state
    H, D, b16 = case["H"], case["D"], B16[case["dtype"]]
    t = {
        "q": normal((T, H, D), b16),
        "ori_kv": normal((blocks, PAGE, 1, D), b16),
        "cmp_kv": normal((blocks, PAGE // R, 1, D), b16),
        "ori_topk_length": torch.zeros((T, 1), dtype=torch.int32, device=device),
        "sinks": torch.linspace(-2.0, 2.0, H, device=device),
        **meta,
    }
    state["t"], state["scale"] = t, D ** -0.5
    if kind == "mla":
        t["cmp_sparse_indices"] = _random_indices(case, gen, device)
        t["attention_out"] = torch.empty_like(t["q"])
        state["lse"] = torch.empty((T, H), device=device) if case["lse"] else None
        order = ("q", "ori_kv", "cmp_kv", "cmp_sparse_indices", "ori_block_table", "cmp_block_table", "cu_seqlens_q",
                 "seqused_ori_kv", "seqused_cmp_kv", "cmp_residual_kv", "ori_topk_length", "sinks", "attention_out")
        state["args"] = [t[name] for name in order]
        BM = 64 if H % 64 == 0 else 32
        state["kw"] = dict(B=case["B"], T=T, H=H, D=D, PAGE=PAGE, RATIO=R, MAX_SEQ=width * PAGE, ORI_BLOCKS=blocks,
                           CMP_BLOCKS=blocks, WINDOW=WINDOW, TOPK=topk, S=WINDOW + -(-topk // 512) * 512, BM=BM,
                           VR=16 if BM == 64 else 8, DTYPE=case["dtype"], SCALE=D ** -0.5)
    return state


def run(state):
    kind = state["kind"]
    if kind == "simple":
        return simple_attention(*state["args"], **state["kw"])
    if kind == "fa":
        return attention_target(*state["args"], **state["kw"])
    if kind == "topk":
        m = state["meta"]
        return sparse_topk_indices(state["scores"], m["cu_seqlens_q"], m["seqused_cmp_kv"], m["cmp_residual_kv"],
                                   TOPK=state["topk"], RATIO=state["R"], out=state["out"])
    if kind == "mla":
        if state["lse"] is None:
            return sparse_mla(*state["args"], **state["kw"])
        return sparse_mla(*state["args"], **state["kw"], softmax_lse=state["lse"]), state["lse"]
    t = state["t"]
    indices = torch.ops.ascendflow_amd.sparse_topk_indices(
        state["scores"], t["cu_seqlens_q"], t["seqused_cmp_kv"], t["cmp_residual_kv"], state["topk"], state["R"])
    out, lse = torch.ops.ascendflow_amd.sparse_flash_mla(
        t["q"], t["ori_kv"], t["cmp_kv"], indices, t["ori_block_table"], t["cmp_block_table"], t["cu_seqlens_q"],
        t["seqused_ori_kv"], t["seqused_cmp_kv"], t["cmp_residual_kv"], t["ori_topk_length"], t["sinks"],
        state["scale"], state["R"], return_softmax_lse=True)
    return indices, out, lse


def work(case):
    kind = case["kind"]
    if kind == "simple":
        H, S = case["H"], case["S"]
        return {"bytes": 2 * 128 * H * (2 * S + 2 * 128), "flops": 4 * 128 * 128 * S * H}
    if kind == "fa":
        B, HQ, HKV, Sq, Sk = (case[x] for x in ("B", "HQ", "HKV", "Sq", "Sk"))
        pairs, keys = Sq * Sk, Sk
        if case["causal"]:
            m = min(Sq, Sk)
            pairs, keys = m * (m + 1) // 2 + (Sq - m) * Sk, m
        return {"bytes": 2 * 128 * B * (2 * HQ * Sq + 2 * HKV * keys), "flops": 4 * 128 * B * HQ * pairs}
    topk = case["topk"]
    _, right, candidates = _bounds(case)
    T = len(right)
    total = {"bytes": 0, "flops": 0}
    if kind in ("topk", "layer"):
        total["bytes"] += 4 * sum(candidates) + 4 * T * topk
    if kind == "topk":
        return total
    H, D = case["H"], case["D"]
    rows = sum(min(WINDOW, r) + min(topk, c) for r, c in zip(right, candidates))
    unique = 0.0  # rows that some token of the request reads, each once
    for n, s in zip(*_requests(case)):
        have = s // case["R"]
        unique += min(s, WINDOW + n - 1)
        if have:
            # In a layer the neighbouring tokens' scores are alike and so are their rows: at least one selection.
            unique += min(topk, have) if kind == "layer" else have * (1 - (1 - min(1.0, topk / have)) ** n)
    total["bytes"] += 2 * 2 * T * H * D + 4 * T * topk + int(unique) * D * 2
    total["bytes"] += 4 * T * H if kind == "layer" or case["lse"] else 0
    total["flops"] = 4 * H * D * rows
    return total


def tolerance(case):
    """Four times the error against float64 that the 16-bit storage of the inputs' products and outputs was measured
    to leave: bf16 2.0e-3 to 2.6e-3 (single values up to 3.9e-2), f16 2.6e-4 to 3.3e-4 (4.2e-3)."""
    kind = case["kind"]
    if kind == "topk":
        return "exact"
    bf16 = kind != "simple" and case["dtype"] == "bf16"
    return {"rel": 1.0e-2, "max": 1.5e-1} if bf16 else {"rel": 1.3e-3, "max": 1.7e-2}


# ---- the same results in float64 --------------------------------------------------


def _exact_topk(scores, limits, topk):
    """Positions of the topk largest of each row's first limits[t] scores, ties to the lower one, ascending, -1 after."""
    T, C = scores.shape
    position = torch.arange(C, device=scores.device)
    out = torch.full((T, 1, topk), -1, dtype=torch.int32, device=scores.device)
    limit = torch.tensor(limits, device=scores.device).view(-1, 1)
    k = min(topk, C)
    step = max(1, 2 ** 25 // C)
    for t in range(0, T, step):
        lim = limit[t:t + step]
        value = scores[t:t + step].double().masked_fill(position >= lim, -math.inf)
        index = value.sort(dim=1, descending=True, stable=True).indices[:, :k]
        index = index.masked_fill(index >= lim, C).sort(dim=1).values
        out[t:t + step, 0, :k] = index.masked_fill(index == C, -1).to(torch.int32)
    return out


def _exact_mla(case, t, indices, want_lse):
    T, H, D = t["q"].shape
    device = t["q"].device
    R = case["R"]
    request, right, limits = (torch.tensor(x, device=device) for x in _bounds(case))
    ori, cmp = t["ori_kv"].view(-1, D), t["cmp_kv"].view(-1, D)
    out = torch.empty((T, H, D), dtype=torch.float64, device=device)
    lse = torch.empty((T, H), dtype=torch.float64, device=device)
    slots = torch.arange(WINDOW, device=device)
    step = 64
    for a in range(0, T, step):
        b, r, lim = request[a:a + step, None], right[a:a + step, None], limits[a:a + step, None]
        visible = r.clamp(max=WINDOW)
        position = (r - visible + slots).clamp(min=0)
        in_window = slots < visible
        position = position.masked_fill(~in_window, 0)
        window = t["ori_block_table"][b, position // PAGE].long() * PAGE + position % PAGE
        index = indices[a:a + step, 0].long()
        chosen = (index >= 0) & (index < lim)
        index = index.masked_fill(~chosen, 0)
        page = PAGE // R
        compressed = t["cmp_block_table"][b, index // page].long() * page + index % page
        kv = torch.cat([ori[window], cmp[compressed]], dim=1).double()
        used = torch.cat([in_window, chosen], dim=1)[:, None, :]
        s = torch.matmul(t["q"][a:a + step].double(), kv.transpose(1, 2).contiguous()) * D ** -0.5
        s = s.masked_fill(~used, -math.inf)
        sink = t["sinks"].double()[None, :, None].expand(s.shape[0], H, 1)
        total = torch.logsumexp(torch.cat([s, sink], dim=2), dim=2)
        out[a:a + step] = torch.matmul(torch.exp(s - total[..., None]), kv)
        lse[a:a + step] = total
    return (out, lse) if want_lse else out


def exact(case, seed):
    kind = case["kind"]
    if work(case)["flops"] > 1.3e12:
        return None
    state = prepare(case, seed)
    if kind in ("topk", "layer"):
        indices = _exact_topk(state["scores"], _bounds(case)[2], state["topk"])
        if kind == "topk":
            return indices
        out, lse = _exact_mla(case, state["t"], indices, True)
        return indices, out, lse
    if kind == "mla":
        return _exact_mla(case, state["t"], state["t"]["cmp_sparse_indices"], case["lse"])
    q, k, v = state["args"][:3]
    if kind == "simple":
        q, k, v, causal = q[None], k[None], v[None], False
    else:
        causal = case["causal"]
    B, HQ, Sq, D = q.shape
    group = HQ // k.shape[1]
    out = torch.empty(q.shape, dtype=torch.float64, device=q.device)
    key = torch.arange(k.shape[2], device=q.device)
    for b in range(B):
        for h in range(HQ):
            kt = k[b, h // group].double().t().contiguous()
            vd = v[b, h // group].double()
            for i in range(0, Sq, 2048):
                s = (q[b, h, i:i + 2048].double() @ kt) * D ** -0.5
                if causal:
                    row = torch.arange(i, i + s.shape[0], device=q.device)[:, None]
                    s = s.masked_fill(key > row, -math.inf)
                out[b, h, i:i + 2048] = torch.softmax(s, dim=1) @ vd
    return out[0] if kind == "simple" else out

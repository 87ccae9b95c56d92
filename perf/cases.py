"""Performance cases of the DSA framework: what its users have it do, through
the public entry points of ``dsa_amd``.

Attention cases call ``kernel(q_nope, q_pe, ckv_cache, kpe_cache,
sparse_indices, sm_scale)`` on a paged bf16 latent cache; indexer cases select
the top-k cache slots of every query token of a sequence, over a flat fp8 K
cache, a paged one, or K operand planes kept beside the cache; the pipeline
case is one whole sparse-attention step.  Sizes are those of the repository's
workloads (``dsa_amd.workloads``), tests and benchmark, and their neighbours.

A case is a dict:
  path      "attention", "indexer" or "pipeline"
  T         query tokens of the call
  heads     attention heads (attention, pipeline)
  topk      selected positions per token
  context   "decode": every token is another sequence with a context length
            drawn from [1024, positions]; "prefill": token i is position
            positions - T + i of one sequence; "whole": every token sees all
            positions
  positions cache positions in reach (the longest context)
  page      cache page size
  index_heads, k_source ("flat", "paged", "planes"), full_range (indexer,
            pipeline): full_range codes use the whole e4m3 range, as
            quantisation by a row's largest magnitude makes them (k_append
            for K, the same rule per head for q with its scale folded into the
            head's weight); otherwise they are N(0, 1) values cast
  append    the step writes its own T rows of K to the paged cache first
"""
from __future__ import annotations

import math
import os
import sys

import torch

# the package of the tree that is the working folder
_PKG = os.path.join(os.getcwd(), "flashinfer-repo_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

DEV = "cuda:0"
SM_SCALE = 1.0 / math.sqrt(192.0)
CKV, KPE, DIM = 512, 64, 128


def _attention(name, T, heads, topk, context, positions, page=64, outliers=False):
    return {"name": name, "path": "attention", "T": T, "heads": heads, "topk": topk,
            "context": context, "positions": positions, "page": page, "outliers": outliers}


def _indexer(name, T, topk, positions, index_heads=64, k_source="flat", full_range=False,
             append=False, page=64):
    return {"name": name, "path": "indexer", "T": T, "topk": topk, "context": "prefill",
            "positions": positions, "page": page, "index_heads": index_heads,
            "k_source": k_source, "full_range": full_range, "append": append}


def listed():
    return [
        # one sequence decoding alone, 16 heads (128 heads over 8 GPUs), a big cache:
        # the latency a single user sees
        _attention("attn_t1", 1, 16, 2048, "whole", 8462 * 64),
        # a small batch with a short selection over an unpaged cache: launches and host time
        _attention("attn_t4_k256", 4, 16, 256, "decode", 4096, page=1),
        # the decode batch of a serving loop
        _attention("attn_t64", 64, 16, 2048, "decode", 131072),
        # a small decode batch with all 128 heads on one GPU
        _attention("attn_t13_h128", 13, 128, 2048, "decode", 131072),
        # a ragged chunk of prompt tokens in a mixed batch
        _attention("attn_t300", 300, 16, 2048, "prefill", 20011),
        # a long prompt's later chunk
        _attention("attn_prefill_t2048", 2048, 16, 2048, "prefill", 34816),
        # a prompt's first chunk, all heads on one GPU: every token sees few positions, the
        # selection is mostly padding
        _attention("attn_prefill_start_h128", 1023, 128, 2048, "prefill", 1023),
        # a large batch with all heads, cache rows with outliers
        _attention("attn_t256_h128", 256, 128, 2048, "whole", 65536, outliers=True),
        # a few draft tokens after a long context: append their K, refresh its planes, select
        _indexer("index_decode_131k", 2, 2048, 131071, k_source="planes", full_range=True,
                 append=True),
        # a short sequence, fewer index heads, K as it lies in a flat cache
        _indexer("index_t3_s2500", 3, 512, 2500, index_heads=32),
        # a prompt chunk: append its K to the paged cache, select from the whole context
        _indexer("index_prefill_t1024", 1024, 2048, 16384, k_source="paged", full_range=True,
                 append=True),
        # one whole step: indexer over prepared K planes, top-k slots, attention
        {"name": "pipeline_t64", "path": "pipeline", "T": 64, "heads": 16, "topk": 2048,
         "context": "prefill", "positions": 32768, "page": 64, "index_heads": 64,
         "k_source": "planes", "full_range": False, "append": False, "outliers": False},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.random()
    if kind < 0.5:
        heads = rng.choice([16, 16, 32, 48, 64, 128])
        topk = rng.choice([256, 1000, 2048, 2048, 2048])
        T = _log(rng, 1, 32768 // heads)  # 2048 tokens of 16 heads, 256 of 128
        context = rng.choice(["decode", "prefill", "whole"])
        positions = _log(rng, max(1024, T), 131072)
        if T > 64:  # the inputs of a large draw stay quick to make
            positions = max(T, min(positions, 40000))
        c = _attention("", T, heads, topk, context, positions, page=rng.choice([1, 64, 64]),
                       outliers=rng.random() < 0.25)
    else:
        T = _log(rng, 1, 1024)
        positions = _log(rng, max(1024, T), 131072)
        while T * positions > 1024 * 16384:
            T = max(1, T // 2)
        src = rng.choice(["flat", "paged", "planes"])
        c = _indexer("", T, rng.choice([512, 2048, 2048]), positions,
                     index_heads=rng.choice([16, 32, 64, 64]), k_source=src,
                     full_range=rng.random() < 0.5, append=src != "flat" and rng.random() < 0.5)
        if kind > 0.85 and T <= 64:
            c.update(path="pipeline", heads=rng.choice([16, 32, 128]), outliers=False)
    c.pop("name")
    return c


# ---- inputs ---------------------------------------------------------------

def _gen(seed):
    g = torch.Generator(device=DEV)
    g.manual_seed(int(seed) & 0x7FFFFFFF)
    return g


def _limits(case, g):
    """Positions every token sees (its context length), int64 [T]."""
    T, P = case["T"], case["positions"]
    if case["context"] == "decode":
        return torch.randint(min(1024, P), P + 1, (T,), generator=g, device=DEV)
    if case["context"] == "prefill":
        return P - T + 1 + torch.arange(T, device=DEV)
    return torch.full((T,), P, dtype=torch.int64, device=DEV)


def _selection(case, g):
    """A selection as the indexer hands it on: per token min(topk, context)
    distinct positions in ascending order, then -1; int64 [T, topk]."""
    T, K, P = case["T"], case["topk"], case["positions"]
    n = _limits(case, g)
    pos = torch.full((T, K), -1, dtype=torch.int64, device=DEV)
    k = min(K, P)
    rows = max(1, (1 << 26) // P)
    col = torch.arange(P, device=DEV)
    for a in range(0, T, rows):
        b = min(T, a + rows)
        r = torch.rand((b - a, P), generator=g, device=DEV)
        r = torch.where(col[None] < n[a:b, None], r, torch.full_like(r, -1.0))
        v, i = torch.topk(r, k, dim=1)
        i = torch.where(v >= 0, i, torch.full_like(i, 1 << 40)).sort(dim=1).values
        pos[a:b, :k] = torch.where(i < (1 << 40), i, torch.full_like(i, -1))
    return pos


def _pages(case):
    return -(-case["positions"] // case["page"])


def _cache(case, g):
    pages, ps = _pages(case), case["page"]
    ckv = torch.randn((pages * ps, CKV), generator=g, device=DEV) * math.sqrt(0.5)
    kpe = torch.randn((pages * ps, KPE), generator=g, device=DEV) * math.sqrt(0.5)
    if case["outliers"]:  # one row in twenty, eight times as large
        big = torch.rand((pages * ps, 1), generator=g, device=DEV) < 0.05
        ckv = torch.where(big, ckv * 8, ckv)
        kpe = torch.where(big, kpe * 8, kpe)
    return (ckv.to(torch.bfloat16).view(pages, ps, CKV), kpe.to(torch.bfloat16).view(pages, ps, KPE))


def _queries(case, g):
    T, H = case["T"], case["heads"]
    return (torch.randn((T, H, CKV), generator=g, device=DEV).to(torch.bfloat16),
            torch.randn((T, H, KPE), generator=g, device=DEV).to(torch.bfloat16))


def _e4m3(x):
    return x.to(torch.float8_e4m3fn).view(torch.uint8)


def _quantise(x):
    """(codes, scale) of rows by their largest magnitude, as k_append makes them."""
    scale = x.float().abs().amax(-1, keepdim=True).clamp_min(1e-4) / 448.0
    return _e4m3((x.float() / scale).clamp(-448.0, 448.0)), scale.squeeze(-1)


def _index_inputs(case, g):
    """The indexer's inputs before any of this framework's formats: q codes,
    weights, limits, bf16 K rows (or codes and scales), block table."""
    T, Hi, P = case["T"], case["index_heads"], case["positions"]
    q = torch.randn((T, Hi, DIM), generator=g, device=DEV)
    w = torch.randn((T, Hi), generator=g, device=DEV) * math.sqrt(1.0 / 8.0)
    if case["full_range"]:
        qc, qs = _quantise(q)
        w = w * qs
        k = torch.randn((P, DIM), generator=g, device=DEV).to(torch.bfloat16)
        kc, ks = _quantise(k)
    else:
        qc = _e4m3(q)
        k = None
        kc = _e4m3(torch.randn((P, DIM), generator=g, device=DEV))
        ks = torch.rand((P,), generator=g, device=DEV) * 1.5 + 0.5
    limit = (_limits(case, g) - 1).to(torch.int32)
    table = torch.randperm(_pages(case), generator=g, device=DEV).to(torch.int32)
    return {"q": qc, "w": w, "limit": limit, "k": k, "kc": kc, "ks": ks, "table": table}


def _filled_cache(case, kc, ks, table):
    """A paged fp8 K cache holding every position at the page the table names
    (the documented format: a page's codes, then its fp32 scales)."""
    P, ps, pages = case["positions"], case["page"], _pages(case)
    codes = torch.zeros((pages * ps, DIM), dtype=torch.uint8, device=DEV)
    scale = torch.zeros((pages * ps,), dtype=torch.float32, device=DEV)
    pos = torch.arange(P, device=DEV)
    slot = table.long()[pos // ps] * ps + pos % ps
    codes[slot], scale[slot] = kc, ks
    return torch.cat([codes.view(pages, ps * DIM), scale.view(pages, ps).view(torch.uint8)],
                     dim=1).contiguous()


def prepare(case, seed):
    import dsa_amd
    g = _gen(seed)
    st = {"case": case, "dsa": dsa_amd}
    if case["path"] == "attention":
        pos = _selection(case, g)
        ps = case["page"]
        table = torch.randperm(_pages(case), generator=g, device=DEV)
        p = pos.clamp_min(0)
        slot = table[p // ps] * ps + p % ps
        st["slots"] = torch.where(pos >= 0, slot, torch.full_like(slot, -1)).to(torch.int32)
        st["ckv"], st["kpe"] = _cache(case, g)
        st["qn"], st["qp"] = _queries(case, g)
        return st
    x = _index_inputs(case, g)
    st.update(x)
    if case["k_source"] != "flat":
        st["cache"] = _filled_cache(case, x["kc"], x["ks"], x["table"])
    if case["k_source"] == "planes":
        st["planes"] = dsa_amd.prepare_k_paged(st["cache"], x["table"], case["positions"])
    if case["append"]:
        P, T, ps = case["positions"], case["T"], case["page"]
        pos = torch.arange(P - T, P, device=DEV)
        st["new_slots"] = (x["table"].long()[pos // ps] * ps + pos % ps).to(torch.int32)
        rows = x["k"][P - T:] if x["k"] is not None else None
        if rows is None:
            rows = torch.randn((T, DIM), generator=g, device=DEV).to(torch.bfloat16)
        st["new_k"] = rows.contiguous()
    if case["path"] == "pipeline":
        st["ckv"], st["kpe"] = _cache(case, g)
        st["qn"], st["qp"] = _queries(case, g)
    return st


def run(st):
    case, dsa = st["case"], st["dsa"]
    if case["path"] == "attention":
        return dsa.kernel(st["qn"], st["qp"], st["ckv"], st["kpe"], st["slots"], SM_SCALE)
    P, T, src = case["positions"], case["T"], case["k_source"]
    if case["append"]:
        dsa.k_append(st["new_k"], st["new_slots"], st["cache"])
        if src == "planes":
            dsa.prepare_k_paged(st["cache"], st["table"], P, st["planes"], first_position=P - T)
    if case["path"] == "pipeline":
        k = {"planes": {"k_planes": st.get("planes")},
             "paged": {"k_cache": st.get("cache"), "num_positions": P}, "flat": {}}[src]
        flat = src == "flat"
        return dsa.run_sparse_attention_pipeline(
            st["q"], st["kc"] if flat else None, st["ks"] if flat else None, st["w"], st["limit"],
            st["table"], st["qn"], st["qp"], st["ckv"], st["kpe"], SM_SCALE, topk=case["topk"], **k)
    if src == "planes":
        out = dsa.run_indexer_and_topk(st["q"], None, None, st["w"], st["limit"], case["topk"],
                                       block_table=st["table"], page_size=case["page"],
                                       k_planes=st["planes"])
    elif src == "paged":
        out = dsa.run_indexer_and_topk_paged(st["q"], st["cache"], st["table"], P, st["w"],
                                             st["limit"], case["topk"], block_table=st["table"],
                                             page_size=case["page"])
    else:
        out = dsa.run_indexer_and_topk(st["q"], st["kc"], st["ks"], st["w"], st["limit"],
                                       case["topk"], block_table=st["table"],
                                       page_size=case["page"])
    return (out, st["cache"]) if case["append"] else out


# ---- what a pass cannot do without ----------------------------------------

def _expected_rows(case):
    """Sum over tokens of the positions to score (none where all in reach are
    selected), and of the selected ones."""
    T, P, K = case["T"], case["positions"], case["topk"]
    if case["context"] == "prefill":
        n = [P - T + 1 + i for i in range(T)]
    elif case["context"] == "decode":  # lengths are uniform: their mean
        lo = min(1024, P)
        sel = sum(min(x, K) for x in range(lo, P + 1, max(1, (P - lo) // 1000)))
        cnt = len(range(lo, P + 1, max(1, (P - lo) // 1000)))
        return T * (lo + P) / 2, T * sel / cnt  # (attention only: nothing is scored)
    else:
        n = [P] * T
    return float(sum(x for x in n if x > K)), float(sum(min(x, K) for x in n))


def work(case):
    T, P, K = case["T"], case["positions"], case["topk"]
    seen, selected = _expected_rows(case)
    nbytes = flops = 0.0
    if case["path"] != "attention":
        Hi = case["index_heads"]
        nbytes += T * Hi * (DIM + 4) + P * (DIM + 4) + T * K * 4
        flops += seen * Hi * (2 * DIM + 3)
        if case["append"]:
            nbytes += T * (2 * DIM + DIM + 4)
    if case["path"] != "indexer":
        H = case["heads"]
        rows = min(selected, float(P))  # each cache row once
        nbytes += rows * (CKV + KPE) * 2 + T * H * (CKV + KPE + CKV) * 2 + T * H * 4 + T * K * 4
        flops += selected * 2 * H * (CKV + KPE + CKV)
    return {"bytes": nbytes, "flops": flops}


def tolerance(case):
    # Slots and cache bytes are whole numbers.  Attention outputs are bf16 rounded from fp32
    # sums: 1.5e-3 to 1.7e-3 from the 64-bit result (measured), one value at most one
    # rounding (2^-8) from another implementation's.
    if case["path"] == "indexer":
        return "exact"
    return {"rel": 7e-3, "max": 0.03}


# ---- the same in 64 bits --------------------------------------------------

def _exact_slots(case, x):
    """The selection the score's definition gives: exact dots, fp32 rounding
    of every dot and of the weighted sum in the documented order, ties to the
    lower position, ascending, -1 padded."""
    T, P, K, Hi, ps = case["T"], case["positions"], case["topk"], case["index_heads"], case["page"]
    k = x["kc"].view(torch.float8_e4m3fn).double() * 512.0
    cs = (x["ks"] * 2.0 ** -18).float()
    lim = x["limit"].long()
    out = torch.full((T, K), -1, dtype=torch.int32, device=DEV)
    rows = max(1, (1 << 24) // P)
    col = torch.arange(P, device=DEV)
    for a in range(0, T, rows):
        b = min(T, a + rows)
        q = x["q"][a:b].view(torch.float8_e4m3fn).double() * 512.0
        G = []
        for g in range(4):
            acc = torch.zeros((b - a, P), dtype=torch.float32, device=DEV)
            for h in range(g * Hi // 4, (g + 1) * Hi // 4):
                r = (q[:, h] @ k.t()).clamp_min(0.0).float()
                acc = (x["w"][a:b, h, None].double() * r.double() + acc.double()).float()
            G.append(acc)
        s = ((G[0] + G[1]) + (G[2] + G[3])) * cs[None]
        s = torch.where(col[None] <= lim[a:b, None], s, torch.full_like(s, -math.inf))
        order = torch.sort(s, dim=1, descending=True, stable=True).indices[:, :K]
        valid = order <= lim[a:b, None]
        pos = torch.where(valid, order, torch.full_like(order, 1 << 40)).sort(dim=1).values
        p = torch.where(pos < (1 << 40), pos, torch.zeros_like(pos))
        slot = x["table"].long()[p // ps] * ps + p % ps
        n = pos.shape[1]
        out[a:b, :n] = torch.where(pos < (1 << 40), slot, torch.full_like(slot, -1)).to(torch.int32)
    return out


def _exact_attention(st, slots):
    H = st["qn"].shape[1]
    T = slots.shape[0]
    ckv = st["ckv"].reshape(-1, CKV)
    kpe = st["kpe"].reshape(-1, KPE)
    out = torch.empty((T, H, CKV), dtype=torch.float64, device=DEV)
    lse = torch.empty((T, H), dtype=torch.float64, device=DEV)
    for a in range(0, T, 16):
        b = min(T, a + 16)
        s = slots[a:b].long()
        ok = s >= 0
        i = s.clamp_min(0)
        kc, kp = ckv[i].double(), kpe[i].double()
        x = torch.matmul(st["qn"][a:b].double(), kc.transpose(1, 2).contiguous())
        x = x + torch.matmul(st["qp"][a:b].double(), kp.transpose(1, 2).contiguous())
        x = (x * SM_SCALE).masked_fill(~ok[:, None], -math.inf)
        l = torch.logsumexp(x, dim=2)
        out[a:b] = torch.matmul(torch.exp(x - l[..., None]), kc)
        lse[a:b] = l / math.log(2.0)
    return out, lse


def exact(case, seed):
    st = prepare(case, seed)
    if case["path"] == "attention":
        return _exact_attention(st, st["slots"])
    x = {k: st[k] for k in ("q", "w", "limit", "kc", "ks", "table")}
    if case["append"]:
        P, T = case["positions"], case["T"]
        kc, ks = _quantise(st["new_k"])
        x["kc"], x["ks"] = x["kc"].clone(), x["ks"].clone()
        x["kc"][P - T:], x["ks"][P - T:] = kc, ks
    slots = _exact_slots(case, x)
    if case["path"] == "pipeline":
        out, lse = _exact_attention(st, slots)
        return out, lse, slots
    if case["append"]:
        return slots, _filled_cache(case, x["kc"], x["ks"], x["table"])
    return slots

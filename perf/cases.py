"""The work a program has this library do, as cases that can be timed and checked.

Every case is one call (or the short run of calls a program makes in one place)
through the public entry points of ``qwfnfer_amd.qsa``, over caches filled as an
engine fills them.  Shapes are the ones of the tests and of ``bench.py``: the
16 x 128 query / 2 KV head layer with 64-token blocks, and the released
checkpoint's layer (24 x 256, 4-token blocks, an indexer of its own).

K/V rows are N(0, 1) with a log-uniform [0.1, 10] scale a 32-value block and
queries N(0, 1), the draw of ``bench.py`` and the tests.
"""
from __future__ import annotations

import math
import random

import numpy as np
import torch

from qwfnfer_amd import qsa

Q8_0, Q4_0, F16 = 0, 1, 2
TYPE_BYTES = {Q8_0: 34 / 32, Q4_0: 18 / 32, F16: 2.0}        # a cached value

CHUNK = 32768                                                # rows a fill appends at a time


# ---- the cases -------------------------------------------------------------

def _decode(name=None, longest=4096, shortest=None, n_seq=1, kv=Q8_0, dense=False, f16=False, spread=0):
    return _named(name, path="decode", longest=longest, shortest=shortest or longest, n_seq=n_seq, kv=kv,
                  dense=dense, f16=f16, spread=spread)


def _chain(name=None, longest=4096, shortest=None, n_seq=1, n_pos=4, f16=False, spread=0):
    return _named(name, path="chain", longest=longest, shortest=shortest or longest, n_seq=n_seq, kv=Q8_0,
                  dense=False, n_pos=n_pos, f16=f16, spread=spread)


def _prefill(name=None, pos0=0, n_q=1024, kv=Q8_0, dense=False, f16=True):
    return _named(name, path="prefill", pos0=pos0, n_q=n_q, kv=kv, dense=dense, f16=f16)


def _ckpt_decode(name=None, longest=4096, shortest=None, n_seq=1, f16=False, spread=0):
    return _named(name, path="ckpt_decode", longest=longest, shortest=shortest or longest, n_seq=n_seq, kv=Q8_0,
                  dense=False, f16=f16, spread=spread)


def _ckpt_prefill(name=None, pos0=0, n_q=1024, f16=True):
    return _named(name, path="ckpt_prefill", pos0=pos0, n_q=n_q, kv=Q8_0, dense=False, f16=f16)


def _session(name=None, n_tokens=4096, kv=Q8_0):
    return _named(name, path="session", n_tokens=n_tokens, kv=kv)


def _named(name, **case):
    return dict(case, name=name) if name else case


def listed():
    return [
        # one token of a chat at a short context: the smallest call, all latency
        _decode("decode_4k", longest=4096),
        # the same at the longest context of the benchmark
        _decode("decode_160k", longest=163840),
        # the benchmark's batch: eight paged sequences, short to very long
        _decode("decode_batch8", longest=262144, shortest=4096, n_seq=8, f16=True, spread=5),
        # a server's batch: many sequences of ordinary, ragged lengths
        _decode("decode_batch32", longest=40000, shortest=1000, n_seq=32, f16=True, spread=7),
        # the dense layer over an fp16 cache (selection switched off)
        _decode("decode_dense_f16", longest=16001, kv=F16, dense=True),
        # speculative decoding: four positions verified in one call
        _chain("chain_verify4", longest=32771, n_pos=4),
        # a prompt read from nothing, of no round length
        _prefill("prefill_prompt", pos0=0, n_q=3001),
        # a user's turn of a long chat: few new tokens over a long cache
        _prefill("prefill_turn", pos0=32700, n_q=203),
        # a chunk of a very long document: the benchmark's prefill chunk
        _prefill("prefill_chunk", pos0=155648, n_q=8192),
        # the released checkpoint's layer: a token at the longest context
        _ckpt_decode("ckpt_decode_160k", longest=163840),
        # the released checkpoint's layer: a document's chunk
        _ckpt_prefill("ckpt_prefill", pos0=40003, n_q=1900),
        # a saved session: its rows read in, pooled and written out again
        _session("session_rows", n_tokens=65537),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    path = rng.choice(["decode", "decode", "decode", "chain", "prefill", "prefill", "prefill", "ckpt_decode",
                       "ckpt_prefill", "session"])
    spread, f16 = rng.randrange(1000), rng.random() < 0.5
    if path == "decode":
        n_seq = rng.choice([1, 1, _log(rng, 2, 32)])
        dense = rng.random() < 0.25
        longest = _log(rng, 200, (32768 if dense else 163840) // (1 if n_seq <= 8 else 4))
        return _decode(longest=longest, shortest=max(1, longest // rng.choice([1, 8, 64])), n_seq=n_seq,
                       kv=rng.choice([Q8_0, Q8_0, Q4_0, F16]), dense=dense, f16=f16, spread=spread)
    if path == "chain":
        longest = _log(rng, 300, 163840)
        return _chain(longest=longest, shortest=max(1, longest // rng.choice([1, 8])), n_seq=rng.choice([1, 1, 2, 4]),
                      n_pos=rng.randint(2, 8), f16=f16, spread=spread)
    if path == "prefill":
        kv, dense = rng.choice([Q8_0, Q8_0, Q8_0, Q4_0, F16]), rng.random() < 0.15
        n_q = _log(rng, 16, 8192 if kv == Q8_0 and not dense else 3000)
        pos0 = rng.choice([0, _log(rng, 100, 9000 if dense else 155000)])
        return _prefill(pos0=pos0, n_q=n_q, kv=kv, dense=dense, f16=f16)
    if path == "ckpt_decode":
        longest = _log(rng, 300, 163840)
        return _ckpt_decode(longest=longest, shortest=max(1, longest // rng.choice([1, 8])),
                            n_seq=rng.choice([1, 1, 2, 5, 8]), f16=f16, spread=spread)
    if path == "ckpt_prefill":
        return _ckpt_prefill(pos0=rng.choice([0, _log(rng, 100, 155000)]), n_q=_log(rng, 16, 2600), f16=f16)
    return _session(n_tokens=_log(rng, 300, 163840), kv=rng.choice([Q8_0, Q8_0, Q4_0, F16]))


# ---- geometry of a case ----------------------------------------------------

def _cfg(case):
    if case["path"].startswith("ckpt"):
        return qsa.checkpoint_config()
    cfg = qsa.QsaConfig(kv_type=case["kv"])
    return cfg.dense() if case.get("dense") else cfg


def _lengths(case):
    """Tokens of each sequence, the one being decoded among them."""
    lo, hi, n = case["shortest"], case["longest"], case["n_seq"]
    r = random.Random(case["spread"])
    got = [int(round(math.exp(r.uniform(math.log(lo), math.log(hi))))) for _ in range(n)]
    got[0] = hi
    return got


def _up(x, m):
    return -(-x // m) * m


# ---- inputs ----------------------------------------------------------------

def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed))


def _rows(gen, n, cfg):
    """n rows of K (or V): N(0, 1), a log-uniform [0.1, 10] scale a 32-value block."""
    nb = cfg.head_dim // 32
    x = torch.randn((n, cfg.n_head_kv, nb, 32), device="cuda", generator=gen)
    s = torch.empty((n, cfg.n_head_kv, nb, 1), device="cuda")
    s.uniform_(math.log(0.1), math.log(10.0), generator=gen).exp_()
    return (x * s).reshape(n, cfg.n_head_kv, cfg.head_dim)


def _past(gen, length, cfg):
    """The rows of a sequence's first `length` tokens, a chunk at a time: (first, K, V)."""
    for t0 in range(0, length, CHUNK):
        n = min(CHUNK, length - t0)
        k = _rows(gen, n, cfg)
        yield t0, k, _rows(gen, n, cfg)


def _past_keys(gen, length, icfg):
    for t0 in range(0, length, CHUNK):
        yield t0, torch.randn((min(CHUNK, length - t0), icfg.idx_dim), device="cuda", generator=gen)


def _page_table(gen, n_seq, pages):
    """Pages in the order of a paged allocator that has been in use (one sequence: in order)."""
    if n_seq == 1:
        return torch.arange(pages, dtype=torch.int32).view(1, pages)
    return torch.randperm(n_seq * pages, device="cuda", generator=gen).to(torch.int32).view(n_seq, pages)


def _new(gen, case, cfg, *lead):
    """The new tokens' queries and K/V rows."""
    q = torch.randn((*lead, cfg.n_head, cfg.head_dim), device="cuda", generator=gen)
    k, v = (_rows(gen, math.prod(lead), cfg).view(*lead, cfg.n_head_kv, cfg.head_dim) for _ in range(2))
    return (q, k.half(), v.half()) if case["f16"] else (q, k.contiguous(), v.contiguous())


def _new_keys(gen, case, icfg, n):
    qi = torch.randn((n, icfg.n_idx_head, icfg.idx_dim), device="cuda", generator=gen)
    kr = torch.randn((n, icfg.idx_dim), device="cuda", generator=gen)
    return qi, kr.half() if case["f16"] else kr


def _inputs(case, seed):
    """Everything the seed draws, in one order: (past lengths, page table, generator)."""
    gen = _gen(seed)
    cfg = _cfg(case)
    if "pos0" in case:
        past, end = [case["pos0"]], [case["pos0"] + case["n_q"]]
    else:
        end = [n + case.get("n_pos", 1) - 1 for n in _lengths(case)]
        past = [n - 1 for n in _lengths(case)]
    pages = _up(max(end), cfg.page_tokens) // cfg.page_tokens
    return gen, cfg, past, pages, _page_table(gen, len(past), pages)


def _k_norm(gen, icfg):
    return torch.rand(icfg.idx_dim, device="cuda", generator=gen) + 0.5


def prepare(case, seed):
    if case["path"] == "session":
        return _prepare_session(case, seed)
    gen, cfg, past, pages, table = _inputs(case, seed)
    cache = qsa.KvCache.allocate(cfg, len(past), pages, page_table=table)
    ckpt = case["path"].startswith("ckpt")
    for s, n in enumerate(past):
        for t0, k, v in _past(gen, n, cfg):
            pos = torch.arange(t0, t0 + len(k), dtype=torch.int32, device="cuda")
            qsa.append_q8_0(cache, k, v, pos, torch.full_like(pos, s))
        if not ckpt and n // cfg.block_tokens:
            qsa.pool_rebuild(cache, s, n // cfg.block_tokens)
    state = {"case": case, "cfg": cfg, "cache": cache}
    n_seq, max_len = len(past), pages * cfg.page_tokens
    if ckpt:
        icfg = qsa.IdxConfig()
        ic = qsa.IdxCache.allocate(icfg, cache, _k_norm(gen, icfg))
        for s, n in enumerate(past):
            for t0, kr in _past_keys(gen, n, icfg):
                pos = torch.arange(t0, t0 + len(kr), dtype=torch.int32, device="cuda")
                qsa.idx_append_pool(ic, kr, pos, torch.full_like(pos, s))
        state["ic"] = ic
    if "pos0" in case:
        n_q = case["n_q"]
        state["q"], state["k"], state["v"] = _new(gen, case, cfg, n_q)
        state["ws"] = qsa.Workspace.for_prefill(cfg, case["pos0"] + n_q, n_q)
    else:
        lead = (case["n_pos"], n_seq) if case["path"] == "chain" else (n_seq,)
        state["q"], state["k"], state["v"] = _new(gen, case, cfg, *lead)
        state["seq_len"] = torch.tensor([n + 1 for n in past], dtype=torch.int32, device="cuda")
        state["max_len"] = max_len
        nbytes = cfg.workspace_bytes(n_seq, max_len)
        if ckpt:
            nbytes = max(nbytes, state["ic"].workspace_bytes(n_seq, max_len))
        state["ws"] = qsa.Workspace(cfg, n_seq, max_len, nbytes=nbytes)
        msel = cfg.max_selected(max_len)
        lead = (*lead, cfg.n_head_kv)
        state["sel"] = torch.zeros((*lead, msel), dtype=torch.int32, device="cuda")
        state["n_sel"] = torch.zeros(lead, dtype=torch.int32, device="cuda")
    if ckpt:
        state["q_idx"], state["k_raw"] = _new_keys(gen, case, state["ic"].icfg, len(state["q"]))
    state["out"] = torch.zeros_like(state["q"])
    return state


def _session_rows(case, seed):
    """A saved session's K and V rows in the engine's cache format: uint8 [tokens, row bytes]."""
    gen, cfg, n = _gen(seed), qsa.QsaConfig(kv_type=case["kv"]), case["n_tokens"]
    got = []
    for _ in range(2):
        if case["kv"] == F16:
            got.append(_rows(gen, n, cfg).half().reshape(n, -1).view(torch.uint8))
            continue
        nb, width = cfg.kv_dim // 32, 32 if case["kv"] == Q8_0 else 16
        d = torch.empty((n, nb, 1), device="cuda").uniform_(math.log(0.1), math.log(10.0), generator=gen).exp_()
        quants = torch.randint(0, 256, (n, nb, width), device="cuda", generator=gen, dtype=torch.int32)
        if case["kv"] == Q8_0:
            quants.masked_fill_(quants == 128, 127)          # -128 is no value the quantizer writes
        rows = torch.cat([(d / 42).half().view(torch.uint8), quants.to(torch.uint8)], dim=2)
        got.append(rows.reshape(n, -1).contiguous())
    return cfg, got[0], got[1]


def _prepare_session(case, seed):
    cfg, k, v = _session_rows(case, seed)
    cache = qsa.KvCache.allocate(cfg, 1, _up(case["n_tokens"], cfg.page_tokens) // cfg.page_tokens)
    return {"case": case, "cfg": cfg, "cache": cache, "k": k, "v": v}


# ---- one pass --------------------------------------------------------------

def run(s):
    path = s["case"]["path"]
    cache = s["cache"]
    if path in ("decode", "chain"):
        step = qsa.sparse_attn_decode if path == "decode" else qsa.sparse_attn_decode_chain
        step(cache, s["q"], s["k"], s["v"], s["seq_len"], s["max_len"], s["ws"], out=s["out"], sel=s["sel"],
             n_sel=s["n_sel"])
    elif path == "prefill":
        qsa.sparse_attn_prefill(cache, s["q"], 0, s["case"]["pos0"], s["ws"], s["k"], s["v"], out=s["out"])
    elif path == "ckpt_decode":
        qsa.idx_sparse_attn_decode(s["ic"], s["q"], s["q_idx"], s["k"], s["v"], s["k_raw"], s["seq_len"],
                                   s["max_len"], s["ws"], out=s["out"], sel=s["sel"], n_sel=s["n_sel"])
    elif path == "ckpt_prefill":
        qsa.idx_sparse_attn_prefill(s["ic"], s["q"], s["q_idx"], 0, s["case"]["pos0"], s["ws"], k_new=s["k"],
                                    v_new=s["v"], k_raw=s["k_raw"], out=s["out"])
    else:
        n = s["case"]["n_tokens"]
        qsa.import_rows_q8_0(cache, 0, 0, s["k"], s["v"])
        qsa.pool_rebuild(cache, 0, n // s["cfg"].block_tokens)
        k, v = qsa.export_rows_q8_0(cache, 0, 0, n)
        return {"k_rows": k, "v_rows": v, "pooled": cache.pooled, "k_pages": cache.k_pages,
                "v_pages": cache.v_pages}
    got = {"out": s["out"], "k_pages": cache.k_pages, "v_pages": cache.v_pages}
    if "sel" in s:
        got["sel"], got["n_sel"] = s["sel"], s["n_sel"]
    if "ic" in s:
        got["idx_raw"], got["idx_pooled"] = s["ic"].raw, s["ic"].pooled
    else:
        got["pooled"] = cache.pooled
    return got


# ---- what a pass cannot do without ----------------------------------------

def _kept(cfg, length):
    """(cells attended, blocks scored) a query head group of a sequence of `length` tokens."""
    bt = cfg.block_tokens
    nb = (length - 1) // bt + 1
    fw = max(0, length - cfg.local_tokens) // bt
    if not cfg.top_k_blocks:
        return length, 0
    forced = sum(1 for b in range(min(cfg.sink_blocks, nb)) if b < fw) + nb - fw
    eligible = max(0, fw - cfg.sink_blocks)
    k = cfg.top_k_blocks - (forced if cfg.topk_counts_forced else 0)
    if eligible <= k:
        return length, 0
    return length - (eligible - k) * bt, eligible


def work(case):
    if case["path"] == "session":
        cfg = qsa.QsaConfig(kv_type=case["kv"])
        rows = 2 * case["n_tokens"] * cfg.kv_dim * TYPE_BYTES[case["kv"]]
        # rows into pages, pages into rows, and the pooled keys of the whole blocks
        return {"bytes": 4 * rows + case["n_tokens"] // cfg.block_tokens * cfg.kv_dim * 4,
                "flops": case["n_tokens"] * cfg.kv_dim}
    cfg = _cfg(case)
    ckpt = case["path"].startswith("ckpt")
    icfg = qsa.IdxConfig()
    row = cfg.kv_dim * TYPE_BYTES[case["kv"]] * 2
    if "pos0" in case:
        ends = [case["pos0"] + i + 1 for i in range(case["n_q"])]
        kept = [_kept(cfg, n) for n in ends]
        cells, scored = sum(c for c, _ in kept), sum(b for _, b in kept)
        read = min(cells, ends[-1]) * row
        pooled = max(b for _, b in kept)
    else:
        kept = [_kept(cfg, n + k) for k in range(case.get("n_pos", 1)) for n in _lengths(case)]
        cells, scored = sum(c for c, _ in kept), sum(b for _, b in kept)
        read, pooled, ends = cells * row, scored, kept
    new = len(ends)
    key_bytes, score_flops = cfg.kv_dim * 4, cfg.n_head * cfg.head_dim * 2
    if ckpt:
        key_bytes, score_flops = icfg.idx_dim * 2, icfg.n_idx_head * icfg.idx_dim * 2
    src = 2 if case["f16"] else 4
    moved = new * (cfg.n_head * cfg.head_dim * 8 + 2 * cfg.kv_dim * src + row)
    return {"bytes": read + pooled * key_bytes + moved,
            "flops": cells * cfg.n_head * cfg.head_dim * 4 + scored * score_flops}


def tolerance(case):
    # float32 sums of exact products: 3e-7 to 8e-7 off the 64-bit result over these ranges; cache
    # bytes and selections are whole numbers and stay
    return {"rel": 3e-6, "max": 1e-4, "differ": 0.0}


# ---- the same in 64 bits ---------------------------------------------------

def _cached(x, kv):
    """The values a cache of this type holds of rows x, in float64."""
    if kv == F16:
        return x.half().double()
    b = x.float().unflatten(-1, (-1, 32))
    if kv == Q8_0:
        amax = b.abs().amax(-1, keepdim=True)
        top = torch.full_like(amax, 127.0)              # a tensor: torch divides by one exactly, by a number not
        d, inv = amax / top, torch.where(amax > 0, top / amax, torch.zeros_like(amax))
        quants = torch.round(b * inv)
    else:
        m = b.gather(-1, b.abs().argmax(-1, keepdim=True))
        d = m / -8.0
        inv = torch.where(d != 0, torch.ones_like(d) / d, torch.zeros_like(d))
        quants = torch.clamp_max(torch.trunc(b * inv + 8.5), 15.0) - 8.0
    return (quants.double() * d.half().double()).flatten(-2)


def _keep(cfg, scores, lengths):
    """Kept blocks of queries with these block scores [n, blocks]: (block ids [n, most], valid [n, most])."""
    n, nb = scores.shape
    bt = cfg.block_tokens
    b = torch.arange(nb, device=scores.device)
    last = (lengths - 1)[:, None] // bt
    fw = torch.clamp_min(lengths - cfg.local_tokens, 0)[:, None] // bt
    forced = (b < cfg.sink_blocks) | (b >= fw)
    if not cfg.top_k_blocks:
        forced |= True
    forced &= b <= last
    eligible = (b <= last) & ~forced
    k = torch.full((n, 1), cfg.top_k_blocks, device=scores.device)
    if cfg.topk_counts_forced:
        k = k - forced.sum(1, keepdim=True)
    keep = forced
    if cfg.top_k_blocks:
        order = torch.sort(scores.masked_fill(~eligible, -math.inf), dim=1, descending=True, stable=True).indices
        rank = torch.empty_like(order).scatter_(1, order, b.expand(n, nb).contiguous())
        keep = forced | (eligible & (rank < k))
    most = int(keep.sum(1).max())
    ids = torch.sort(keep.to(torch.int8), dim=1, descending=True, stable=True).indices[:, :most]
    return ids, keep.gather(1, ids)


def _attend(cfg, q, K, V, ids, valid, lengths):
    """Softmax attention of q [n, group, hd] over the kept blocks of K, V [blocks, bt, hd]."""
    n, bt = q.shape[0], cfg.block_tokens
    cells = ids[:, :, None] * bt + torch.arange(bt, device=q.device)
    seen = (valid[:, :, None] & (cells < lengths[:, None, None])).flatten(1)
    k, v = K[ids].view(n, -1, cfg.head_dim), V[ids].view(n, -1, cfg.head_dim)
    logits = torch.bmm(q, k.transpose(1, 2).contiguous()) / math.sqrt(cfg.head_dim)
    p = torch.softmax(logits.masked_fill(~seen[:, None], -math.inf), dim=-1)
    return torch.bmm(p, v)


def _blocks(cfg, x):
    """Rows [n, heads, hd] as whole blocks [heads, blocks, bt, hd], the last one padded with zeros."""
    n, bt = x.shape[0], cfg.block_tokens
    x = torch.cat([x, x.new_zeros(_up(n, bt) - n, *x.shape[1:])]).transpose(0, 1)
    return x.reshape(x.shape[0], -1, bt, x.shape[-1])


def _idx_pooled(icfg, cfg, raw, k_norm):
    """The pooled indexer keys of fp16 rows [n, dim]: mean, RMSNorm, rotation at the block's first token, fp16."""
    bt, half = cfg.block_tokens, icfg.rope_dim // 2
    n = raw.shape[0]
    x = torch.cat([raw, raw.new_zeros(_up(n, bt) - n, icfg.idx_dim)]).double().view(-1, bt, icfg.idx_dim).mean(1)
    y = x / torch.sqrt(x.square().mean(1, keepdim=True) + icfg.rms_eps) * k_norm.double()
    # the angle is the format's own: a running fp32 product, one factor a pair
    theta = np.empty((len(y), half), np.float32)
    step = np.float32(np.float32(icfg.rope_freq_base) ** np.float32(-2.0 / icfg.rope_dim))
    theta[:, 0] = np.arange(len(y), dtype=np.int64) * bt
    for i in range(1, half):
        theta[:, i] = theta[:, i - 1] * step
    a = torch.from_numpy(theta).to(y.device).double()
    c, s = a.cos(), a.sin()
    lo, hi = y[:, :half], y[:, half:icfg.rope_dim]
    return torch.cat([lo * c - hi * s, lo * s + hi * c, y[:, icfg.rope_dim:]], 1).half().double()


def _exact_queries(cfg, q, K, V, lengths, pool, q_score, relu, chunk=64):
    """Attention of queries q [n, heads, hd] of one sequence, query i seeing lengths[i] tokens.

    pool [score heads, blocks, dim] and q_score [n, score heads * group, dim] give the block scores."""
    group = cfg.n_head // cfg.n_head_kv
    Kb, Vb = _blocks(cfg, K), _blocks(cfg, V)
    nb, out = Kb.shape[1], torch.empty_like(q)
    for i in range(0, len(q), chunk):
        at, L = slice(i, i + chunk), lengths[i:i + chunk]
        kept = []
        for g in range(pool.shape[0]):
            qs = q_score[at].view(len(L), pool.shape[0], -1, pool.shape[-1])[:, g]
            s = torch.matmul(qs, pool[g].t().contiguous())
            s = (s.clamp_min(0) if relu else s).sum(1)
            kept.append(_keep(cfg, s[:, :nb], L))
        for g in range(cfg.n_head_kv):
            ids, valid = kept[g % len(kept)]
            h = slice(g * group, (g + 1) * group)
            out[at, h] = _attend(cfg, q[at, h].contiguous(), Kb[g], Vb[g], ids, valid, L)
    return out


def exact(case, seed):
    if case["path"] == "session":
        return _exact_session(case, seed)
    gen, cfg, past, _, _ = _inputs(case, seed)
    kv, ckpt = case["kv"], case["path"].startswith("ckpt")
    icfg = qsa.IdxConfig()

    def joined(chunks):
        got = [torch.cat([x.to(torch.float64) for x in col]) for col in zip(*chunks)]
        return got

    rows = []
    for n in past:
        chunks = [(_cached(k, kv), _cached(v, kv)) for _, k, v in _past(gen, n, cfg)]
        rows.append(joined(chunks) if chunks else [torch.zeros((0, cfg.n_head_kv, cfg.head_dim), device="cuda",
                                                               dtype=torch.float64)] * 2)
    keys = []
    if ckpt:
        norm = _k_norm(gen, icfg)
        for n in past:
            chunks = [kr.half() for _, kr in _past_keys(gen, n, icfg)]
            keys.append(torch.cat(chunks) if chunks else torch.zeros((0, icfg.idx_dim), device="cuda").half())
    n_seq = len(past)
    if "pos0" in case:
        lead = (case["n_q"],)
    else:
        lead = (case["n_pos"], n_seq) if case["path"] == "chain" else (n_seq,)
    q, kn, vn = _new(gen, case, cfg, *lead)
    qi, kr = _new_keys(gen, case, icfg, len(q)) if ckpt else (None, None)
    n_pos = lead[0] if len(lead) == 2 or "pos0" in case else 1
    q, kn, vn = (x.reshape(n_pos, n_seq, *x.shape[-2:]) for x in (q, kn, vn))
    out = torch.empty(q.shape, dtype=torch.float64, device="cuda")
    for s in range(n_seq):
        K = torch.cat([rows[s][0], _cached(kn[:, s], kv)])
        V = torch.cat([rows[s][1], _cached(vn[:, s], kv)])
        rows[s] = None
        lengths = past[s] + 1 + torch.arange(n_pos, device="cuda")
        qs = q[:, s].double()
        if ckpt:
            at = slice(None) if "pos0" in case else slice(s, s + 1)
            raw = torch.cat([keys[s], kr[at].half()])
            pool, q_score = _idx_pooled(icfg, cfg, raw, norm)[None], qi[at].double()
        else:
            pool, q_score = _blocks(cfg, K).mean(2), qs
        out[:, s] = _exact_queries(cfg, qs, K, V, lengths, pool, q_score, bool(cfg.relu_per_head))
        del K, V, pool
    shape = (*lead, cfg.n_head, cfg.head_dim)
    return {"out": out.reshape(shape)}


def _exact_session(case, seed):
    cfg, k, _ = _session_rows(case, seed)
    n, nb = case["n_tokens"], case["n_tokens"] // cfg.block_tokens
    if case["kv"] == F16:
        x = k.view(torch.float16).double().view(n, cfg.n_head_kv, cfg.head_dim)
    else:
        b = k.view(n, cfg.kv_dim // 32, -1)
        d = b[:, :, :2].contiguous().view(torch.float16).double()
        if case["kv"] == Q8_0:
            quants = b[:, :, 2:].contiguous().view(torch.int8).double()
        else:
            quants = torch.cat([b[:, :, 2:] & 15, b[:, :, 2:] >> 4], 2).double() - 8
        x = (d * quants).view(n, cfg.n_head_kv, cfg.head_dim)
    whole = x[: nb * cfg.block_tokens].view(nb, cfg.block_tokens, cfg.n_head_kv, cfg.head_dim).mean(1).transpose(0, 1)
    bps = _up(n, cfg.page_tokens) // cfg.block_tokens
    pooled = torch.zeros((1, cfg.n_head_kv, bps, cfg.head_dim), dtype=torch.float64, device="cuda")
    pooled[0, :, :nb] = whole
    return {"pooled": pooled}

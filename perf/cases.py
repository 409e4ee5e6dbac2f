"""The KV-cache attention path as a serving program drives it, as cases that can be timed and compared.

Two kinds of case, both through the cache managers' own interface:

* "attend": the attention of one forward. `prepare` builds a cache whose sequences hold
  cached context and begins a forward (positions, block table and write plan are then
  made, once for all layers); one pass runs every layer's attention call: the new rows'
  K/V written into the pool and the attention over context and new rows, with the
  rotary embedding in front where the case says so.
* "serve": requests from admission to release. One pass allocates the sequences,
  prefills their prompts in chunks, decodes a number of tokens and releases them,
  planning included.

Shapes are those of this repository's workloads, tests and benchmark: 32 query heads
over 8 KV heads of 128 (and the other head shapes the kernels take), pages of 16
tokens, contexts up to 32k, fp16 and bf16 paged pools, fp32 contiguous pools.
"""
import math
import random

import torch

from nanoslg_amd.kv_cache import ContiguousKVCache, KVCacheConfig, PagedKVCache, attention_forward

DEV = "cuda:0"
DTYPES = {"fp16": torch.float16, "bf16": torch.bfloat16, "fp32": torch.float32}
VOCAB = 128256


def _case(name=None, kind="attend", backend="paged", dtype="fp16", hq=32, hkv=8, d=128, page=16, layers=4, batch=1,
          ctx_lo=0, ctx_hi=0, new_lo=1, new_hi=1, prefix=0, rope=False, chunk=0, steps=0, lens_seed=0):
    """ctx_lo..ctx_hi: tokens a sequence has cached, its prefix apart (log-uniform);
    new_lo..new_hi: its new tokens; prefix: leading tokens that all sequences share
    through the prefix tree; chunk, steps: prefill chunk and decode steps of "serve"."""
    c = dict(kind=kind, backend=backend, dtype=dtype, hq=hq, hkv=hkv, d=d, page=page, layers=layers, batch=batch,
             ctx_lo=ctx_lo, ctx_hi=ctx_hi, new_lo=new_lo, new_hi=new_hi, prefix=prefix, rope=rope, chunk=chunk,
             steps=steps, lens_seed=lens_seed)
    if name:
        c["name"] = name
    return c


def listed():
    return [
        # one user of an fp32 model on the contiguous backend, a token after a 512-token
        # prompt: the smallest call, all latency
        _case("decode_fp32_contiguous_b1", backend="contiguous", dtype="fp32", layers=2, ctx_lo=512, ctx_hi=575),
        # a lightly loaded server: 4 conversations of 1k to 4k tokens
        _case("decode_fp16_b4", batch=4, ctx_lo=1024, ctx_hi=4095),
        # a loaded server under KV pressure: 64 conversations of 2k to 32k tokens
        _case("decode_fp16_b64_32k", layers=1, batch=64, ctx_lo=2048, ctx_hi=32767),
        # requests on one 2040-token system prompt, decoding: shared pages read once per group
        _case("decode_fp16_shared_prefix_b16", batch=16, prefix=2040, ctx_lo=128, ctx_hi=1024),
        # a rotary-embedding model in the default dtype, mixed conversations
        _case("decode_bf16_rope_b16", dtype="bf16", batch=16, ctx_lo=256, ctx_hi=8191, rope=True, lens_seed=1),
        # a batch of 4096-token prompts prefilled in 512-token chunks: admission to release
        _case("serve_prefill_fp16_8x4096", kind="serve", layers=1, batch=8, new_lo=4096, new_hi=4096, chunk=512),
        # one long request's next chunk, in the default dtype
        _case("chunk_bf16_b1_over_6k", dtype="bf16", layers=2, ctx_lo=6007, ctx_hi=6007, new_lo=512, new_hi=512),
        # the suffixes of requests on one cached system prompt: ragged, left-padded rows
        _case("suffix_fp16_shared_prefix_b16", layers=2, batch=16, prefix=2040, new_lo=128, new_hi=1024),
        # a padded batch of fresh prompts of an fp32 model on the contiguous backend
        _case("prompt_fp32_contiguous_b4", backend="contiguous", dtype="fp32", layers=2, batch=4, new_lo=100,
              new_hi=512, lens_seed=2),
        # a padded batch of fresh prompts of a rotary model with 64-wide heads
        _case("prompt_bf16_rope_d64_b4", dtype="bf16", d=64, layers=2, batch=4, new_lo=250, new_hi=2000, rope=True,
              lens_seed=3),
        # chunks of two requests of a model with 256-wide heads
        _case("chunk_bf16_d256_b2", dtype="bf16", hq=16, hkv=4, d=256, layers=2, batch=2, ctx_lo=1500, ctx_hi=3000,
              new_lo=512, new_hi=512, lens_seed=4),
        # short chats of a rotary model, from admission to release: prompts, then 8 tokens each
        _case("serve_chat_bf16_rope_b4", kind="serve", dtype="bf16", batch=4, new_lo=90, new_hi=400, rope=True,
              chunk=512, steps=8, lens_seed=5),
    ]


def _log_int(rng, lo, hi):
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


#: (query heads, KV heads, head dim): mostly the grouped 128-wide heads
_HEADS = [(32, 8, 128)] * 5 + [(64, 8, 128), (8, 8, 128), (16, 1, 128), (32, 8, 64), (16, 4, 256)]
#: A drawn case does at most this much work (the largest listed one's, with room for slower types)
_MOST_KV_BYTES = 2.8e9
_MOST_FLOPS = {"fp16": 3e11, "bf16": 3e11, "fp32": 1.2e10}


def draw(rng):
    while True:
        c = _draw(rng)
        w = work(c)
        if w["bytes"] <= _MOST_KV_BYTES and w["flops"] <= _MOST_FLOPS[c["dtype"]] * (2 if c["hq"] * c["d"] > 4096 else 1):
            return c


def _draw(rng):
    family = rng.choice(["decode", "decode", "shared", "chunk", "chunk", "suffix", "prompt", "fp32_decode", "fp32_prompt",
                         "chat"])
    hq, hkv, d = rng.choice(_HEADS)
    c = dict(dtype=rng.choice(["fp16", "bf16"]), hq=hq, hkv=hkv, d=d, page=rng.choice([16, 16, 16, 8, 32, 64]),
             layers=rng.randint(1, 3), rope=rng.random() < 0.4, lens_seed=rng.randrange(1 << 20))
    if family == "decode":
        hi = _log_int(rng, 64, 32767)
        c.update(batch=_log_int(rng, 1, 64), ctx_lo=max(1, hi // rng.choice([1, 2, 4, 16])), ctx_hi=hi)
    elif family == "shared":
        c.update(batch=rng.randint(2, 16), prefix=_log_int(rng, 100, 8000), ctx_lo=16, ctx_hi=_log_int(rng, 64, 2048))
    elif family == "chunk":
        n = _log_int(rng, 16, 1024)
        hi = _log_int(rng, 64, 16000)
        c.update(batch=_log_int(rng, 1, 8), ctx_lo=max(1, hi // rng.choice([1, 3])), ctx_hi=hi,
                 new_lo=rng.choice([n, max(1, n // 2)]), new_hi=n)
    elif family == "suffix":
        c.update(batch=rng.randint(2, 16), prefix=_log_int(rng, 100, 4000), new_lo=16, new_hi=_log_int(rng, 32, 1024))
    elif family == "prompt":
        hi = _log_int(rng, 32, 2048)
        c.update(batch=_log_int(rng, 1, 8), new_lo=max(1, hi // 3), new_hi=hi)
    elif family == "fp32_decode":
        hi = _log_int(rng, 64, 4000)
        c.update(backend="contiguous", dtype="fp32", batch=rng.randint(1, 8), ctx_lo=max(1, hi // 2), ctx_hi=hi)
    elif family == "fp32_prompt":
        hi = _log_int(rng, 24, 600)
        c.update(backend="contiguous", dtype="fp32", batch=rng.randint(1, 4), new_lo=max(1, hi // 2), new_hi=hi)
    else:
        hi = _log_int(rng, 24, 800)
        c.update(kind="serve", batch=rng.randint(1, 6), new_lo=max(1, hi // 2), new_hi=hi, chunk=rng.choice([256, 512]),
                 steps=rng.randint(2, 10))
    return _case(**c)


# ---- sizes ---------------------------------------------------------------------------


def _lens(case):
    """Per sequence: tokens cached (the shared prefix apart), new tokens."""
    rng = random.Random(case["lens_seed"])
    ctx, new = [], []
    for _ in range(case["batch"]):
        ctx.append(_log_int(rng, case["ctx_lo"], case["ctx_hi"]) if case["ctx_lo"] else 0)
        new.append(rng.randint(case["new_lo"], case["new_hi"]))
    return ctx, new


def _chunks(case, new):
    """The forwards of a "serve" case: new tokens of each sequence in each."""
    out, done = [], [0] * len(new)
    while any(a < n for a, n in zip(done, new)):
        step = [min(case["chunk"], n - a) for a, n in zip(done, new)]
        out.append(step)
        done = [a + s for a, s in zip(done, step)]
    return out + [[1] * len(new)] * case["steps"]


def work(case):
    """K/V of every distinct cached token read once, the new rows read and written, q
    read and out written; 4 * D flops per query head and visible key."""
    ctx, new = _lens(case)
    s = 4 if case["dtype"] == "fp32" else 2
    row, qrow = 2 * case["hkv"] * case["d"] * s, 2 * case["hq"] * case["d"] * s
    if case["kind"] == "attend":
        forwards, cached = [new], [case["prefix"] + a for a in ctx]
    else:
        forwards, cached = _chunks(case, new), [0] * len(new)
    nbytes = pairs = 0
    for f in forwards:
        shared = case["prefix"] * (len(new) - 1)
        nbytes += (sum(cached) - shared) * row + sum(f) * (2 * row + qrow)
        pairs += sum(a * n + n * (n + 1) // 2 for a, n in zip(cached, f))
        cached = [a + n for a, n in zip(cached, f)]
    return {"bytes": nbytes * case["layers"], "flops": 4 * case["hq"] * case["d"] * pairs * case["layers"]}


def tolerance(case):
    """About four times the error against 64 bits, as measured: 3e-7 to 6e-7 in fp32, 2.5e-4
    to 4.2e-4 in fp16 (one rounding of the outputs, and of the probabilities in the
    products), 1.7e-3 in bf16 and up to 3.8e-3 where q and k are rotated (and rounded)
    first; more in fp32, where long sums in another order are a little further apart."""
    if case["dtype"] == "fp32":
        return {"rel": 5e-6, "max": 2e-4}
    if case["dtype"] == "fp16":
        return {"rel": 1.5e-3, "max": 2e-2}
    return {"rel": 1e-2, "max": 8e-2}


# ---- inputs --------------------------------------------------------------------------


def _generator(seed):
    return torch.Generator(device=DEV).manual_seed(1_000_003 * seed + 17)


def _randn(g, case, *shape):
    return torch.randn(*shape, generator=g, device=DEV, dtype=DTYPES[case["dtype"]])


def _cached_kv(case, ctx, g):
    """K and V of the cached tokens: the shared prefix, then each sequence's own."""
    n, L = case["prefix"] + sum(ctx), case["layers"]
    return _randn(g, case, L, n, case["hkv"], case["d"]), _randn(g, case, L, n, case["hkv"], case["d"])


def _forward_inputs(case, rows, g):
    """q, k_new, v_new of one forward of `rows` padded rows per sequence, every layer."""
    B, L = case["batch"], case["layers"]
    return (_randn(g, case, L, B, rows, case["hq"], case["d"]), _randn(g, case, L, B, rows, case["hkv"], case["d"]),
            _randn(g, case, L, B, rows, case["hkv"], case["d"]))


def _rope_tables(case, rows):
    inv = 1.0 / (500000.0 ** (torch.arange(0, case["d"], 2, device=DEV, dtype=torch.float64) / case["d"]))
    a = torch.outer(torch.arange(rows, device=DEV, dtype=torch.float64), inv)
    a = torch.cat([a, a], 1)
    return a.cos().float(), a.sin().float()


def _max_len(case):
    ctx, new = _lens(case)
    return case["prefix"] + max(a + n for a, n in zip(ctx, new)) + case["steps"]


def _manager(case, ctx, new):
    cfg = dict(num_layers=case["layers"], num_kv_heads=case["hkv"], num_qo_heads=case["hq"], head_dim=case["d"],
               dtype=DTYPES[case["dtype"]], device=torch.device(DEV), backend=case["backend"])
    if case["backend"] == "contiguous":
        return ContiguousKVCache(KVCacheConfig(max_batch_size=case["batch"], max_seq_len=_max_len(case) + 64, **cfg))
    ps = case["page"]
    need = sum(-(-(a + n + case["steps"]) // ps) + 2 for a, n in zip(ctx, new)) + 2 * (-(-case["prefix"] // ps) + 1)
    # a pool in use to about nine tenths
    return PagedKVCache(KVCacheConfig(max_pages=need + need // 9 + 8, page_size=ps,
                                      enable_prefix_caching=case["prefix"] > 0, **cfg))


def _put(mgr, sid, first, k, v):
    """K and V [L, n, Hkv, D] of sequence sid's tokens from position `first` into the pool, as its prefill would."""
    n = k.shape[1]
    if isinstance(mgr, ContiguousKVCache):
        slot = mgr.states[sid].slot
        mgr.k[:, slot, first:first + n] = k
        mgr.v[:, slot, first:first + n] = v
        return
    ps = mgr.cfg.page_size
    table = torch.tensor(mgr.seqs[sid].block_table, device=DEV)
    pos = torch.arange(first, first + n, device=DEV)
    slots = table[pos // ps] * ps + pos % ps
    for pool, rows in ((mgr.pool.k, k), (mgr.pool.v, v)):
        pool.view(pool.shape[0], -1, *pool.shape[3:])[:, slots] = rows


def _prepare_attend(case, seed):
    ctx, new = _lens(case)
    g = _generator(seed)
    k, v = _cached_kv(case, ctx, g)
    mgr = _manager(case, ctx, new)
    ids = ["s%d" % i for i in range(case["batch"])]
    rng = random.Random(seed)
    pre = case["prefix"]
    if pre:
        # an earlier request left the prefix in the prefix tree; each sequence then finds it there
        tokens = [rng.randrange(VOCAB) for _ in range(pre)]
        mgr.allocate_sequence("first", token_ids=tokens)
        mgr.end_forward(mgr.begin_forward(["first"], [pre]))
        _put(mgr, "first", 0, k[:, :pre], v[:, :pre])
        mgr.release_sequence("first")
        for s, a, n in zip(ids, ctx, new):
            own = [rng.randrange(VOCAB) for _ in range(a if a else n)]
            mgr.allocate_sequence(s, token_ids=tokens + own)
    else:
        for s in ids:
            mgr.allocate_sequence(s)
        if case["backend"] == "paged":
            # pages taken in turns, so that a sequence's pages lie all over the pool
            turns = [i for i, a in enumerate(ctx) for _ in range(-(-a // case["page"]))]
            rng.shuffle(turns)
            have = [0] * case["batch"]
            for i in turns:
                have[i] = min(ctx[i], have[i] + case["page"])
                mgr.extend_sequence(ids[i], have[i])
    if any(ctx):
        mgr.end_forward(mgr.begin_forward(ids, ctx))
        at = pre
        for s, a in zip(ids, ctx):
            _put(mgr, s, pre, k[:, at:at + a], v[:, at:at + a])
            at += a
    del k, v
    S = max(new)
    q, kn, vn = _forward_inputs(case, S, g)
    fwd = mgr.begin_forward(ids, new, [S - n for n in new] if S > 1 else None)
    rope = _rope_tables(case, _max_len(case)) if case["rope"] else None
    return {"case": case, "mgr": mgr, "ctx": fwd, "inputs": (q, kn, vn), "rope": rope}


def _prepare_serve(case, seed):
    ctx, new = _lens(case)
    g = _generator(seed)
    forwards = [(n, _forward_inputs(case, max(n), g)) for n in _chunks(case, new)]
    rope = _rope_tables(case, _max_len(case)) if case["rope"] else None
    return {"case": case, "mgr": _manager(case, ctx, new), "forwards": forwards, "rope": rope}


def prepare(case, seed):
    return (_prepare_attend if case["kind"] == "attend" else _prepare_serve)(case, seed)


# ---- one pass ------------------------------------------------------------------------


def _attention(case, ctx, inputs, rope):
    """Every layer's attention of one forward."""
    q, k, v = inputs
    hq, hkv = case["hq"], case["hkv"]
    if rope is None:
        return [ctx.attend(i, q[i], k[i], v[i], hq, hkv) for i in range(case["layers"])]
    return [attention_forward(q[i], k[i], v[i], i, hq, hkv, rope[0], rope[1], ctx) for i in range(case["layers"])]


def run(state):
    case, mgr = state["case"], state["mgr"]
    if case["kind"] == "attend":
        out = _attention(case, state["ctx"], state["inputs"], state["rope"])
        pool = mgr if case["backend"] == "contiguous" else mgr.pool
        return {"out": out, "k": pool.k, "v": pool.v}
    ids = ["s%d" % i for i in range(case["batch"])]
    for s in ids:
        mgr.allocate_sequence(s)
    out = []
    for n, inputs in state["forwards"]:
        S = max(n)
        ctx = mgr.begin_forward(ids, n, None if min(n) == S else [S - x for x in n])
        out.append(_attention(case, ctx, inputs, state["rope"]))
        mgr.end_forward(ctx)
    for s in ids:
        mgr.release_sequence(s)
    return {"out": out}


# ---- the same in 64 bits --------------------------------------------------------------


def _rotate(x, tables, first):
    """Rotary embedding of x [n, heads, D] at positions first .. first + n - 1."""
    c, s = (t[first:first + x.shape[0], None].double() for t in tables)
    h = x.shape[-1] // 2
    return x * c + torch.cat([-x[..., h:], x[..., :h]], -1) * s


def _attend64(q, k, v):
    """Causal attention, bottom-right aligned: q [n, Hq, D] over k, v [m, Hkv, D]."""
    n, hq, d = q.shape
    m, hkv = k.shape[:2]
    out = torch.empty(n, hq, d, dtype=torch.float64, device=q.device)
    step = max(1, (1 << 27) // max(1, m * (hq // hkv)))
    for h in range(hkv):
        heads = slice(h * (hq // hkv), (h + 1) * (hq // hkv))
        kt, vh = k[:, h].t().contiguous(), v[:, h].contiguous()
        for a in range(0, n, step):
            b = min(n, a + step)
            x = q[a:b, heads].reshape(-1, d).contiguous() @ kt / math.sqrt(d)
            x = x.view(b - a, -1, m)
            seen = torch.arange(m, device=q.device)[None] <= torch.arange(m - n + a, m - n + b, device=q.device)[:, None]
            x.masked_fill_(~seen[:, None], -math.inf)
            out[a:b, heads] = (torch.softmax(x, -1).view(-1, m) @ vh).view(b - a, -1, d)
    return out


def exact(case, seed):
    ctx, new = _lens(case)
    g = _generator(seed)
    B, L, hkv, d, pre = case["batch"], case["layers"], case["hkv"], case["d"], case["prefix"]
    rope = _rope_tables(case, _max_len(case)) if case["rope"] else None
    if case["kind"] == "attend":
        ck, cv = _cached_kv(case, ctx, g)
        forwards = [(new, _forward_inputs(case, max(new), g))]
        starts = [pre + sum(ctx[:b]) for b in range(B)]
        kv = [[[torch.cat([c[i, :pre], c[i, starts[b]:starts[b] + ctx[b]]]) for c in (ck, cv)] for b in range(B)]
              for i in range(L)]
        del ck, cv
    else:
        forwards = [(n, _forward_inputs(case, max(n), g)) for n in _chunks(case, new)]
        empty = torch.empty(0, hkv, d, dtype=DTYPES[case["dtype"]], device=DEV)
        kv = [[[empty, empty] for _ in range(B)] for _ in range(L)]
    outs = []
    for n, (q, k, v) in forwards:
        S = max(n)
        layer_outs = []
        for i in range(L):
            o = torch.zeros(B, S, case["hq"], d, dtype=torch.float64, device=DEV)
            for b in range(B):
                rows = slice(S - n[b], S)
                have_k, have_v = kv[i][b]
                qb, kb, first = q[i, b, rows].double(), k[i, b, rows].double(), have_k.shape[0]
                if rope is not None:
                    qb, kb = _rotate(qb, rope, first), _rotate(kb, rope, first)
                keys = torch.cat([have_k.double(), kb])
                values = torch.cat([have_v, v[i, b, rows]])
                o[b, rows] = _attend64(qb, keys, values.double())
                # the next forward's cached tokens (in 64 bits only where they were rotated)
                kv[i][b] = [keys if rope is not None else torch.cat([have_k, k[i, b, rows]]), values]
            layer_outs.append(o.view(B, S, -1))
        outs.append(layer_outs)
    if case["kind"] == "attend":
        return {"out": outs[0], "k": None, "v": None}
    return {"out": outs}

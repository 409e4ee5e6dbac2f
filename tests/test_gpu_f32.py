"""The fp32 attention kernels at the edges of their tiles, waves, runs and pages, against
the oracle's fp32 SDPA (within summation-order differences), and the decode's fused write
of the new rows against append_kv."""
import math

import numpy as np
import pytest
import torch

from test_gpu_kernels import ATOL, F32_TOL, RTOL, _csr_random, _decode_case, _prefill_case

DEV = "cuda:0"


@pytest.mark.gpu
@pytest.mark.parametrize("lens,Hq,Hkv,D,ps", [
    ([1, 15, 16, 17, 63, 64, 65, 0], 8, 2, 128, 16),   # one tile and its neighbours, one wave each and more
    ([129, 4, 640, 1000], 16, 1, 128, 5),              # G = 16, tiles across pages
    ([4500], 4, 4, 128, 1),                            # G = 1, 64 runs
    ([70, 2000, 0, 33], 32, 8, 64, 48),
    ([31, 900], 12, 2, 256, 16),
    ([700] * 40, 8, 8, 128, 700),                      # whole slots, one run each
    ([4000, 3100], 32, 8, 128, 16),                    # 32 runs: the merge in four parts
])
def test_f32_decode_edges(lens, Hq, Hkv, D, ps):
    out, ref = _decode_case(lens, Hq, Hkv, D, ps, torch.float32, seed=800 + D + ps)
    torch.testing.assert_close(out, ref, **F32_TOL)


@pytest.mark.gpu
@pytest.mark.parametrize("lens,news,Hq,Hkv,D,ps", [
    ([1, 16, 17, 33], [1, 16, 17, 2], 32, 8, 128, 16),     # row tiles of one token to one and a bit
    ([100, 300, 64], [100, 0, 31], 12, 4, 128, 5),         # G = 3: tokens across waves; no new tokens
    ([1200, 520], [40, 7], 8, 8, 128, 16),                 # runs of keys, merged
    ([700], [300], 16, 1, 64, 1),                          # G = 16, one-token pages
    ([90, 600], [90, 33], 16, 4, 256, 48),
    ([530] * 24, [40] * 24, 32, 8, 128, 16),               # two key groups a row tile
    ([40], [10], 32, 8, 128, 16),                          # too few workgroups for two
    ([70], [5], 12, 4, 64, 16),
    ([33, 100], [2, 9], 16, 4, 256, 16),
])
def test_f32_prefill_edges(lens, news, Hq, Hkv, D, ps):
    out, ref = _prefill_case(lens, news, Hq, Hkv, D, ps, torch.float32, seed=820 + D + ps)
    torch.testing.assert_close(out, ref, **F32_TOL)


@pytest.mark.gpu
@pytest.mark.parametrize("D", [64, 128, 256])
def test_f32_prefill_of_many_workgroups(D):
    """A ragged batch of more workgroups than take two key groups a row tile, in one run:
    the kernel of every large fp32 prompt batch."""
    news = [60 + (7 * b) % 31 for b in range(48)]
    lens = [n + (5 * b) % 40 for b, n in enumerate(news)]
    out, ref = _prefill_case(lens, news, 32, 8, D, 16, torch.float32, seed=840 + D)
    assert (-(-sum(news) * 4 // 64) + len(news)) * 8 > 2048  # launch_f32's limit (D = 64; 1024 otherwise)
    torch.testing.assert_close(out, ref, **F32_TOL)


@pytest.mark.gpu
@pytest.mark.parametrize("D", [64, 128, 256])
def test_f32_decode_writes_the_new_rows(D):
    """paged_decode_append on rows 4-byte aligned only: the pool as append_kv leaves it,
    the result that of append_kv then paged_decode, bit for bit."""
    from nanoslg_amd import kernels as K
    Hq, Hkv, ps, lens = 8, 2, 16, [1, 16, 17, 64, 65, 900]
    g = torch.Generator().manual_seed(D)
    P = sum(-(-n // ps) for n in lens) + 2
    _, (indptr, indices, lpl) = _csr_random(lens, ps, P, D)
    slots = np.array([indices[indptr[b + 1] - 1] * ps + (n - 1) % ps for b, n in enumerate(lens)], np.int32)
    rows = torch.randn(2, len(lens), Hkv * D + 1, generator=g).to(DEV)
    k, v = (x[:, 1:].unflatten(1, (Hkv, D)) for x in rows)  # rows at an odd stride, off 16 bytes
    q = torch.randn(len(lens), Hq, D, generator=g).to(DEV)
    k1, v1 = (torch.randn(P, ps, Hkv, D, generator=g).to(DEV) for _ in range(2))
    k2, v2 = k1.clone(), v1.clone()
    plan = tuple(torch.from_numpy(a).to(DEV) for a in (indptr, indices, lpl)) + (int(indptr[-1]),)
    o1 = K.paged_decode_append(q, k, v, k1, v1, *plan)
    K.append_kv(k, v, torch.from_numpy(slots).to(DEV), k2, v2)
    o2 = K.paged_decode(q, k2, v2, *plan)
    torch.cuda.synchronize()
    assert torch.equal(k1, k2) and torch.equal(v1, v2) and torch.equal(o1, o2)


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.float32, torch.float16])
def test_contiguous_decode_in_one_launch(dtype):
    """Decode steps of the contiguous cache against append_kv then paged_decode on a copy:
    pool bytes and outputs equal; two contexts of different batches alive at once, a
    negative layer index, rows off 16 bytes and a changed batch included."""
    from nanoslg_amd import kernels as K
    from nanoslg_amd.kv_cache import ContiguousKVCache, KVCacheConfig
    L, Hq, Hkv, D, Smax = 2, 8, 2, 64, 77
    m = ContiguousKVCache(KVCacheConfig(num_layers=L, num_kv_heads=Hkv, num_qo_heads=Hq, head_dim=D, max_batch_size=3,
                                        max_seq_len=Smax, dtype=dtype, device=torch.device(DEV), backend="contiguous"))
    g = torch.Generator().manual_seed(5)
    rnd = lambda *s: torch.randn(*s, generator=g).to(dtype).to(DEV)  # noqa: E731
    ids = ["a", "b", "c"]
    for s in ids:
        m.allocate_sequence(s)
    ctx = m.begin_forward(ids, [40, 3, 75])
    for layer in range(L):
        ctx.attend(layer, rnd(3, 75, Hq, D), rnd(3, 75, Hkv, D), rnd(3, 75, Hkv, D), Hq, Hkv)
    m.end_forward(ctx)

    def step(ctx, batch, layer):
        B, plan = len(batch), ctx._plan
        q, rows = rnd(B, 1, Hq, D), rnd(2, B, Hkv * D + 1)
        k, v = (x[:, 1:].reshape(B, 1, Hkv, D) if layer else x[:, 1:].unflatten(1, (Hkv, D)).unsqueeze(1) for x in rows)
        kc, vc = m.k[layer].clone(), m.v[layer].clone()
        out = ctx.attend(layer, q, k, v, Hq, Hkv)
        K.append_kv(k, v, plan.slot, kc, vc)
        want = K.paged_decode(q[:, 0], kc, vc, plan.indptr, plan.indices, plan.lpl, plan.total_pages)
        torch.cuda.synchronize()
        assert torch.equal(m.k[layer], kc) and torch.equal(m.v[layer], vc)
        assert torch.equal(out.view(B, Hq, D), want)

    for batch in (ids, ["c", "a"], ["a", "b"]):
        one = m.begin_forward(batch, [1] * len(batch))
        two = m.begin_forward(batch[:1], [1])  # another forward's plan in between
        step(one, batch, 0)
        step(two, batch[:1], 0)
        step(one, batch, -1)
        q, kv = rnd(len(batch), 1, Hq, D), rnd(len(batch), 1, Hkv, D)
        for bad in (L, -L - 1):
            with pytest.raises(IndexError):
                one.attend(bad, q, kv, kv, Hq, Hkv)
        m.end_forward(one)


def _attention64(q, k, v, n):
    """Causal attention of the last n tokens, bottom-right aligned, in 64 bits: q [n, Hq, D]
    over k, v [m, Hkv, D]; a NaN or infinity goes where softmax and product take it."""
    q, k, v = (x.double().transpose(0, 1) for x in (q, k, v))
    G, m = q.shape[0] // k.shape[0], k.shape[1]
    s = q @ k.repeat_interleave(G, 0).transpose(1, 2) / math.sqrt(q.shape[2])
    seen = torch.arange(m)[None] <= torch.arange(m - n, m)[:, None]
    p = torch.softmax(s.masked_fill(~seen, -math.inf), -1)
    return (p @ v.repeat_interleave(G, 0)).transpose(0, 1)


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.float32, torch.float16, torch.bfloat16])
@pytest.mark.parametrize("L,n", [(900, 0), (4000, 0), (900, 3), (1300, 40)])  # n = 0: a decode token
@pytest.mark.parametrize("bad", ["nan", "nan_row", "inf"])
def test_nonfinite_keys_reach_the_rows_that_see_them(bad, L, n, dtype):
    """Whole runs of keys, or one key, that score NaN or +-inf, in calls cut into runs and
    merged: a row of the KV head is NaN where softmax over its keys is, and no other is."""
    from nanoslg_amd import kernels as K
    Hq, Hkv, D, ps = 8, 2, 128, 16
    g = torch.Generator().manual_seed(L + n)
    q = torch.randn(max(n, 1), Hq, D, generator=g).to(dtype)
    k, v = (torch.randn(L, Hkv, D, generator=g).to(dtype) for _ in range(2))
    if bad == "nan":
        k[:512, 1] = math.nan     # all the keys of the first runs (64 or 128 keys, or key tiles of 128)
    elif bad == "nan_row":
        k[700, 1, 5] = math.nan
    else:
        k[3, 1, 5] = math.inf     # +inf or -inf by the sign of the row's element 5
    npg = -(-L // ps)
    pool = torch.zeros(2, npg * ps, Hkv, D, dtype=dtype)
    pool[0, :L], pool[1, :L] = k, v
    kp, vp = pool.view(2, npg, ps, Hkv, D).to(DEV)
    i32 = lambda *a: torch.tensor(a, dtype=torch.int32, device=DEV)  # noqa: E731
    plan = (i32(0, npg), torch.arange(npg, dtype=torch.int32, device=DEV), i32((L - 1) % ps + 1))
    if n:
        out = K.paged_prefill(q.to(DEV), i32(0, n), n, n, kp, vp, *plan)
    else:
        out = K.paged_decode(q.to(DEV), kp, vp, *plan, npg)
    ref = _attention64(q, k, v, max(n, 1))
    out = out.cpu()
    assert torch.equal(out.isnan(), ref.isnan())
    assert ref[:, :Hq // Hkv].isfinite().all() and ref.isnan().any()
    tol = F32_TOL if dtype == torch.float32 else dict(atol=ATOL, rtol=RTOL)
    torch.testing.assert_close(out.float(), ref.float(), equal_nan=True, **tol)


@pytest.mark.gpu
def test_contiguous_forwards_attended_in_between(monkeypatch):
    """A decode forward of the contiguous cache attended while another one's call is under
    way (between its launcher being found and its launch, as from a second thread): each
    writes and reads the slots of its own sequences."""
    from nanoslg_amd import kernels as K
    from nanoslg_amd.kv_cache import ContiguousKVCache, KVCacheConfig
    Hq, Hkv, D = 8, 2, 64
    m = ContiguousKVCache(KVCacheConfig(num_layers=1, num_kv_heads=Hkv, num_qo_heads=Hq, head_dim=D, max_batch_size=3,
                                        max_seq_len=80, dtype=torch.float32, device=torch.device(DEV),
                                        backend="contiguous"))
    g = torch.Generator().manual_seed(6)
    rnd = lambda *s: torch.randn(*s, generator=g).to(DEV)  # noqa: E731
    for s in "abc":
        m.allocate_sequence(s)
    ctx = m.begin_forward(list("abc"), [40, 3, 70])
    ctx.attend(0, rnd(3, 70, Hq, D), rnd(3, 70, Hkv, D), rnd(3, 70, Hkv, D), Hq, Hkv)
    m.end_forward(ctx)
    forwards = [m.begin_forward([s], [1]) for s in "abc"]
    inputs = [(rnd(1, 1, Hq, D), rnd(1, 1, Hkv, D), rnd(1, 1, Hkv, D)) for _ in forwards]
    kc, vc = m.k[0].clone(), m.v[0].clone()
    want = []
    for f, (q, k, v) in zip(forwards, inputs):
        K.append_kv(k, v, f._plan.slot, kc, vc)
        want.append(K.paged_decode(q[:, 0], kc, vc, f._plan.indptr, f._plan.indices, f._plan.lpl, 1).view(1, 1, -1))
    forwards[2].attend(0, *inputs[2], Hq, Hkv)  # (an earlier forward of the same batch size)
    got, call = [], K.DecodeLaunch.__call__

    def nested(self, *args, **kw):
        monkeypatch.setattr(K.DecodeLaunch, "__call__", call)
        got.append(forwards[1].attend(0, *inputs[1], Hq, Hkv))
        return call(self, *args, **kw)

    monkeypatch.setattr(K.DecodeLaunch, "__call__", nested)
    got.insert(0, forwards[0].attend(0, *inputs[0], Hq, Hkv))
    torch.cuda.synchronize()
    assert torch.equal(m.k[0], kc) and torch.equal(m.v[0], vc)
    assert torch.equal(got[0], want[0]) and torch.equal(got[1], want[1])


FORMS = ["heads", "heads_no_multiple", "shared_kv", "flat_kv", "heads_apart", "one_head", "one_row", "cpu_sin", "cpu_q",
         "f64_k"]


@pytest.mark.gpu
@pytest.mark.parametrize("rope", [False, True])
@pytest.mark.parametrize("form", FORMS)
def test_contiguous_decode_takes_the_forms_of_the_separate_calls(form, rope):
    """A decode step of the contiguous cache serves what append_kv (rope_append) and
    paged_decode serve, with their result, and refuses with their error what they refuse:
    other query heads in one forward, heads that are no multiple, one K row for the whole
    batch, rows of other ranks, heads apart in memory, one head or row at any stride,
    tensors of another device or dtype."""
    from nanoslg_amd import kernels as K
    from nanoslg_amd.kv_cache import ContiguousKVCache, KVCacheConfig
    Hq, Hkv, D, B = (1, 1, 64, 2) if form == "one_head" else (8, 2, 64, 1 if form == "one_row" else 2)
    m = ContiguousKVCache(KVCacheConfig(num_layers=1, num_kv_heads=Hkv, num_qo_heads=Hq, head_dim=D, max_batch_size=B,
                                        max_seq_len=80, dtype=torch.float16, device=torch.device(DEV),
                                        backend="contiguous"))
    g = torch.Generator().manual_seed(6)
    rnd = lambda *s: torch.randn(*s, generator=g).half().to(DEV)  # noqa: E731
    ids = ["a", "b"][:B]
    for s in ids:
        m.allocate_sequence(s)
    ctx = m.begin_forward(ids, [40, 3][:B])
    ctx.attend(0, rnd(B, 40, Hq, D), rnd(B, 40, Hkv, D), rnd(B, 40, Hkv, D), Hq, Hkv)
    m.end_forward(ctx)
    ctx = m.begin_forward(ids, [1] * B)
    cos, sin = (torch.randn(80, D, generator=g).to(DEV) for _ in range(2))
    q, k, v = rnd(B, 1, Hq, D), rnd(B, 1, Hkv, D), rnd(B, 1, Hkv, D)
    if form == "heads":
        (ctx.attend_rope(0, q, k, v, cos, sin, Hq, Hkv) if rope else ctx.attend(0, q, k, v, Hq, Hkv))
        q = rnd(B, 1, 2 * Hq, D)
    elif form == "heads_no_multiple":
        q = rnd(B, 1, 5, D)
    elif form == "one_row":  # a single row: its stride says nothing
        q, k, v = (x.as_strided(x.shape, (3, D, D, 1)) for x in (q, k, v))
    elif form == "shared_kv":
        k, v = k[:1].expand(B, 1, Hkv, D), v[:1].expand(B, 1, Hkv, D)
    elif form == "flat_kv":
        k, v = k[:, 0], v[:, 0]
    elif form == "heads_apart":
        q = rnd(B, Hq, 3, D).transpose(1, 2)[:, :1]
    elif form == "one_head":
        q = rnd(B, Hq, 3, D).transpose(1, 2)[:, :1]
    elif form == "cpu_sin":
        sin = sin.cpu()
    elif form == "cpu_q":
        q = q.cpu()
    else:
        k = k.double()

    def separate(kc, vc):
        p = ctx._plan
        if rope:
            r = K.rope_append(q, k, v, p.pos_for(1), p.slots_for(1), cos, sin, kc, vc)
        else:
            K.append_kv(k, v, p.slots_for(1), kc, vc)
            r = q
        return K.paged_decode(r[:, 0], kc, vc, p.indptr, p.indices, p.lpl, p.total_pages).view(B, 1, -1)

    kc, vc = m.k[0].clone(), m.v[0].clone()
    call = lambda: (ctx.attend_rope(0, q, k, v, cos, sin, Hq, Hkv) if rope  # noqa: E731
                    else ctx.attend(0, q, k, v, Hq, Hkv))
    try:
        want = separate(kc, vc)
    except (ValueError, TypeError, K._lib.KernelLibraryError) as e:
        with pytest.raises(type(e)):
            call()
        return
    out = call()
    torch.cuda.synchronize()
    assert torch.equal(out, want) and torch.equal(m.k[0], kc) and torch.equal(m.v[0], vc)


@pytest.mark.gpu
@pytest.mark.parametrize("backend", ["contiguous", "paged"])
@pytest.mark.parametrize("others", [1, 70])
def test_decode_forwards_of_other_batches_in_between(backend, others):
    """The layers of a decode forward of 40 sequences with another forward's layer after
    each: the chunk layout recorded by the first layer is not read once the other forward's
    call has used the workspace, whatever its size. Outputs and pools as with the forwards
    one after the other."""
    from nanoslg_amd.kv_cache import ContiguousKVCache, KVCacheConfig, PagedKVCache
    L, Hq, Hkv, D, B = 3, 8, 2, 64, 40
    ids = ["s%d" % i for i in range(B + others)]
    lens = [100 + 37 * i % 900 for i in range(B)] + [20 + i for i in range(others)]
    cfg = dict(num_layers=L, num_kv_heads=Hkv, num_qo_heads=Hq, head_dim=D, dtype=torch.float16,
               device=torch.device(DEV), backend=backend)

    def outputs(in_turn):
        g = torch.Generator().manual_seed(8)
        rnd = lambda *s: torch.randn(*s, generator=g).half().to(DEV)  # noqa: E731
        if backend == "paged":
            m = PagedKVCache(KVCacheConfig(max_pages=sum(-(-n // 16) + 1 for n in lens) + 2, page_size=16,
                                           enable_prefix_caching=False, **cfg))
        else:
            m = ContiguousKVCache(KVCacheConfig(max_batch_size=len(ids), max_seq_len=1024, **cfg))
        for s in ids:
            m.allocate_sequence(s)
        m.end_forward(m.begin_forward(ids, lens))
        pool = m if backend == "contiguous" else m.pool
        pool.k.copy_(rnd(*pool.k.shape))
        pool.v.copy_(rnd(*pool.v.shape))
        batches = [ids[:B], ids[B:]]
        inputs = [[(rnd(len(b), 1, Hq, D), rnd(len(b), 1, Hkv, D), rnd(len(b), 1, Hkv, D)) for _ in range(L)]
                  for b in batches]
        out = []
        if in_turn:
            forwards = [m.begin_forward(b, [1] * len(b)) for b in batches]
            for layer in range(L):
                out += [f.attend(layer, *x[layer], Hq, Hkv) for f, x in zip(forwards, inputs)]
        else:
            done = []
            for b, x in zip(batches, inputs):
                f = m.begin_forward(b, [1] * len(b))
                done.append([f.attend(layer, *x[layer], Hq, Hkv) for layer in range(L)])
            out = [o for pair in zip(*done) for o in pair]
        torch.cuda.synchronize()
        return out + [pool.k, pool.v]

    for a, b in zip(outputs(True), outputs(False)):
        assert torch.equal(a, b)

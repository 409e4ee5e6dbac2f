"""Prefill calls of few row tiles, whose keys are cut into runs and merged: against the
oracle's fp32 attention within the attention tolerance, and the forward's K/V write of a
cut call bit-identical to nslg_append_kv. Keys at the edges of key tiles, runs and (in one
workgroup, cut or not) page-id windows; sequences shorter than a run, without new tokens, and of one new token; padded
grids; every head dim, GQA group 1, 4 and 16."""
import numpy as np
import pytest
import torch

from test_gpu_kernels import ATOL, RTOL, _prefill_case

DEV = "cuda:0"

CASES = [  # lens, new tokens, Hq, Hkv, D, page size
    ([768], [1], 32, 8, 128, 16),               # the shortest sequence that is cut
    ([769], [17], 32, 8, 128, 16),              # a last run of one key
    ([4096 + 31], [31], 8, 8, 128, 1),          # G = 1, 32 runs, one-token pages
    ([6000, 300, 900], [33, 0, 5], 32, 8, 128, 16),
    ([1600, 1500], [150, 70], 16, 1, 128, 48),  # G = 16
    ([2100], [300], 32, 8, 64, 16),
    ([700, 3000], [1, 129], 16, 4, 256, 16),
]


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("case", range(len(CASES)))
def test_prefill_in_runs_matches_oracle(case, dtype, monkeypatch):
    from nanoslg_amd import kernels as K
    lens, news, Hq, Hkv, D, ps = CASES[case]
    got = []
    orig = K._prefill_workspace
    monkeypatch.setattr(K, "_prefill_workspace", lambda *a: got.append(orig(*a)) or got[-1])
    out, ref = _prefill_case(lens, news, Hq, Hkv, D, ps, dtype, seed=700 + case)
    assert got and got[0][2] > 256  # the call had room for runs
    torch.testing.assert_close(out, ref, atol=ATOL, rtol=RTOL)


@pytest.mark.gpu
@pytest.mark.parametrize("grid", [False, True])
@pytest.mark.parametrize("dtype,D", [(torch.float16, 128), (torch.bfloat16, 64), (torch.float16, 256)])
def test_prefill_in_runs_writes_the_new_rows(dtype, D, grid):
    """The fused write of a call cut into runs: pool bytes as append_kv leaves them, the
    result that of append_kv then prefill; tokens across a run's end and a page's."""
    from nanoslg_amd import kernels as K
    Hq, Hkv, ps, start, news = 16, 4, 16, [1000, 1270], [90, 25]
    g = torch.Generator().manual_seed(90 + D)
    npg = [-(-(s + n) // ps) for s, n in zip(start, news)]
    P, W = sum(npg) + 2, max(news) + 3
    ids = np.random.default_rng(9).permutation(np.arange(1, P))[:sum(npg)].astype(np.int32)
    indptr = np.array([0, npg[0], sum(npg)], np.int32)
    lpl = np.array([(s + n - 1) % ps + 1 for s, n in zip(start, news)], np.int32)
    qo = np.array([0, news[0], sum(news)], np.int32)
    rows = np.concatenate([b * W + 3 + np.arange(n) for b, n in enumerate(news)]).astype(np.int32)
    slots = np.full(2 * W, -1, np.int32)
    for b in range(2):
        pos = start[b] + np.arange(news[b])
        slots[b * W + 3 + np.arange(news[b])] = ids[indptr[b] + pos // ps] * ps + pos % ps
    n = 2 * W if grid else sum(news)
    if not grid:
        slots = slots[rows]
    q, k, v = (torch.randn(n, h, D, generator=g).to(dtype).to(DEV) for h in (Hq, Hkv, Hkv))
    k1, v1 = (torch.randn(P, ps, Hkv, D, generator=g).to(dtype).to(DEV) for _ in range(2))
    k2, v2 = k1.clone(), v1.clone()
    d = lambda a: torch.from_numpy(a).to(DEV)  # noqa: E731
    plan = (d(indptr), d(ids), d(lpl))
    kw = dict(q_rows=d(rows), grid_width=W) if grid else {}
    o1 = K.paged_prefill_append(q, d(qo), sum(news), max(news), k, v, k1, v1, *plan, **kw)
    K.append_kv(k, v, d(slots), k2, v2)
    o2 = K.paged_prefill(q, d(qo), sum(news), max(news), k2, v2, *plan, **kw)
    torch.cuda.synchronize()
    assert torch.equal(k1, k2) and torch.equal(v1, v2) and torch.equal(o1, o2)


@pytest.mark.gpu
@pytest.mark.parametrize("dtype,D", [(torch.float16, 128), (torch.bfloat16, 256), (torch.float32, 64)])
@pytest.mark.parametrize("news,W", [([1, 0, 700], 700), ([3], 2500), ([0, 0], 9)])
def test_pad_rows_shared_by_the_launch(news, W, dtype, D):
    """Padded grids of mostly pad rows (more of them than the launch has waves, a sequence
    without tokens, no token at all): pad rows zero, token rows those of the ragged call."""
    from nanoslg_amd import kernels as K
    Hq, Hkv, ps, B = 8, 2, 16, len(news)
    g = torch.Generator().manual_seed(W)
    npg = [-(-n // ps) for n in news]
    qo = np.concatenate([[0], np.cumsum(news)]).astype(np.int32)
    indptr = np.concatenate([[0], np.cumsum(npg)]).astype(np.int32)
    ids = np.arange(1, sum(npg) + 1, dtype=np.int32) if sum(npg) else np.zeros(1, np.int32)
    lpl = np.array([(n - 1) % ps + 1 if n else 0 for n in news], np.int32)
    rows = np.concatenate([b * W + W - n + np.arange(n) for b, n in enumerate(news)] + [np.zeros(1)]).astype(np.int32)
    k, v = (torch.randn(sum(npg) + 1, ps, Hkv, D, generator=g).to(dtype).to(DEV) for _ in range(2))
    q = torch.randn(B * W, Hq, D, generator=g).to(dtype).to(DEV)
    d = lambda a: torch.from_numpy(a).to(DEV)  # noqa: E731
    plan = (k, v, d(indptr), d(ids), d(lpl))
    T = sum(news)
    out = torch.full_like(q, 7.0)
    K.paged_prefill(q, d(qo), T, max(news), *plan, out=out, q_rows=d(rows), grid_width=W)
    at = torch.from_numpy(rows[:T].astype(np.int64)).to(DEV)
    want = torch.zeros_like(q)
    if T:
        want[at] = K.paged_prefill(q[at].contiguous(), d(qo), T, max(news), *plan)
    torch.cuda.synchronize()
    assert torch.equal(out, want)


ORDERS = [  # new tokens per sequence (each over a few cached keys)
    [300, 256, 310, 290],                       # near-uniform tile counts: rounds, one sequence short of a tile
    [700, 1, 0, 64, 65, 300],                   # sequence by sequence; none, one and several tiles
    [(7 * i) % 90 for i in range(40)],          # more than 32 sequences
    [(11 * i) % 70 + 1 for i in range(70)],     # more than 64 sequences
]


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.float16, torch.float32])
@pytest.mark.parametrize("case", range(len(ORDERS)))
def test_every_row_tile_is_taken_once(case, dtype):
    """Every order of the row tiles against the oracle: a tile left out leaves its rows
    unwritten."""
    from test_gpu_kernels import F32_TOL
    news = ORDERS[case]
    out, ref = _prefill_case([n + 5 for n in news], news, 8, 2, 64, 16, dtype, seed=760 + case)
    torch.testing.assert_close(out, ref, **(F32_TOL if dtype == torch.float32 else dict(atol=ATOL, rtol=RTOL)))


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.float16, torch.float32])
def test_rows_of_no_sequence_are_left_alone(dtype):
    """A call on part of a larger batch's ragged rows (qo_indptr starts past row 0), cut into
    runs: the part's rows as in a call of their own, the rows before and after unwritten,
    whatever the scratch held."""
    from nanoslg_amd import kernels as K
    Hq, Hkv, D, ps, lens, news, first = 8, 2, 128, 16, [1500, 900], [20, 7], 11
    g = torch.Generator().manual_seed(3)
    npg = [-(-n // ps) for n in lens]
    k, v = (torch.randn(sum(npg), ps, Hkv, D, generator=g).to(dtype).to(DEV) for _ in range(2))
    q = torch.randn(first + sum(news) + 5, Hq, D, generator=g).to(dtype).to(DEV)
    d = lambda *a: torch.tensor(a, dtype=torch.int32, device=DEV)  # noqa: E731
    plan = (k, v, d(0, npg[0], sum(npg)), torch.arange(sum(npg), dtype=torch.int32, device=DEV),
            d(*[(n - 1) % ps + 1 for n in lens]))
    T = sum(news)
    last = first + T
    # the same scratch bytes again, every count and sum in it 2 or more
    need = K._prefill_workspace(q, 2, Hq, D, last, max(news), max(lens))[2]
    assert need > 256
    torch.cuda.synchronize()
    torch.full((need,), 0x40, dtype=torch.uint8, device=DEV)
    out = torch.full_like(q, 7.0)
    K.paged_prefill(q, d(first, first + news[0], last), last, max(news), *plan, out=out)
    want = K.paged_prefill(q[first:last].contiguous(), d(0, news[0], T), T, max(news), *plan)
    torch.cuda.synchronize()
    assert (out[:first] == 7).all() and (out[last:] == 7).all()
    torch.testing.assert_close(out[first:last], want, atol=ATOL, rtol=RTOL)


@pytest.mark.gpu
def test_a_callers_workspace_is_used():
    """Calls cut into runs with the caller's workspace: nothing allocated but the output,
    the result that of a call without one, and a chunk layout that a decode call recorded in
    the workspace still read after them."""
    from nanoslg_amd import kernels as K
    Hq, Hkv, D, ps, L, n = 8, 2, 128, 16, 4000, 20
    g = torch.Generator().manual_seed(4)
    rnd = lambda *s: torch.randn(*s, generator=g).half().to(DEV)  # noqa: E731
    k, v, q, dq = rnd(L // ps, ps, Hkv, D), rnd(L // ps, ps, Hkv, D), rnd(n, Hq, D), rnd(1, Hq, D)
    kn, vn = k[-2:].reshape(-1, Hkv, D)[-n:].clone(), v[-2:].reshape(-1, Hkv, D)[-n:].clone()
    d = lambda *a: torch.tensor(a, dtype=torch.int32, device=DEV)  # noqa: E731
    plan = (d(0, L // ps), torch.arange(L // ps, dtype=torch.int32, device=DEV), d(ps))
    qo, out = d(0, n), torch.empty_like(q)
    ws = K.Workspace(DEV, 64 << 20)
    want = K.paged_prefill(q, qo, n, n, k, v, *plan)
    step = K.paged_decode(dq, k, v, *plan, L // ps, workspace=ws, layout=101)
    before = ws.buf.clone()
    for i in range(2):
        torch.cuda.synchronize()
        torch.cuda.reset_peak_memory_stats()
        base = torch.cuda.memory_allocated()
        K.paged_prefill(q, qo, n, n, k, v, *plan, out=out, workspace=ws)
        peak = torch.cuda.max_memory_allocated() - base
        assert i == 0 or peak == 0
        assert torch.equal(out, want)
    torch.cuda.reset_peak_memory_stats()
    base = torch.cuda.memory_allocated()
    o2 = K.paged_prefill_append(q, qo, n, n, kn, vn, k, v, *plan, workspace=ws)
    assert torch.cuda.max_memory_allocated() - base <= o2.numel() * 2 + 512
    assert torch.equal(o2, want) and torch.equal(ws.buf, before)
    assert torch.equal(K.paged_decode(dq, k, v, *plan, L // ps, workspace=ws, layout=-101), step)


def _room_for(runs, rows, D):
    """Scratch bytes that hold this many runs of a call of `rows` (token, query head) rows."""
    up = lambda x: -(-x // 256) * 256  # noqa: E731
    return 512 + up(rows * 4) + up(rows * runs * 8) + rows * runs * D * 4


@pytest.mark.gpu
@pytest.mark.parametrize("runs,L", [(1, 2070), (2, 4380), (1, 4500)])
@pytest.mark.parametrize("dtype,D", [(torch.float16, 128), (torch.bfloat16, 64), (torch.bfloat16, 256)])
def test_a_workgroup_reloads_its_page_window(dtype, D, runs, L, monkeypatch):
    """Keys of one workgroup past its 2048 page ids (one-token pages): attention against the
    oracle, and the fused write of new tokens on both sides of the window's end (key 2048 of
    an uncut call; 4352 and, at D = 256, 4160 in the second of two runs, which begins at
    2304 and 2112) bit-identical to append_kv."""
    from nanoslg_amd import kernels as K
    if runs == 2 and D == 256:
        L = 4170
    Hq, Hkv, n, orig = 8, 2, 60, K._prefill_workspace
    rows = n * Hq
    room = []

    def cut(*a):
        if runs == 1:
            return None, None, 0
        ws, ptr, nbytes = orig(*a)
        room.append(ws)
        assert nbytes >= _room_for(runs, rows, D)
        return ws, ptr, _room_for(runs, rows, D)

    monkeypatch.setattr(K, "_prefill_workspace", cut)
    out, ref = _prefill_case([L], [n], Hq, Hkv, D, 1, dtype, seed=L + D)
    torch.testing.assert_close(out, ref, atol=ATOL, rtol=RTOL)
    g = torch.Generator().manual_seed(L)
    ids = torch.randperm(L, generator=g).int()
    q, k, v = (torch.randn(n, h, D, generator=g).to(dtype).to(DEV) for h in (Hq, Hkv, Hkv))
    k1, v1 = (torch.randn(L + 3, 1, Hkv, D, generator=g).to(dtype).to(DEV) for _ in range(2))
    k2, v2 = k1.clone(), v1.clone()
    i32 = lambda *a: torch.tensor(a, dtype=torch.int32, device=DEV)  # noqa: E731
    plan = (i32(0, L), ids.to(DEV), i32(1))
    o1 = K.paged_prefill_append(q, i32(0, n), n, n, k, v, k1, v1, *plan)
    if runs > 1:
        assert (room[-1][256:256 + rows * 4].view(torch.int32) == runs).all()  # the runs of each row
    K.append_kv(k, v, ids[L - n:].to(DEV), k2, v2)
    o2 = K.paged_prefill(q, i32(0, n), n, n, k2, v2, *plan)
    torch.cuda.synchronize()
    assert torch.equal(k1, k2) and torch.equal(v1, v2) and torch.equal(o1, o2)


@pytest.mark.gpu
@pytest.mark.parametrize("call", ["prefill", "prefill_f32", "decode_f32", "decode"])
def test_partials_void_a_recorded_chunk_layout(call, monkeypatch):
    """A workspace that holds a decode call's chunk layout, then another call's partials: the
    layout's tag is gone, and the decode's next layer cuts its chunks anew."""
    from nanoslg_amd import kernels as K
    Hq, Hkv, D, ps, L, n = 8, 2, 128, 16, 4000, 20
    g = torch.Generator().manual_seed(4)
    rnd = lambda *s: torch.randn(*s, generator=g).half().to(DEV)  # noqa: E731
    k, v, q, dq = rnd(L // ps, ps, Hkv, D), rnd(L // ps, ps, Hkv, D), rnd(n, Hq, D), rnd(1, Hq, D)
    d = lambda *a: torch.tensor(a, dtype=torch.int32, device=DEV)  # noqa: E731
    plan = (d(0, L // ps), torch.arange(L // ps, dtype=torch.int32, device=DEV), d(ps))
    ws = K.Workspace(DEV, 64 << 20)
    tag = lambda: int(ws.buf[:8].view(torch.int64))  # noqa: E731
    step = K.paged_decode(dq, k, v, *plan, L // ps, workspace=ws, layout=102)
    assert tag() == 102
    monkeypatch.setattr(K.Workspace, "get_prefill", K.Workspace.get)  # one memory for both, as in a C program
    if call.startswith("prefill"):
        x = [t.float() for t in (q, k, v)] if call.endswith("f32") else [q, k, v]
        K.paged_prefill(x[0], d(0, n), n, n, x[1], x[2], *plan, workspace=ws)
    elif call == "decode_f32":
        K.paged_decode(dq.float(), k.float(), v.float(), *plan, L // ps, workspace=ws)
    else:
        K.paged_decode(dq, k, v, *plan, L // ps, workspace=ws)
    assert tag() == 0
    assert torch.equal(K.paged_decode(dq, k, v, *plan, L // ps, workspace=ws, layout=-102), step)

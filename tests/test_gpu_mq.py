"""GPU parity of the multi-query Q8_0-key decode that reads every tile once for
up to 64 (query, head) columns: against the single-query launches of the same
rows (query t of a call over n keys is a one-query call over its own key
count), at the edges of tiles, chunks, column groups and query groups."""
import numpy as np
import pytest

from oracle import oracle as O
from tests._data import kv_f16, q_f16, rel_err

pytestmark = pytest.mark.gpu


def _dev(a, dev):
    import torch
    return torch.from_numpy(np.ascontiguousarray(a)).to(dev)


def _both(dev, fmt, q, kb, vb, n, num_q, num_kv):
    """(one call with every query, one call per query) as float arrays."""
    import torch
    from qengine_amd import kvcache
    sub_n = q.shape[0]
    make, call = ((kvcache.decode_attn_q8_workspace, kvcache.decode_attn_q8) if fmt == "q8" else
                  (kvcache.decode_attn_q8k_tq3v_workspace, kvcache.decode_attn_q8k_tq3v))
    qd = _dev(q.view(np.uint16), dev).view(torch.float16)
    ws = make(num_q, num_kv, sub_n, n, dev)
    one = torch.zeros((sub_n, num_q, 256), dtype=torch.float16, device=dev)
    many = torch.zeros_like(one)
    kw = dict(num_q=num_q, num_kv=num_kv, scale=1 / 16)
    for _ in range(2):   # the second call finds the workspace as the first left it
        call(qd, kb, vb, one, ws, start_pos=n - sub_n, sub_n=sub_n, **kw)
    for t in range(sub_n):
        call(qd[t:t + 1].contiguous(), kb, vb, many[t:t + 1], ws, start_pos=n - sub_n + t, sub_n=1, **kw)
    torch.cuda.synchronize()
    return one.float().cpu().numpy(), many.float().cpu().numpy()


# Two fp16 roundings separate the paths: the probabilities (2^-11 relative, taken
# against different reference maxima; they average out over the keys) and the
# output (2^-11 of an element).  Per row, relative to the row's largest element:
# 2^-11 x 2 for the outputs plus as much for the sums.
TOL = 4 * 2.0 ** -11


@pytest.mark.parametrize("fmt", ["q8", "mixed"])
@pytest.mark.parametrize("n,num_q,num_kv,sub_n", [
    (8256, 16, 4, 2),       # whole tiles
    (8257, 16, 4, 3),       # one key past a tile
    (8319, 24, 4, 5),       # one key short of a tile, 30 columns
    (5000, 24, 4, 10),      # 60 columns: 4 dead ones in the last group
    (5000, 16, 4, 16),      # 64 columns
    (5000, 16, 4, 17),      # query groups
    (3000, 4, 4, 64),       # GQA 1: 64 queries
    (3000, 16, 2, 9),       # GQA 8, two kv heads
    (33000, 8, 1, 7),       # one kv head, many chunks
    (70, 16, 4, 70),        # no history: chunks with causal keys only, some queries see none of theirs
    (2100, 40, 8, 40),      # GQA 5, queries past one 64-column group
])
def test_multi_query_matches_single_queries(dev, fmt, n, num_q, num_kv, sub_n):
    print(f"mq {fmt} n={n} num_q={num_q} num_kv={num_kv} sub_n={sub_n}", flush=True)
    rng = np.random.default_rng(n + num_q + sub_n)
    kb = _dev(O.q8_encode(kv_f16(rng, n, num_kv, 256)).view(np.uint8), dev)
    v16 = kv_f16(rng, n, num_kv, 256)
    vb = _dev((O.q8_encode(v16) if fmt == "q8" else O.tq3_encode(v16)).view(np.uint8), dev)
    # queries of growing magnitude: sharp rows raise their reference maximum late
    q = (q_f16(rng, sub_n, num_q, 256).astype(np.float32) * np.linspace(0.5, 4, sub_n)[:, None, None]).astype(np.float16)
    one, many = _both(dev, fmt, q, kb, vb, n, num_q, num_kv)
    assert np.isfinite(many).all()
    assert rel_err(one, many) < TOL


@pytest.mark.parametrize("fmt,plane", [("q8", "k"), ("q8", "v"), ("mixed", "k"), ("mixed", "v")])
def test_non_finite_rows_stay_with_the_queries_that_see_them(dev, fmt, plane):
    """An inf in the row of key n - 6 (a row of the block itself) reaches no
    query before it.  Later ones: an inf value row makes the same elements
    non-finite as in single-query calls; an inf key row makes the sum of its
    chunk NaN, and the merge drops a chunk without a positive sum, so those
    rows depend on where the chunks lie and are not compared."""
    n, num_q, num_kv, sub_n = 4300, 16, 4, 16
    seen = sub_n - 6
    rng = np.random.default_rng(5)
    k16, v16 = kv_f16(rng, n, num_kv, 256), kv_f16(rng, n, num_kv, 256)
    (k16 if plane == "k" else v16)[n - 6, 1, 37] = np.inf
    kb = _dev(O.q8_encode(k16).view(np.uint8), dev)
    vb = _dev((O.q8_encode(v16) if fmt == "q8" else O.tq3_encode(v16)).view(np.uint8), dev)
    one, many = _both(dev, fmt, q_f16(rng, sub_n, num_q, 256), kb, vb, n, num_q, num_kv)
    assert np.isfinite(many[:seen]).all() and np.isfinite(one[:seen]).all()
    assert rel_err(one[:seen], many[:seen]) < TOL
    if plane == "v":
        bad = ~np.isfinite(many)
        assert bad[seen:].any() and np.array_equal(bad, ~np.isfinite(one))
        assert rel_err(np.where(bad, 0.0, one), np.where(bad, 0.0, many)) < TOL


def _call(fmt):
    from qengine_amd import kvcache
    return {"q8": (kvcache.decode_attn_q8_workspace, kvcache.decode_attn_q8),
            "mixed": (kvcache.decode_attn_q8k_tq3v_workspace, kvcache.decode_attn_q8k_tq3v),
            "tq3": (kvcache.decode_attn_tq3_workspace, kvcache.decode_attn_tq3)}[fmt]


def _caches(rng, dev, fmt, n, num_kv):
    k16, v16 = kv_f16(rng, n, num_kv, 256), kv_f16(rng, n, num_kv, 256)
    return (_dev((O.tq3_encode(k16) if fmt == "tq3" else O.q8_encode(k16)).view(np.uint8), dev),
            _dev((O.q8_encode(v16) if fmt == "q8" else O.tq3_encode(v16)).view(np.uint8), dev))


@pytest.mark.parametrize("fmt", ["q8", "mixed", "tq3"])
@pytest.mark.parametrize("n,num_q,num_kv,sub_n", [
    (2048, 16, 4, 1040),    # 260 working workgroups: the first count past 256
    (2048, 16, 4, 2048),    # no history, two rounds
    (4000, 64, 8, 300),     # GQA 8
    (1500, 24, 3, 345),     # 3 kv heads: the grid's rounding to 8 chunks leaves work past id 255
])
def test_calls_past_one_round_of_the_gpu(dev, fmt, n, num_q, num_kv, sub_n):
    """More (query group, kv head) pairs than CUs: the call is several rounds of
    workgroups, none of which may wait for one that has no CU yet.  Against the
    same queries 8 at a time (at most 64 workgroups each)."""
    import torch
    print(f"mq rounds {fmt} n={n} num_q={num_q} num_kv={num_kv} sub_n={sub_n}", flush=True)
    make, call = _call(fmt)
    rng = np.random.default_rng(n + sub_n)
    kb, vb = _caches(rng, dev, fmt, n, num_kv)
    qd = _dev(q_f16(rng, sub_n, num_q, 256).view(np.uint16), dev).view(torch.float16)
    one, many = torch.zeros_like(qd), torch.zeros_like(qd)
    ws = make(num_q, num_kv, sub_n, n, dev)
    kw = dict(num_q=num_q, num_kv=num_kv, scale=1 / 16)
    call(qd, kb, vb, one, ws, start_pos=n - sub_n, sub_n=sub_n, **kw)
    torch.cuda.synchronize()
    for t in range(0, sub_n, 8):
        m = min(8, sub_n - t)
        call(qd[t:t + m], kb, vb, many[t:t + m], ws, start_pos=n - sub_n + t, sub_n=m, **kw)
    torch.cuda.synchronize()
    one, many = one.float().cpu().numpy().reshape(sub_n, -1), many.float().cpu().numpy().reshape(sub_n, -1)
    assert np.isfinite(many).all()
    # Per query, 2-norms over all its heads: each path rounds its weights and its
    # outputs to fp16 (2^-11 / sqrt(3) rms each), so two differ by about 1.15 x 2^-11.
    # (rel_err's single elements are no measure over 8 million of them: the error of an
    # outlier channel, 8 x the others', may fall in a row whose largest element is small.)
    assert (np.linalg.norm(one - many, axis=1) / np.linalg.norm(many, axis=1)).max() < TOL


@pytest.mark.parametrize("fmt", ["q8", "tq3"])
def test_two_calls_on_two_streams(dev, fmt):
    """Two verify calls of 256 workgroups each, one workgroup per CU, side by side
    on two streams with workspaces of their own: neither may need all of its
    workgroups to be resident."""
    import torch
    make, call = _call(fmt)
    n, num_q, num_kv, sub_n = 32784, 16, 4, 16
    rng = np.random.default_rng(9)
    kb, vb = _caches(rng, dev, fmt, n, num_kv)
    q = [_dev(q_f16(rng, sub_n, num_q, 256).view(np.uint16), dev).view(torch.float16) for _ in range(2)]
    ws = [make(num_q, num_kv, sub_n, n, dev) for _ in range(2)]
    kw = dict(num_q=num_q, num_kv=num_kv, start_pos=n - sub_n, sub_n=sub_n, scale=1 / 16)
    want = [torch.zeros_like(x) for x in q]
    for i in range(2):
        call(q[i], kb, vb, want[i], ws[i], **kw)
    torch.cuda.synchronize()
    streams = [torch.cuda.Stream() for _ in range(2)]
    got = [[torch.zeros_like(x) for _ in range(8)] for x in q]
    torch.cuda.synchronize()
    for r in range(8):
        for i, s in enumerate(streams):
            with torch.cuda.stream(s):
                call(q[i], kb, vb, got[i][r], ws[i], **kw)
    torch.cuda.synchronize()
    for i in range(2):
        for r in range(8):
            assert torch.equal(got[i][r], want[i]), f"stream {i}, call {r}"


def _exact_q8(rng, n, num_kv):
    """Q8_0 rows whose scales are powers of two, so that their fp16 values are
    exact: (blocks, values float64 [n][num_kv][256])."""
    code = rng.integers(-127, 128, size=(n, num_kv, 8, 32)).astype(np.int8)
    scale = (2.0 ** -rng.integers(5, 9, size=(n, num_kv, 8))).astype(np.float16)
    b = np.zeros((n, num_kv, 8, 36), np.uint8)
    b[..., :32] = code.view(np.uint8)
    b[..., 34:] = scale[..., None].view(np.uint8)
    return b, (code * scale[..., None].astype(np.float64)).reshape(n, num_kv, 256)


@pytest.mark.parametrize("sub_n,num_q,num_kv", [(6, 16, 4), (16, 16, 4), (9, 24, 4)])
def test_weights_keep_more_than_fp16(dev, sub_n, num_q, num_kv):
    """Over caches whose decoded values are exact only the weights are left to round.
    Their fp16 roundings alone would be 2^-12 of a row; with their rests in a product
    of their own what remains is the fp32 sums (2,000 terms, about 2^-20), so the
    split API's rows are held to 2^-15 and all but the ties among the decode's fp16
    rows are the exact ones rounded (error 2^-20 against a spacing of at least 2^-11:
    1 in 500 lies across; with rounded weights every third did)."""
    import torch
    from qengine_amd import kvcache
    n, ks, gqa = 2000, 32, num_q // num_kv
    rng = np.random.default_rng(sub_n + num_q)
    (kb, k), (vb, v) = _exact_q8(rng, n, num_kv), _exact_q8(rng, n, num_kv)
    q = (q_f16(rng, sub_n, num_q, 256).astype(np.float32) * 0.4).astype(np.float16)
    s = np.einsum("tqd,nqd->tqn", q.astype(np.float64), np.repeat(k, gqa, 1)) / 16
    s = np.where(np.arange(n) > n - sub_n + np.arange(sub_n)[:, None, None], -np.inf, s)
    p = np.exp(s - s.max(-1, keepdims=True))
    vq = np.repeat(v, gqa, 1)
    want = np.einsum("tqn,nqd->tqd", p / p.sum(-1, keepdims=True), vq)
    kd, vd, qd = _dev(kb, dev), _dev(vb, dev), _dev(q.view(np.uint16), dev).view(torch.float16)
    kw = dict(num_q=num_q, num_kv=num_kv, start_pos=n - sub_n, sub_n=sub_n, scale=1 / 16)
    out = torch.zeros_like(qd)
    kvcache.decode_attn_q8(qd, kd, vd, out, kvcache.decode_attn_q8_workspace(num_q, num_kv, sub_n, n, dev), **kw)
    pm, pl = (torch.zeros((num_q, sub_n, ks), device=dev) for _ in range(2))
    po = torch.zeros((num_q, sub_n, ks, 256), device=dev)
    kvcache.attn_split_q8(qd, kd, vd, pm, pl, po, sub_n_max=sub_n, active_end_max=n, k_splits=ks, **kw)
    torch.cuda.synchronize()
    differ = np.mean(out.cpu().numpy().view(np.uint16) != want.astype(np.float16).view(np.uint16))
    assert differ < 0.01, differ
    pm, pl, po = (x.cpu().numpy().astype(np.float64) for x in (pm, pl, po))
    w = np.exp(pm - pm.max(-1, keepdims=True))
    got = np.einsum("qtz,qtzd->tqd", w / (w * pl).sum(-1, keepdims=True), po)
    assert np.linalg.norm(got - want) / np.linalg.norm(want) < 2.0 ** -15


@pytest.mark.parametrize("sub_n", [16, 7])
def test_tq3_workspace_of_the_longer_chunks(dev, sub_n):
    """A workspace that holds one record per 512 keys, which is what a TQ3 call of
    many queries needs at least, serves it with chunks of that length; so does the
    8 MiB scratch of the allocation-free call, too small for the shorter chunks of 16
    queries over 4,096 keys.  One byte less is refused."""
    import torch
    from qengine_amd import kvcache
    n, num_q, num_kv, chunks = 4096, 16, 4, 8
    rng = np.random.default_rng(sub_n)
    kb, vb = _caches(rng, dev, "tq3", n, num_kv)
    qd = _dev(q_f16(rng, sub_n, num_q, 256).view(np.uint16), dev).view(torch.float16)
    kw = dict(num_q=num_q, num_kv=num_kv, start_pos=n - sub_n, sub_n=sub_n, scale=1 / 16)
    rows = num_q * sub_n * chunks
    need = (256 + 16 * rows + 255) // 256 * 256 + 1024 * rows
    full_ws = kvcache.decode_attn_tq3_workspace(num_q, num_kv, sub_n, n, dev)
    assert need < full_ws.numel() * full_ws.element_size()
    full, small, noalloc = (torch.zeros_like(qd) for _ in range(3))
    kvcache.decode_attn_tq3(qd, kb, vb, full, full_ws, **kw)
    kvcache.decode_attn_tq3(qd, kb, vb, small, torch.zeros(need, dtype=torch.uint8, device=dev), **kw)
    kvcache.decode_attn_tq3_noalloc(qd, kb, vb, noalloc, **kw)
    torch.cuda.synchronize()
    assert rel_err(full.float().cpu().numpy(), small.float().cpu().numpy()) < TOL
    if sub_n == 16:
        assert torch.equal(noalloc, small)
    else:   # (the shorter chunks fit the scratch)
        assert torch.equal(noalloc, full)
    with pytest.raises(Exception):
        kvcache.decode_attn_tq3(qd, kb, vb, small, torch.zeros(need - 1, dtype=torch.uint8, device=dev), **kw)


@pytest.mark.parametrize("sink,window", [(0, 100), (64, 0), (33, 1000), (70, 64), (1, 3000), (4, 1 << 20), (5000, 1)])
@pytest.mark.parametrize("sub_n,num_q", [(16, 16), (7, 16), (5, 24)])
def test_tq3_sink_and_window(dev, sub_n, num_q, sink, window):
    """Tiles that the sink / window rule shows whole to every query of a block, to
    none of them (their rows, with an inf norm among them, are left out), and to
    some, against the same queries one at a time (over rows without the inf)."""
    import torch
    from qengine_amd import kvcache
    n, num_kv = 4300, 4
    rng = np.random.default_rng(sink + window + sub_n)
    k16, v16 = kv_f16(rng, n, num_kv, 256), kv_f16(rng, n, num_kv, 256)
    kb, vb = O.tq3_encode(k16).view(np.uint8).reshape(n, -1), O.tq3_encode(v16).view(np.uint8).reshape(n, -1)
    end = n - sub_n + 1
    unseen = [r for r in range(end) if not any(
        r // 32 * 32 < sink or min(r // 32 * 32 + 32, e) > e - window for e in range(end, n + 1))]
    clean = _dev(vb.copy(), dev)
    for r in unseen[::97]:
        vb[r, :4] = np.frombuffer(np.float32(np.inf).tobytes(), np.uint8)
    kd, vd = _dev(kb, dev), _dev(vb, dev)
    qd = _dev(q_f16(rng, sub_n, num_q, 256).view(np.uint16), dev).view(torch.float16)
    one, many = torch.zeros_like(qd), torch.zeros_like(qd)
    ws = kvcache.decode_attn_tq3_workspace(num_q, num_kv, sub_n, n, dev)
    kw = dict(num_q=num_q, num_kv=num_kv, scale=1 / 16, sink_tok=sink, window_tok=window)
    kvcache.decode_attn_tq3(qd, kd, vd, one, ws, start_pos=n - sub_n, sub_n=sub_n, **kw)
    for t in range(sub_n):
        kvcache.decode_attn_tq3(qd[t:t + 1].contiguous(), kd, clean, many[t:t + 1], ws, start_pos=n - sub_n + t, sub_n=1, **kw)
    torch.cuda.synchronize()
    one, many = one.float().cpu().numpy(), many.float().cpu().numpy()
    assert np.isfinite(many).all() and rel_err(one, many) < TOL


@pytest.mark.parametrize("fmt", ["tq3", "q8", "mixed"])
def test_one_workspace_for_calls_of_every_kind(dev, fmt):
    """One workspace in turn for one query, for a few and for many: each kind lays its
    records out in its own way and leaves every tag clear for the next."""
    import torch
    make, call = _call(fmt)
    num_q, num_kv, n_max = 16, 4, 6000
    rng = np.random.default_rng(17)
    kb, vb = _caches(rng, dev, fmt, n_max, num_kv)
    ws = make(num_q, num_kv, 20, n_max, dev)
    kw = dict(num_q=num_q, num_kv=num_kv, scale=1 / 16)
    for n, sub_n in [(6000, 1), (5000, 16), (301, 1), (6000, 20), (4097, 3), (700, 12), (6000, 16), (6000, 1)]:
        qd = _dev(q_f16(rng, sub_n, num_q, 256).view(np.uint16), dev).view(torch.float16)
        got, want = torch.zeros_like(qd), torch.zeros_like(qd)
        call(qd, kb, vb, got, ws, start_pos=n - sub_n, sub_n=sub_n, **kw)
        call(qd, kb, vb, want, make(num_q, num_kv, 20, n_max, dev), start_pos=n - sub_n, sub_n=sub_n, **kw)
        torch.cuda.synchronize()
        assert torch.isfinite(got).all() and torch.equal(got, want), (n, sub_n)


@pytest.mark.parametrize("fmt", ["tq3", "mixed"])
@pytest.mark.parametrize("rows,scale", [(slice(100, 140), 40), (slice(1800, 1801), 2500), (slice(2990, 3000), 300)])
def test_large_value_norms(dev, fmt, rows, scale):
    """Block norms above 128 (here 500 to 50,000) end the slack of the reference maximum
    from their tile on, so that weight x norm stays inside fp16; tiles before them were
    taken with it."""
    import torch
    make, call = _call(fmt)
    n, num_q, num_kv, sub_n = 3000, 16, 4, 12
    rng = np.random.default_rng(scale)
    k16, v16 = kv_f16(rng, n, num_kv, 256), kv_f16(rng, n, num_kv, 256).astype(np.float32)
    v16[rows] = np.clip(v16[rows], -8, 8) * scale
    kb = _dev((O.tq3_encode(k16) if fmt == "tq3" else O.q8_encode(k16)).view(np.uint8), dev)
    vb = _dev(O.tq3_encode(v16.astype(np.float16)).view(np.uint8), dev)
    q = (q_f16(rng, sub_n, num_q, 256).astype(np.float32) * np.linspace(0.5, 4, sub_n)[:, None, None]).astype(np.float16)
    qd = _dev(q.view(np.uint16), dev).view(torch.float16)
    ws = make(num_q, num_kv, sub_n, n, dev)
    one, many = torch.zeros_like(qd), torch.zeros_like(qd)
    kw = dict(num_q=num_q, num_kv=num_kv, scale=1 / 16)
    call(qd, kb, vb, one, ws, start_pos=n - sub_n, sub_n=sub_n, **kw)
    for t in range(sub_n):
        call(qd[t:t + 1].contiguous(), kb, vb, many[t:t + 1], ws, start_pos=n - sub_n + t, sub_n=1, **kw)
    torch.cuda.synchronize()
    one, many = one.float().cpu().numpy(), many.float().cpu().numpy()
    assert np.isfinite(many).all() and rel_err(one, many) < TOL


def test_non_finite_value_scale_in_a_whole_tile(dev):
    """An inf in a value row of the history, which every query sees: the same elements
    are non-finite as in single-query calls, the others as near to them as ever."""
    n, num_q, num_kv, sub_n = 4300, 16, 4, 16
    rng = np.random.default_rng(6)
    k16, v16 = kv_f16(rng, n, num_kv, 256), kv_f16(rng, n, num_kv, 256)
    v16[1500, 2, 77] = np.inf
    kb, vb = (_dev(O.q8_encode(x).view(np.uint8), dev) for x in (k16, v16))
    one, many = _both(dev, "q8", q_f16(rng, sub_n, num_q, 256), kb, vb, n, num_q, num_kv)
    bad = ~np.isfinite(many)
    assert bad.any() and np.array_equal(bad, ~np.isfinite(one))
    assert rel_err(np.where(bad, 0.0, one), np.where(bad, 0.0, many)) < TOL

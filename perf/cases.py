"""The work that a program using this library has it do, as cases that can be timed.

A program that serves a model over compressed KV caches calls, per layer: the
decode step of one token (new K/V row appended, one query per head attended),
the verify of a speculative block, a chunk of a prompt, a batched step over a
paged pool, the reference's split + merge pair, and the bulk codecs.  Head
counts are the ones this repository is configured, tested and benchmarked
with: 4 KV heads of dimension 256 under 16 or 24 query heads (GQA 4 and 6).

Caches are built here in plain torch from fp16 rows of N(0, 1) with 2% of the
channels of each head scaled by 8, so that `exact` can decode the same bytes
in 64 bits without the library.
"""
import math

import numpy as np
import torch

from qengine_amd import kvcache

HD = 256
DEV = "cuda"


# ---------------------------------------------------------------------------
# cases
# ---------------------------------------------------------------------------

def listed():
    return [
        # a chat's first tokens: one layer's decode step over a few hundred
        # keys, where launch, setup and merge latency are all there is
        dict(name="step_short", kind="decode", num_q=16, num_kv=4, ctx=701, sub_n=1, layers=1,
             append=True, tree=False),
        # the benchmark's headline: one token through 8 layers at 32K keys
        dict(name="token_32k", kind="decode", num_q=16, num_kv=4, ctx=32767, sub_n=1, layers=8,
             append=False, tree=False),
        # the drop-in pair of the reference's decode step (split-K 8, partials
        # in its layout, then the merge) at the 18K context it quotes, GQA 6
        dict(name="split_18k", kind="split", fmt="tq3", num_q=24, num_kv=4, ctx=18016, sub_n=1,
             k_splits=8),
        # speculative decoding: a 16-token block appended and attended, 128K keys
        dict(name="verify16_128k", kind="decode", num_q=16, num_kv=4, ctx=131072, sub_n=16, layers=1,
             append=True, tree=False),
        # the same through block selection (64 of 2049 blocks of 64 keys)
        dict(name="sparse16_128k", kind="sparse", num_q=16, num_kv=4, ctx=131072, sub_n=16, top_k=64,
             k_splits=8),
        # Q8_0 cache: a decode step at 4K keys, the append in the launch
        dict(name="q8_step_4k", kind="q8", num_q=16, num_kv=4, ctx=4096, sub_n=1),
        # Q8_0 cache: a 16-token speculative block over an 18K context
        dict(name="q8_verify16_18k", kind="q8", num_q=16, num_kv=4, ctx=18016, sub_n=16),
        # Q8_0 keys, TQ3 values: a decode step (both appends, the attention) at 32K
        dict(name="mixed_step_32k", kind="mixed", num_q=16, num_kv=4, ctx=32767, sub_n=1),
        # continuous batching: 8 slots of 1K..64K keys in 256-token blocks, four
        # of them on a shared 4096-token prefix, one token appended to each, GQA 6
        dict(name="paged_8slots", kind="paged", num_q=24, num_kv=4, n_slots=8, ctx_lo=1024,
             ctx_hi=65536, block_tokens=256, ctx_seed=4, shared=True),
        # a long prompt's later chunk: 2048 tokens over a 128K history
        dict(name="prefill_128k", kind="prefill", num_q=16, num_kv=4, start=131072, n_tok=2048),
        # a short prompt: its only chunk, ragged, no history, GQA 6
        dict(name="prefill_first", kind="prefill", num_q=24, num_kv=4, start=0, n_tok=777),
        # a prompt's K and V rows encoded into the TQ3 cache in bulk
        dict(name="append_32k", kind="codec", fmt="tq3", op="append", num_kv=4, n_tok=32768),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["decode", "decode", "decode", "split", "sparse", "q8", "q8", "mixed", "paged",
                       "prefill", "prefill", "codec"])
    gqa6 = rng.random() < 0.35
    c = dict(kind=kind, num_q=24 if gqa6 else 16, num_kv=4)
    if kind == "decode":
        sub_n = rng.choice([1, 1, rng.randint(2, 16)])
        c.update(ctx=_log(rng, 300, 131072), sub_n=sub_n, layers=rng.choice([1, 1, 4]) if sub_n == 1 else 1,
                 append=rng.random() < 0.6, tree=sub_n > 1 and rng.random() < 0.4)
    elif kind == "split":
        c.update(fmt=rng.choice(["tq3", "q8"]), ctx=_log(rng, 2048, 65536), sub_n=rng.choice([1, 1, 16, rng.randint(2, 15)]),
                 k_splits=rng.choice([8, 16, 32]))
    elif kind == "sparse":
        c.update(ctx=_log(rng, 16384, 131072), sub_n=rng.randint(4, 16), top_k=rng.choice([32, 48, 64]), k_splits=8)
    elif kind == "q8":
        c.update(ctx=_log(rng, 300, 32768), sub_n=rng.choice([1, 16, rng.randint(2, 15)]))
    elif kind == "mixed":
        c.update(ctx=_log(rng, 1024, 65536), sub_n=rng.choice([1, 1, rng.randint(2, 16)]))
    elif kind == "paged":
        lo = _log(rng, 256, 8192)
        c.update(n_slots=rng.randint(2, 16), ctx_lo=lo, ctx_hi=min(65536, lo * rng.randint(2, 32)),
                 block_tokens=rng.choice([64, 256]), ctx_seed=rng.randint(0, 10 ** 6), shared=rng.random() < 0.5)
    elif kind == "prefill":
        c.update(start=rng.choice([0, _log(rng, 500, 131072)]), n_tok=_log(rng, 64, 2048))
    else:
        fmt = rng.choice(["tq3", "tq3", "q8"])
        c = dict(kind=kind, fmt=fmt, op=rng.choice(["append", "dequant"]), num_kv=4, n_tok=_log(rng, 16, 32768))
    return c


# ---------------------------------------------------------------------------
# the two block formats in plain torch
# ---------------------------------------------------------------------------
# 52-byte TQ3 block of 128 values: fp32 norm, then 3-bit codes of the rotated
# unit vector; 36-byte Q8_0 block of 32 values: int8 codes, a 16-bit pad, fp16 scale.

_CENTROIDS = [-0.190303, -0.118828, -0.066847, -0.021664, 0.021664, 0.066847, 0.118828, 0.190303]
_BOUNDS = [-0.154566, -0.092838, -0.044256, 0.0, 0.044256, 0.092838, 0.154566]


def _signs():
    s, out = 0xCAFEF00D, []
    for _ in range(128):
        s ^= (s << 13) & (2 ** 64 - 1)
        s ^= s >> 7
        s ^= (s << 17) & (2 ** 64 - 1)
        out.append(1.0 if s & 1 else -1.0)
    return torch.tensor(out, device=DEV)


def _wht(x):
    """Unnormalised 128-point Walsh-Hadamard transform of the last axis."""
    shape = x.shape
    h = 1
    while h < 128:
        y = x.reshape(-1, 128 // (2 * h), 2, h)
        x = torch.cat([y[:, :, :1] + y[:, :, 1:], y[:, :, :1] - y[:, :, 1:]], dim=2)
        h *= 2
    return x.reshape(shape)


def _tq3_encode(rows):
    """fp16 rows [n, heads, 256] -> uint8 blocks [n * heads * 2, 52]."""
    sg, bounds = _signs(), torch.tensor(_BOUNDS, device=DEV)
    parts = []
    for x in rows.reshape(-1, 128).split(1 << 17):
        x = x.float()
        norm = x.square().sum(1, keepdim=True).sqrt()
        y = _wht(x * (1.0 / norm.clamp_min(1e-30)) * sg) * (1.0 / math.sqrt(128.0))
        code = torch.bucketize(y, bounds).to(torch.int32).reshape(-1, 16, 8)
        w = torch.zeros(code.shape[:2], dtype=torch.int32, device=DEV)
        for i in range(8):
            w |= code[:, :, i] << (3 * i)
        qs = torch.stack([w & 255, (w >> 8) & 255, (w >> 16) & 255], dim=2).to(torch.uint8).reshape(-1, 48)
        parts.append(torch.cat([norm.contiguous().view(torch.uint8), qs], dim=1))
    return torch.cat(parts)


def _tq3_decode64(blocks):
    """uint8 blocks [n, 52] -> float64 values [n, 128]."""
    sg, cen = _signs().double(), torch.tensor(_CENTROIDS, dtype=torch.float32, device=DEV).double()
    b = blocks.reshape(-1, 52)
    norm = b[:, :4].contiguous().view(torch.float32).double()
    q = b[:, 4:].reshape(-1, 16, 3).to(torch.int32)
    w = q[:, :, 0] | (q[:, :, 1] << 8) | (q[:, :, 2] << 16)
    code = torch.stack([(w >> (3 * i)) & 7 for i in range(8)], dim=2).reshape(-1, 128)
    return _wht(cen[code]) * (1.0 / math.sqrt(128.0)) * sg * norm


def _q8_encode(rows):
    """fp16 rows [n, heads, 256] -> uint8 blocks [n * heads * 8, 36]."""
    x = rows.reshape(-1, 32).float()
    scale = x.abs().amax(1, keepdim=True) / 127.0
    inv = torch.where(scale > 0, 1.0 / scale, torch.zeros_like(scale))
    q = (x * inv).round().clamp(-128, 127).to(torch.int8).view(torch.uint8)
    pad = torch.zeros((x.shape[0], 2), dtype=torch.uint8, device=DEV)
    return torch.cat([q, pad, scale.half().view(torch.uint8)], dim=1)


def _q8_decode64(blocks):
    b = blocks.reshape(-1, 36)
    return b[:, :32].contiguous().view(torch.int8).double() * b[:, 34:].contiguous().view(torch.float16).double()


_FMT = {"tq3": (_tq3_encode, _tq3_decode64, 52, 128), "q8": (_q8_encode, _q8_decode64, 36, 32)}


def _head_rows64(cache, fmt, num_kv, h, n):
    """Head h of cache rows 0..n-1 as float64 [n, 256]."""
    _, dec, size, per = _FMT[fmt]
    rows = cache.reshape(-1)[: n * num_kv * (HD // per) * size].reshape(n, num_kv, HD // per, size)[:, h]
    return torch.cat([dec(r.contiguous()).reshape(-1, HD) for r in rows.split(1 << 15)])


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------

class _Rng:
    def __init__(self, seed):
        self.g = torch.Generator(device=DEV).manual_seed(int(seed))

    def normal(self, *shape):
        return torch.randn(*shape, generator=self.g, device=DEV)

    def kv(self, n_tok, num_kv, channels=None):
        """fp16 [n_tok, num_kv, 256]; `channels`: the outlier channels' scale of this tensor."""
        return (self.normal(n_tok, num_kv, HD) * channels).half()

    def channels(self, num_kv):
        at = torch.rand(num_kv, HD, generator=self.g, device=DEV).argsort(dim=1)
        return torch.where(at < round(0.02 * HD), 8.0, 1.0)


def _cache(rng, fmt, num_kv, n_rows, extra, ch):
    """A cache of n_rows encoded rows, and room for `extra` more."""
    enc, _, size, per = _FMT[fmt]
    bpr = num_kv * HD // per
    c = torch.zeros(((n_rows + extra) * bpr, size), dtype=torch.uint8, device=DEV)
    for r0 in range(0, n_rows, 1 << 15):
        n = min(1 << 15, n_rows - r0)
        c[r0 * bpr: (r0 + n) * bpr] = enc(rng.kv(n, num_kv, ch))
    return c


def _formats(case):
    kind = case["kind"]
    if kind == "q8" or (kind == "split" and case["fmt"] == "q8"):
        return "q8", "q8"
    return ("q8", "tq3") if kind == "mixed" else ("tq3", "tq3")


def _tree_masks(sub_n, seed):
    """A random draft tree: node t sees its ancestors and itself (bit j: block key j)."""
    r, masks = np.random.default_rng(seed), []
    for t in range(sub_n):
        up = masks[int(r.integers(max(0, t - 4), t))] if t else 0
        masks.append(up | (1 << t))
    return masks


def _slots(case):
    r = np.random.default_rng(case["ctx_seed"])
    ctx = r.integers(case["ctx_lo"], case["ctx_hi"] + 1, size=case["n_slots"])
    prefix = min(4096, case["ctx_lo"]) // case["block_tokens"] * case["block_tokens"] if case["shared"] else 0
    return ctx.astype(np.int64), prefix


def _tables(case):
    """Block tables of the slots (int32 [n_slots][max_blocks], blocks handed out in
    a shuffled order, the first slots' prefix blocks shared) and the pool's rows."""
    ctx, prefix = _slots(case)
    bt = case["block_tokens"]
    mb = int(-(-(int(ctx.max()) + 1) // bt))
    need = [int(-(-(int(c) + 1) // bt)) for c in ctx]
    order = list(np.random.default_rng(case["ctx_seed"] + 1).permutation(sum(need)))
    table = np.zeros((case["n_slots"], mb), dtype=np.int32)
    for s, n in enumerate(need):
        for b in range(n):
            table[s, b] = table[0, b] if 0 < s < 4 and b < prefix // bt else order.pop()
    return table, sum(need) * bt


# ---------------------------------------------------------------------------
# prepare / run
# ---------------------------------------------------------------------------

def prepare(case, seed):
    return globals()["_prepare_" + case["kind"]](case, _Rng(seed), seed)


def run(state):
    return state["run"](state)


def _attention_state(case, rng, rows, extra):
    c, (fk, fv) = case, _formats(case)
    ck, cv = rng.channels(c["num_kv"]), rng.channels(c["num_kv"])
    return dict(case=c, scale=1.0 / math.sqrt(HD), ck=ck, cv=cv,
                k=_cache(rng, fk, c["num_kv"], rows, extra, ck), v=_cache(rng, fv, c["num_kv"], rows, extra, cv))


def _block(s, rng):
    """A step's queries and, beside them, its new K and V rows."""
    c = s["case"]
    n = c["sub_n"]
    s["q"] = rng.normal(n, c["num_q"], HD).half()
    s["kn"], s["vn"] = rng.kv(n, c["num_kv"], s["ck"]), rng.kv(n, c["num_kv"], s["cv"])
    s["out"] = torch.empty_like(s["q"])
    return s


def _prepare_decode(case, rng, seed):
    c, n = case, case["sub_n"]
    layers = []
    for _ in range(c["layers"]):
        # without the append the block's rows are in the cache already
        rows = c["ctx"] if c["append"] else c["ctx"] + n
        layers.append(_block(_attention_state(c, rng, rows, n if c["append"] else 0), rng))
    tree = None
    if c["tree"]:
        tree = torch.tensor(_tree_masks(n, seed), dtype=torch.int64, device=DEV).to(torch.int32)
    ws = kvcache.decode_attn_tq3_workspace(c["num_q"], c["num_kv"], n, c["ctx"] + n, DEV)
    return dict(case=c, run=_run_decode, layers=layers, tree=tree, ws=ws)


def _run_decode(s):
    c = s["case"]
    kw = dict(num_q=c["num_q"], num_kv=c["num_kv"], start_pos=c["ctx"], sub_n=c["sub_n"], tree_mask=s["tree"])
    for a in s["layers"]:
        if c["append"]:
            kvcache.decode_attn_tq3_append(a["q"], a["kn"], a["vn"], a["k"], a["v"], a["out"], s["ws"],
                                           scale=a["scale"], **kw)
        else:
            kvcache.decode_attn_tq3(a["q"], a["k"], a["v"], a["out"], s["ws"], scale=a["scale"], **kw)
    out = [a["out"] for a in s["layers"]]
    return dict(out=out, k=[a["k"] for a in s["layers"]], v=[a["v"] for a in s["layers"]]) if c["append"] else dict(out=out)


def _prepare_split(case, rng, seed):
    c, n = case, case["sub_n"]
    s = _block(_attention_state(c, rng, c["ctx"] + n, 0), rng)
    shape = (c["num_q"], n, c["k_splits"])
    s.update(run=_run_split, pm=torch.zeros(shape, device=DEV), pl=torch.zeros(shape, device=DEV),
             po=torch.zeros(shape + (HD,), device=DEV))
    return s


def _run_split(s):
    c = s["case"]
    kw = dict(num_q=c["num_q"], num_kv=c["num_kv"], sub_n=c["sub_n"], sub_n_max=c["sub_n"], k_splits=c["k_splits"])
    split = kvcache.attn_split_tq3 if c["fmt"] == "tq3" else kvcache.attn_split_q8
    split(s["q"], s["k"], s["v"], s["pm"], s["pl"], s["po"], start_pos=c["ctx"],
          active_end_max=c["ctx"] + c["sub_n"], scale=s["scale"], **kw)
    kvcache.attn_split_merge(s["pm"], s["pl"], s["po"], s["out"], **kw)
    return dict(out=s["out"], part_m=s["pm"], part_l=s["pl"], part_o=s["po"])


def _prepare_q8(case, rng, seed):
    c = case
    s = _block(_attention_state(c, rng, c["ctx"], c["sub_n"]), rng)
    s.update(run=_run_q8, ws=kvcache.decode_attn_q8_workspace(c["num_q"], c["num_kv"], c["sub_n"], c["ctx"] + c["sub_n"], DEV))
    return s


def _run_q8(s):
    c = s["case"]
    kw = dict(num_q=c["num_q"], num_kv=c["num_kv"], start_pos=c["ctx"], scale=s["scale"])
    if c["sub_n"] == 1:
        kvcache.decode_attn_q8_append(s["q"], s["kn"], s["vn"], s["k"], s["v"], s["out"], s["ws"], **kw)
    else:
        at = c["ctx"] * c["num_kv"] * 8
        kvcache.q8_append_kv(s["kn"], s["vn"], s["k"][at:], s["v"][at:])
        kvcache.decode_attn_q8(s["q"], s["k"], s["v"], s["out"], s["ws"], sub_n=c["sub_n"], **kw)
    return dict(out=s["out"], k=s["k"], v=s["v"])


def _prepare_mixed(case, rng, seed):
    c = case
    s = _block(_attention_state(c, rng, c["ctx"], c["sub_n"]), rng)
    s.update(run=_run_mixed, ws=kvcache.decode_attn_q8k_tq3v_workspace(c["num_q"], c["num_kv"], c["sub_n"],
                                                                      c["ctx"] + c["sub_n"], DEV))
    return s


def _run_mixed(s):
    c = s["case"]
    kvcache.q8_append(s["kn"], s["k"][c["ctx"] * c["num_kv"] * 8:])
    kvcache.tq3_append(s["vn"], s["v"][c["ctx"] * c["num_kv"] * 2:])
    kvcache.decode_attn_q8k_tq3v(s["q"], s["k"], s["v"], s["out"], s["ws"], num_q=c["num_q"], num_kv=c["num_kv"],
                                 start_pos=c["ctx"], sub_n=c["sub_n"], scale=s["scale"])
    return dict(out=s["out"], k=s["k"], v=s["v"])


def _prepare_sparse(case, rng, seed):
    c, n = case, case["sub_n"]
    s = _block(_attention_state(c, rng, c["ctx"], n), rng)
    nb = (c["ctx"] + n + 63) // 64
    shape = (c["num_q"], n, c["k_splits"])
    s.update(run=_run_sparse, nb=nb, pool=torch.zeros((c["num_kv"], nb, HD), dtype=torch.float16, device=DEV),
             pool_max=torch.zeros((c["num_kv"], nb, HD), dtype=torch.float16, device=DEV),
             index=torch.full((c["num_kv"], n, c["top_k"]), -1, dtype=torch.int32, device=DEV),
             ws=torch.empty(c["num_kv"] * n * nb * 4 + 256, dtype=torch.uint8, device=DEV),
             pm=torch.zeros(shape, device=DEV), pl=torch.zeros(shape, device=DEV), po=torch.zeros(shape + (HD,), device=DEV))
    # the history's block signatures, which such a program has kept up with its cache
    kvcache.tq3_kpool_update(s["k"], s["pool"], s["pool_max"], num_kv=c["num_kv"], total_kv=c["ctx"], blk_lo=0)
    return s


def _run_sparse(s):
    c = s["case"]
    at = c["ctx"] * c["num_kv"] * 2
    kw = dict(num_q=c["num_q"], num_kv=c["num_kv"], sub_n=c["sub_n"])
    kvcache.tq3_append_kv(s["kn"], s["vn"], s["k"][at:], s["v"][at:])
    kvcache.tq3_kpool_update(s["k"], s["pool"], s["pool_max"], num_kv=c["num_kv"], total_kv=c["ctx"] + c["sub_n"],
                             blk_lo=c["ctx"] // 64)
    kvcache.block_index_ms(s["q"], s["pool"], s["pool_max"], s["index"], start_pos=c["ctx"], top_k=c["top_k"],
                           n_blocks=s["nb"], workspace=s["ws"], **kw)
    kvcache.attn_block_sparse_split_tq3(s["q"], s["k"], s["v"], s["index"], s["pm"], s["pl"], s["po"],
                                        start_pos=c["ctx"], sub_n_max=c["sub_n"], scale=s["scale"], top_k=c["top_k"],
                                        k_splits=c["k_splits"], **kw)
    kvcache.attn_split_merge(s["pm"], s["pl"], s["po"], s["out"], sub_n_max=c["sub_n"], k_splits=c["k_splits"], **kw)
    return dict(out=s["out"], index=s["index"], pool=s["pool"], pool_max=s["pool_max"], k=s["k"], v=s["v"])


def _prepare_paged(case, rng, seed):
    c = case
    ctx, _ = _slots(c)
    table, rows = _tables(c)
    s = _attention_state(c, rng, rows, 0)
    n = c["n_slots"]
    max_ctx = int(ctx.max()) + 1
    s.update(run=_run_paged, max_ctx=max_ctx, q=rng.normal(n, c["num_q"], HD).half(),
             kn=rng.kv(n, c["num_kv"], s["ck"])[:, None].contiguous(),
             vn=rng.kv(n, c["num_kv"], s["cv"])[:, None].contiguous(),
             table=torch.from_numpy(table).to(DEV), pos=torch.from_numpy(ctx.astype(np.int32)).to(DEV),
             lens=torch.from_numpy((ctx + 1).astype(np.int32)).to(DEV),
             ws=kvcache.decode_attn_tq3_paged_workspace(c["num_q"], c["num_kv"], n, max_ctx, DEV))
    s["out"] = torch.empty_like(s["q"])
    return s


def _run_paged(s):
    c = s["case"]
    kvcache.tq3_append_kv_paged(s["kn"], s["vn"], s["k"], s["v"], s["table"], s["pos"], block_tokens=c["block_tokens"])
    kvcache.decode_attn_tq3_paged(s["q"], s["k"], s["v"], s["out"], s["ws"], s["table"], s["lens"], num_q=c["num_q"],
                                  num_kv=c["num_kv"], max_ctx=s["max_ctx"], block_tokens=c["block_tokens"],
                                  scale=s["scale"])
    return dict(out=s["out"], k=s["k"], v=s["v"])


def _prepare_prefill(case, rng, seed):
    c, n = case, case["n_tok"]
    s = _block(_attention_state(dict(c, sub_n=n), rng, c["start"], n), rng)
    s.update(run=_run_prefill, ws=kvcache.prefill_attn_tq3_workspace(c["num_q"], c["num_kv"], n, c["start"], DEV))
    return s


def _run_prefill(s):
    c = s["case"]
    at = c["start"] * c["num_kv"] * 2
    kvcache.tq3_append_kv(s["kn"], s["vn"], s["k"][at:], s["v"][at:])
    kvcache.prefill_attn_tq3(s["q"], s["k"], s["v"], s["kn"], s["vn"], s["out"], s["ws"], num_q=c["num_q"],
                             num_kv=c["num_kv"], start_pos=c["start"], scale=s["scale"])
    return dict(out=s["out"], k=s["k"], v=s["v"])


def _prepare_codec(case, rng, seed):
    c = case
    enc, _, size, per = _FMT[c["fmt"]]
    n = c["n_tok"] * c["num_kv"] * HD // per
    x = [rng.kv(c["n_tok"], c["num_kv"], rng.channels(c["num_kv"])) for _ in range(2)]
    if c["op"] == "append":
        return dict(case=c, run=_run_codec, x=x, y=[torch.zeros((n, size), dtype=torch.uint8, device=DEV) for _ in x])
    return dict(case=c, run=_run_codec, x=[torch.cat([enc(r) for r in t.split(1 << 15)]) for t in x],
                y=[torch.empty(n * per, dtype=torch.float16, device=DEV) for _ in x])


def _run_codec(s):
    c, (xk, xv), (yk, yv) = s["case"], s["x"], s["y"]
    if c["op"] == "append":
        (kvcache.tq3_append_kv if c["fmt"] == "tq3" else kvcache.q8_append_kv)(xk, xv, yk, yv)
    else:
        dequant = kvcache.tq3_dequant if c["fmt"] == "tq3" else kvcache.q8_dequant
        dequant(xk, yk)
        dequant(xv, yv)
    return dict(k=yk, v=yv)


# ---------------------------------------------------------------------------
# what a pass cannot do without
# ---------------------------------------------------------------------------

def work(case):
    c, kind = case, case["kind"]
    row = {f: c["num_kv"] * (HD // per) * size for f, (_, _, size, per) in _FMT.items()}
    if kind == "codec":
        fp16 = c["num_kv"] * HD * 2
        return {"bytes": 2 * c["n_tok"] * (fp16 + row[c["fmt"]]), "flops": 0}
    fk, fv = _formats(c)
    kv = row[fk] + row[fv]               # bytes of one cached token
    new = 2 * c["num_kv"] * HD * 2       # fp16 K and V of one token
    qo = 2 * c["num_q"] * HD * 2         # one query token in, one out
    pair = 4 * c["num_q"] * HD           # flops per (query token, key)
    if kind == "paged":
        ctx, prefix = _slots(c)
        shared = prefix * (min(4, c["n_slots"]) - 1)   # a shared prefix is in the pool once
        keys = int(ctx.sum()) + c["n_slots"]
        return {"bytes": (keys - shared) * kv + c["n_slots"] * (qo + new), "flops": keys * pair}
    if kind == "prefill":
        n, h = c["n_tok"], c["start"]
        return {"bytes": (h + n) * kv + n * (qo + new), "flops": (n * h + n * (n + 1) // 2) * pair}
    n = c["sub_n"]
    if kind == "sparse":
        nb = (c["ctx"] + n + 63) // 64
        blocks = min(c["top_k"] * n, nb)   # the queries' picks overlap or not
        upd = nb - c["ctx"] // 64
        return {"bytes": nb * c["num_kv"] * HD * 4 + blocks * 64 * kv + upd * c["num_kv"] * (64 * row[fk] // c["num_kv"] + HD * 4)
                + n * (kv + qo + new) + n * c["num_kv"] * c["top_k"] * 4,
                "flops": n * (c["top_k"] * 64 * pair + nb * c["num_kv"] * HD * 4)}
    layers = c.get("layers", 1)
    append = kind in ("q8", "mixed") or c.get("append", False)
    b = (c["ctx"] + n) * kv + n * qo + (n * new if append else 0)
    if kind == "split":
        b += c["num_q"] * n * c["k_splits"] * (HD + 2) * 4
    return {"bytes": layers * b, "flops": layers * (n * c["ctx"] + n * (n + 1) // 2) * pair}


def tolerance(case):
    if case["kind"] == "codec":
        return "exact"   # the codecs are bit-exact
    # fp16 outputs (2^-12 rms) of sums whose probabilities are fp16; the caches,
    # indices and signatures beside them are bytes and whole numbers
    return {"rel": 2e-3, "max": 2e-2}


# ---------------------------------------------------------------------------
# the same in 64 bits
# ---------------------------------------------------------------------------

def _softmax_pv(q, k, v, scale, visible):
    """Attention of float64 rows q [m, 256] over k, v [n, 256]; visible [m, n] or None."""
    s = torch.mm(q, k.t().contiguous()) * scale
    if visible is not None:
        s.masked_fill_(~visible, -math.inf)
    m = s.amax(1, keepdim=True)
    p = torch.exp(s - torch.where(torch.isinf(m), torch.zeros_like(m), m))
    l = p.sum(1, keepdim=True)
    return m[:, 0], l[:, 0], torch.mm(p, v)


def _put_new(cache, fmt, at_row, new, num_kv):
    """The cache with its new rows encoded behind row at_row."""
    enc, _, _, per = _FMT[fmt]
    b = enc(new)
    at = at_row * num_kv * HD // per
    c = cache.clone()
    c[at: at + b.shape[0]] = b
    return c


def _dense64(s, fk, fv, ctx, n, tree=None):
    """Causal (or tree-masked) attention of n queries behind ctx keys: [n, num_q, 256]."""
    c = s["case"]
    gqa = c["num_q"] // c["num_kv"]
    out = torch.empty((n, c["num_q"], HD), dtype=torch.float64, device=DEV)
    key = torch.arange(ctx + n, device=DEV)
    for h in range(c["num_kv"]):
        k, v = (_head_rows64(s[x], f, c["num_kv"], h, ctx + n) for x, f in (("k", fk), ("v", fv)))
        for t in range(n):
            vis = key <= ctx + t
            if tree is not None:
                bits = (tree[t] >> (key - ctx).clamp(0, 31)) & 1
                vis = vis & ((key < ctx) | (bits != 0))
            q = s["q"][t, h * gqa: (h + 1) * gqa].double()
            _, l, o = _softmax_pv(q, k, v, s["scale"], vis[None].expand(gqa, -1))
            out[t, h * gqa: (h + 1) * gqa] = o / l[:, None]
    return out


def exact(case, seed):
    s = prepare(case, seed)
    return globals()["_exact_" + case["kind"]](case, s, seed)


def _appended(s, fk, fv, ctx):
    n = s["case"]["num_kv"]
    return dict(s, k=_put_new(s["k"], fk, ctx, s["kn"], n), v=_put_new(s["v"], fv, ctx, s["vn"], n))


def _exact_decode(case, s, seed):
    c = case
    out = []
    for a in s["layers"]:
        if c["append"]:
            a = _appended(a, "tq3", "tq3", c["ctx"])
        out.append(_dense64(a, "tq3", "tq3", c["ctx"], c["sub_n"], _tree_masks(c["sub_n"], seed) if c["tree"] else None))
    none = [None] * c["layers"]
    return dict(out=out, k=none, v=none) if c["append"] else dict(out=out)


def _exact_q8(case, s, seed):
    fk, fv = _formats(case)
    return dict(out=_dense64(_appended(s, fk, fv, case["ctx"]), fk, fv, case["ctx"], case["sub_n"]), k=None, v=None)


_exact_mixed = _exact_q8


def _exact_split(case, s, seed):
    c, (fk, fv) = case, _formats(case)
    gqa, n, end = c["num_q"] // c["num_kv"], c["sub_n"], c["ctx"] + c["sub_n"]
    shape = (c["num_q"], n, c["k_splits"])
    pm, pl = (torch.zeros(shape, dtype=torch.float64, device=DEV) for _ in range(2))
    po = torch.zeros(shape + (HD,), dtype=torch.float64, device=DEV)
    span = -(-(-(-end // 32)) // c["k_splits"]) * 32   # keys of one split
    for h in range(c["num_kv"]):
        k, v = _head_rows64(s["k"], fk, c["num_kv"], h, end), _head_rows64(s["v"], fv, c["num_kv"], h, end)
        for t in range(n):
            q = s["q"][t, h * gqa: (h + 1) * gqa].double()
            for z in range(c["k_splits"]):
                lo, hi = z * span, min((z + 1) * span, c["ctx"] + t + 1)
                at = (slice(h * gqa, (h + 1) * gqa), t, z)
                if lo < hi:
                    pm[at], pl[at], po[at] = _softmax_pv(q, k[lo:hi], v[lo:hi], s["scale"], None)
                else:
                    pm[at] = -math.inf
    w = torch.exp(pm - pm.amax(2, keepdim=True)).nan_to_num(0.0)
    out = (w[..., None] * po).sum(2) / (w * pl).sum(2)[..., None]
    return dict(out=out.transpose(0, 1).contiguous(), part_m=pm, part_l=pl, part_o=po)


def _exact_paged(case, s, seed):
    c = case
    ctx, _ = _slots(c)
    table, _ = _tables(c)
    gqa, bt = c["num_q"] // c["num_kv"], c["block_tokens"]
    out = torch.empty((c["n_slots"], c["num_q"], HD), dtype=torch.float64, device=DEV)
    rows = {x: s[x].reshape(-1, c["num_kv"] * 2, 52).clone() for x in "kv"}
    where = []
    for t in range(c["n_slots"]):
        key = np.arange(int(ctx[t]) + 1)
        where.append(torch.from_numpy(table[t, key // bt].astype(np.int64) * bt + key % bt).to(DEV))
        for x, new in (("k", s["kn"]), ("v", s["vn"])):
            rows[x][where[t][-1]] = _tq3_encode(new[t]).reshape(-1, 52)
    for t in range(c["n_slots"]):
        n = len(where[t])
        k, v = (rows[x][where[t]].reshape(-1, 52) for x in "kv")
        for h in range(c["num_kv"]):
            kh, vh = (_head_rows64(x, "tq3", c["num_kv"], h, n) for x in (k, v))
            q = s["q"][t, h * gqa: (h + 1) * gqa].double()
            _, l, o = _softmax_pv(q, kh, vh, s["scale"], None)
            out[t, h * gqa: (h + 1) * gqa] = o / l[:, None]
    return dict(out=out, k=None, v=None)


def _exact_prefill(case, s, seed):
    c, n, h0 = case, case["n_tok"], case["start"]
    gqa = c["num_q"] // c["num_kv"]
    out = torch.empty((n, c["num_q"], HD), dtype=torch.float64, device=DEV)
    key = torch.arange(h0 + n, device=DEV)
    for h in range(c["num_kv"]):
        # the chunk's own rows are attended as given, the history from the cache
        k, v = (torch.cat([_head_rows64(s[x], "tq3", c["num_kv"], h, h0) if h0 else s[y][:0, h].double(), s[y][:, h].double()])
                for x, y in (("k", "kn"), ("v", "vn")))
        for t0 in range(0, n, 256):
            t = torch.arange(t0, min(n, t0 + 256), device=DEV)
            vis = (key[None] <= h0 + t[:, None]).repeat_interleave(gqa, 0)
            q = s["q"][t0: t0 + 256, h * gqa: (h + 1) * gqa].reshape(-1, HD).double()
            _, l, o = _softmax_pv(q, k, v, s["scale"], vis)
            out[t0: t0 + 256, h * gqa: (h + 1) * gqa] = (o / l[:, None]).reshape(-1, gqa, HD)
    return dict(out=out, k=None, v=None)


def _exact_sparse(case, s, seed):
    """The selection is made on fp16 signatures and an fp16 mean query, which belong to the method."""
    c = case
    n, ctx, nb = c["sub_n"], c["ctx"], s["nb"]
    a = _appended(s, "tq3", "tq3", ctx)
    gqa, end = c["num_q"] // c["num_kv"], ctx + n
    out = torch.empty((n, c["num_q"], HD), dtype=torch.float64, device=DEV)
    pool, pool_max = (torch.empty((c["num_kv"], nb, HD), dtype=torch.float64, device=DEV) for _ in range(2))
    key = torch.arange(nb * 64, device=DEV)
    for h in range(c["num_kv"]):
        k, v = (torch.cat([_head_rows64(a[x], "tq3", c["num_kv"], h, end),
                           torch.zeros((nb * 64 - end, HD), dtype=torch.float64, device=DEV)]) for x in "kv")
        kb = k.half().double().reshape(nb, 64, HD)
        count = (end - 64 * torch.arange(nb, device=DEV)).clamp(max=64)[:, None]
        pool[h] = kb.sum(1) / count
        pool_max[h] = kb.gather(1, kb.abs().argmax(1, keepdim=True))[:, 0]
        mean16, max16 = pool[h].half().double(), pool_max[h].half().double()
        for t in range(n):
            q = s["q"][t, h * gqa: (h + 1) * gqa].double()
            qm = q.mean(0).float().half().double()
            sc = torch.maximum((mean16 * qm).sum(1), 0.5 * (max16 * qm).sum(1))
            sc[(ctx + t) // 64 + 1:] = -math.inf
            pick = sc.topk(min(c["top_k"], (ctx + t) // 64 + 1)).indices
            vis = torch.zeros(nb, dtype=torch.bool, device=DEV)
            vis[pick] = True
            vis = vis.repeat_interleave(64) & (key <= ctx + t)
            _, l, o = _softmax_pv(q, k, v, s["scale"], vis[None].expand(gqa, -1))
            out[t, h * gqa: (h + 1) * gqa] = o / l[:, None]
    return dict(out=out, index=None, pool=pool, pool_max=pool_max, k=None, v=None)


def _exact_codec(case, s, seed):
    if case["op"] == "append":
        return None
    return {x: torch.cat([_FMT[case["fmt"]][1](b).reshape(-1) for b in y.split(1 << 18)]) for x, y in zip("kv", s["x"])}

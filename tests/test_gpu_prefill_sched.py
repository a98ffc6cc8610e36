"""The prefill attention over the shapes that change its schedule: one or two
token groups per workgroup, rows of one key segment (stored by the attention)
beside rows of several (merged), ragged last tiles, both staging kernels.
Reference: float64 attention over the fp16 keys and values that the reference
attends (the bulk dequantization of the history, then the chunk as given)."""
import numpy as np
import pytest

from oracle import oracle as O
from tests._data import kv_f16, q_f16, rel_err

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("start,n_tok,num_q,num_kv,from_cache", [
    (0, 33, 16, 4, False), (0, 300, 16, 4, False), (0, 777, 24, 4, False), (0, 777, 16, 4, False),
    (0, 2048, 16, 4, False), (65, 1000, 12, 2, False), (1000, 512, 16, 4, False), (3001, 200, 24, 4, False),
    (10000, 129, 16, 4, False), (9000, 64, 8, 2, False), (5000, 48, 16, 4, True), (6000, 20, 24, 4, True),
])
def test_prefill_schedules(dev, start, n_tok, num_q, num_kv, from_cache):
    import torch
    from qengine_amd import kvcache
    print(f"prefill start={start} n_tok={n_tok} num_q={num_q} num_kv={num_kv} cache={from_cache}", flush=True)
    rng = np.random.default_rng(start + n_tok + num_q)
    t = lambda a: torch.from_numpy(np.ascontiguousarray(a)).to(dev)   # noqa: E731
    cached = start + n_tok if from_cache else start
    kb, vb = (O.tq3_encode(kv_f16(rng, max(cached, 1), num_kv, 256)) for _ in range(2))
    rows = [O.tq3_decode(b).view(np.float16).reshape(-1, num_kv, 256)[:cached] for b in (kb, vb)]
    chunk = None
    if not from_cache:
        chunk = [kv_f16(rng, n_tok, num_kv, 256) for _ in range(2)]
        rows = [np.concatenate([r, c]) for r, c in zip(rows, chunk)]
    q = q_f16(rng, n_tok, num_q, 256)
    out = torch.full((n_tok, num_q, 256), float("nan"), dtype=torch.float16, device=dev)
    ws = kvcache.prefill_attn_tq3_workspace(num_q, num_kv, n_tok, start, dev)
    ck, cv = (None, None) if chunk is None else (t(chunk[0]), t(chunk[1]))
    kvcache.prefill_attn_tq3(t(q), t(kb.view(np.uint8)), t(vb.view(np.uint8)), ck, cv, out, ws, num_q=num_q,
                             num_kv=num_kv, start_pos=start, scale=1 / 16)
    torch.cuda.synchronize()
    k, v, qd = (t(x).double() for x in (*rows, q))
    gqa = num_q // num_kv
    visible = torch.arange(start + n_tok, device=dev)[None] <= start + torch.arange(n_tok, device=dev)[:, None]
    ref = torch.empty((n_tok, num_q, 256), dtype=torch.float64, device=dev)
    for h in range(num_q):
        s = torch.mm(qd[:, h].contiguous(), k[:, h // gqa].t().contiguous()) / 16
        p = torch.softmax(s.masked_fill(~visible, -float("inf")), dim=1)
        ref[:, h] = torch.mm(p, v[:, h // gqa].contiguous())
    # fp16 weights and outputs: 2^-11 each per element, the bar of the other prefill tests
    assert rel_err(out.float().cpu().numpy(), ref.cpu().numpy()) < 2e-3

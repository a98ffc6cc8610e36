"""Split-API calls of many queries, which the multi-query kernel serves: the partials
of every reference split against the oracle's.  Sizes: splits shorter than a tile,
splits whose last tile belongs half to the next one, empty splits, both workgroup
widths (GQA 6 with many splits: 64 columns), queries that do not fill the last
workgroup, sub_n_max above sub_n, masks; the tolerances of the other split tests."""
import numpy as np
import pytest

from oracle import oracle as O
from tests import test_gpu_attn_q8 as q8
from tests import test_gpu_attn_tq3 as tq3
from tests._data import assert_tq3_attn, q_f16

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("fmt,num_q,num_kv,n,sub_n,sub_n_max,k_splits,sink,window,tree", [
    ("tq3", 16, 4, 1000, 16, 16, 32, 0, 0, False), ("tq3", 24, 4, 777, 16, 20, 32, 32, 100, False),
    ("tq3", 16, 4, 300, 13, 16, 64, 0, 0, True), ("tq3", 8, 1, 900, 16, 16, 64, 0, 0, False),
    ("tq3", 32, 4, 2100, 9, 9, 16, 0, 64, True),
    ("q8", 16, 4, 2000, 16, 17, 8, 0, 0, False), ("q8", 24, 4, 1600, 11, 11, 64, 0, 0, False),
    ("q8", 16, 4, 500, 7, 8, 64, 0, 0, False), ("q8", 24, 4, 2500, 16, 16, 32, 0, 0, False),
    ("q8", 8, 1, 1700, 16, 16, 64, 0, 0, False),
])
def test_split_many_queries(dev, fmt, num_q, num_kv, n, sub_n, sub_n_max, k_splits, sink, window, tree):
    print(f"{fmt} num_q={num_q} num_kv={num_kv} n={n} sub_n={sub_n} splits={k_splits}", flush=True)
    m = tq3 if fmt == "tq3" else q8
    rng, kb, vb = m._cache(n + sub_n, n, num_kv=num_kv)
    q = q_f16(rng, sub_n, num_q, 256)
    kw = dict(num_q=num_q, num_kv=num_kv, start_pos=n - sub_n, sub_n=sub_n, sub_n_max=sub_n_max,
              active_end_max=n, scale=1 / 16, k_splits=k_splits)
    if fmt == "tq3":
        tm = None
        if tree:
            tm = np.array([(1 << t) | (int(rng.integers(0, 1 << max(t, 1))) & ((1 << t) - 1))
                           for t in range(sub_n)], np.uint32)
        kw.update(sink_tok=sink, window_tok=window, tree_mask=tm)
        pm, pl, po, out = tq3._run_split(dev, q, kb, vb, **kw)
        em, el, eo = O.attn_split(O.KV_TQ3, q, kb, vb, hd=256, **kw)
    else:
        pm, pl, po, out = q8._run(dev, q, kb, vb, **kw)
        em, el, eo = O.attn_split(O.KV_Q8, q, kb, vb, hd=256, **kw)
    tq3._check_partials(pm, pl, po, em, el, eo, sub_n)
    exp = O.attn_split_merge(em, el, eo, num_q=num_q, num_kv=num_kv, hd=256, sub_n=sub_n, sub_n_max=sub_n_max,
                             k_splits=k_splits).view(np.float16)
    if fmt == "tq3":
        assert_tq3_attn(out, exp, tq3._exact(q, kb, vb, **kw))
    else:
        q8.check_rel(out, exp, q8.TOL)

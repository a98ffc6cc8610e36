"""Workspace queries of the multi-query decode, which need no GPU."""
import pytest

from qengine_amd._lib import lib


@pytest.mark.parametrize("num_q,num_kv", [(16, 4), (24, 4), (64, 8), (4, 4), (8, 1), (24, 3), (35, 7)])
@pytest.mark.parametrize("sub_n", [3, 16, 65, 300, 1040])
def test_tq3_workspace_of_many_queries(num_q, num_kv, sub_n):
    """A workspace for n keys serves every shorter call (the size never falls as the
    keys grow), and holds no more records than one round of 256 workgroups of up to 64
    (query, head) columns writes, or one per row where the rows alone are more."""
    if sub_n * (num_q // num_kv) <= 16:
        pytest.skip("not a multi-query call")
    size = lib().qkv_decode_attn_tq3_workspace_bytes
    last = 0
    for n_keys in (sub_n, sub_n + 63, 2048, 4096, 18016, 32768, 32833, 131072, 131088):
        if n_keys < sub_n:
            continue
        need = size(num_q, num_kv, sub_n, n_keys)
        assert need >= last
        last = need
    rows = num_q * sub_n
    # the chunks of a round: 256 workgroups over the kv heads and the query groups, of
    # which whole queries fill at least half of the 64 columns
    records = max(rows, 256 * 64 + rows)
    assert last <= 2 * 1040 * records + 512, (last, records)

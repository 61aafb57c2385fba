"""Decode steps without masks, windows and leftover columns, over TQ4 pages and row formats: the kernel that works ahead of the lengths gives the
bytes of the general one, which a batch without context_lens_before takes, and the oracle's values."""
import numpy as np
import pytest

import oracle
from cases import make_case
from oracle import DT_BF16, DT_F16, FMT_TQ4

pytestmark = pytest.mark.gpu

# page size, kv heads, q heads, keys and new tokens per request, bound on the keys (0: exact)
CASES = [
    (16, 2, 16, [1200], [1], 0),           # the request is as long as the bound: the guessed rows
    (16, 2, 16, [1200], [1], 5000),        # it is not
    (64, 2, 16, [1], [1], 0),              # one key
    (48, 2, 16, [769], [1], 0),            # pages that units straddle, one key in the last unit
    (112, 1, 8, [2065], [1], 2066),        # a run that ends behind the last key
    (128, 2, 4, [257], [3], 0),            # three tokens of two heads
    (16, 4, 4, [5000], [8], 0),            # eight tokens of one head
    (64, 1, 5, [300], [1], 0),             # columns that stay dead
    (16, 2, 16, [700, 31, 2500], [1, 1, 1], 0),
    (32, 2, 16, [700, 9, 2500, 64], [1, 0, 1, 1], 10000),  # a request without tokens
]


@pytest.mark.parametrize("dtype", [DT_F16, DT_BF16])
@pytest.mark.parametrize("case", range(len(CASES)))
def test_bytes_of_the_general_kernel(case, dtype):
    import gpu_harness as G

    block, kv_heads, q_heads, seqs, q_lens, bound = CASES[case]
    pool, bt, k, v, q, aq, ctx = make_case(FMT_TQ4, block, seqs, q_lens, 3100 + case, dtype, kv_heads=kv_heads, q_heads=q_heads)
    hb = oracle.HostBatch(aq, seqs, bt, context_lens_before=ctx)
    general = oracle.HostBatch(aq, seqs, bt)
    dpool = G.DevPool(pool)
    dpool.upload()
    outs = []
    for batch in (hb, general):
        rc, got, _ = G.dev_attention(dpool, batch, q, dtype, q_heads, scratch_bytes=64 << 20, max_seq_len=bound or None)
        assert rc == 0
        outs.append(got)
    assert outs[0].tobytes() == outs[1].tobytes()
    want = oracle.paged_attention(pool, hb, q, dtype, q_heads)
    G.assert_close(outs[0], dtype, want, what="plain decode", scale=G.channel_scale(v, dtype, hb, q_heads))

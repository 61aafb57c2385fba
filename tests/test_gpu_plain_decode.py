"""Decode steps without masks, windows and leftover columns, over TQ4 pages and row formats: the kernel that works ahead of the lengths gives the
bytes of the general one, which a batch without context_lens_before takes, and the oracle's values."""
import numpy as np
import pytest

import oracle
from cases import make_case
from oracle import DT_BF16, DT_F16, FMT_BF16, FMT_FP16, FMT_FP8, FMT_Q8_0, FMT_TQ4

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


# format, type, head dimension, then as above, and the mask mode (1: the tokens of a draft block see each other both ways)
ROWS = [
    (FMT_Q8_0, DT_F16, 256, 16, 2, 16, [1200], [1], 0, 0),
    (FMT_Q8_0, DT_BF16, 256, 64, 2, 16, [1200], [1], 5000, 0),
    (FMT_Q8_0, DT_F16, 256, 112, 1, 8, [1], [1], 0, 0),
    (FMT_FP8, DT_F16, 256, 48, 2, 16, [769], [1], 770, 0),
    (FMT_FP8, DT_BF16, 256, 16, 4, 4, [700, 9, 2500, 64], [1, 0, 1, 1], 10000, 0),
    (FMT_Q8_0, DT_F16, 256, 16, 2, 16, [2000], [4], 0, 0),               # two tiles
    (FMT_FP8, DT_F16, 256, 64, 1, 16, [300, 1000, 77], [3, 5, 1], 0, 0),  # tiles of one token, not as many in every request
    (FMT_FP16, DT_F16, 256, 16, 2, 16, [1700], [3], 0, 0),
    (FMT_BF16, DT_BF16, 256, 64, 2, 16, [500, 1030], [4, 2], 2000, 0),
    (FMT_BF16, DT_BF16, 128, 16, 4, 16, [700, 500], [16, 16], 0, 1),
    (FMT_BF16, DT_BF16, 128, 16, 4, 16, [65, 300, 17], [8, 16, 5], 0, 1),
    (FMT_FP16, DT_F16, 128, 32, 2, 8, [900], [6], 901, 0),
]


@pytest.mark.parametrize("case", range(len(ROWS)))
def test_row_formats(case):
    import gpu_harness as G

    fmt, dtype, head_dim, block, kv_heads, q_heads, seqs, q_lens, bound, mask_mode = ROWS[case]
    pool, bt, k, v, q, aq, ctx = make_case(fmt, block, seqs, q_lens, 3200 + case, dtype, kv_heads=kv_heads, q_heads=q_heads, head_dim=head_dim)
    hb = oracle.HostBatch(aq, seqs, bt, context_lens_before=ctx, mask_mode=mask_mode)
    dpool = G.DevPool(pool)
    dpool.upload()
    outs = []
    for batch in (hb, oracle.HostBatch(aq, seqs, bt, mask_mode=mask_mode)):
        rc, got, _ = G.dev_attention(dpool, batch, q, dtype, q_heads, scratch_bytes=64 << 20, max_seq_len=bound or None)
        assert rc == 0
        outs.append(got)
    assert outs[0].tobytes() == outs[1].tobytes()
    want = oracle.paged_attention(pool, hb, q, dtype, q_heads)
    G.assert_close(outs[0], dtype, want, what="plain rows", scale=G.channel_scale(v, dtype, hb, q_heads), plain_excess=0.0 if fmt in (FMT_FP16, FMT_BF16) else 4e-4)


# Several requests of one tile each, on the chunk grid (test_launch_choices.py holds that these forms are): format, type, page size, kv heads, q heads, keys
# and new tokens per request, bound on the keys (0: exact)
ON_GRID = [
    (FMT_TQ4, DT_F16, 32, 2, 16, [700, 9, 2500, 64], [1, 0, 1, 1], 8000),
    (FMT_TQ4, DT_BF16, 16, 2, 16, [700, 9, 2500, 64], [1, 1, 0, 1], 0),
    (FMT_TQ4, DT_F16, 64, 2, 4, [257, 5000, 31], [3, 4, 2], 10700),
    (FMT_Q8_0, DT_F16, 16, 2, 16, [700, 9, 2500, 64], [1, 0, 1, 1], 8000),
    (FMT_Q8_0, DT_BF16, 64, 1, 8, [300, 3000, 1, 2999], [0, 2, 1, 2], 0),
    (FMT_FP8, DT_F16, 48, 4, 4, [700, 9, 2500, 64], [1, 0, 5, 16], 8192),
    (FMT_FP8, DT_BF16, 16, 2, 16, [1200, 1201], [1, 1], 0),
]


@pytest.mark.parametrize("case", range(len(ON_GRID)))
def test_several_requests(case):
    import gpu_harness as G

    fmt, dtype, block, kv_heads, q_heads, seqs, q_lens, bound = ON_GRID[case]
    pool, bt, k, v, q, aq, ctx = make_case(fmt, block, seqs, q_lens, 3300 + case, dtype, kv_heads=kv_heads, q_heads=q_heads)
    hb = oracle.HostBatch(aq, seqs, bt, context_lens_before=ctx)
    dpool = G.DevPool(pool)
    dpool.upload()
    outs = []
    for batch in (hb, oracle.HostBatch(aq, seqs, bt)):
        rc, got, _ = G.dev_attention(dpool, batch, q, dtype, q_heads, scratch_bytes=64 << 20, max_seq_len=bound or None)
        assert rc == 0
        outs.append(got)
    assert np.array_equal(outs[0], outs[1])
    want = oracle.paged_attention(pool, hb, q, dtype, q_heads)
    G.assert_close(outs[0], dtype, want, what="plain decode of several requests", scale=G.channel_scale(v, dtype, hb, q_heads),
                   plain_excess=0.0 if fmt == FMT_TQ4 else 4e-4)

"""The private rest of a verify batch behind a shared prefix, more than 16 query columns per request and kv head: two column tiles
of a workgroup, whose sums join the records of the prefix's parts (no counterpart in the reference, which runs such a batch
without any split, op_paged_attn.cu:1399-1415)."""
import numpy as np
import pytest

import oracle
from oracle import DT_BF16

pytestmark = pytest.mark.gpu

# query heads (two kv heads), query tokens per request, keys per request, shared keys
CASES = {
    # a second tile of one column token, requests of 1 to 4 tokens, one of which has none behind the prefix but its own tokens
    "partly filled tiles": (16, (4, 3, 1, 4, 4), (33000, 33500, 32769, 32772, 34111), 32768),
    # several tiles per request, the last of one token; 16 heads per kv head: two tokens per tile
    "several tiles": (16, (16, 13, 5, 9), (34000, 33001, 40003, 33333), 32768),
    "group of 16": (32, (2, 3, 4, 5, 2), (33010, 33500, 36007, 33800, 32900), 32768),
    "group of 4": (8, (8, 7, 5, 6), (33010, 33500, 36007, 33800), 32768),
    "nothing shared": (16, (4, 4, 4, 4), (33000, 5000, 20011, 17), 0),
    # the fewest keys that count as shared
    "4096 shared": (16, (4, 4, 4, 4), (33000, 5000, 20011, 4103), 4096),
}


@pytest.mark.parametrize("name", sorted(CASES))
def test_private_rest_matches_oracle(name):
    from test_gpu_full_size import BS, BigPool

    q_heads, q_lens, ctx, shared = CASES[name]
    pool = BigPool(ctx, sum((c + BS - 1) // BS for c in ctx) + 8, seed=1201 + len(name), shared_prefix=shared)
    starts = np.concatenate([[0], np.cumsum(q_lens)]).astype(np.int32)
    n = int(starts[-1])
    q = oracle.fill_normal(n * q_heads * 256, 1301, DT_BF16).reshape(n, q_heads, 256)
    hb = oracle.HostBatch(starts, pool.ctx, pool.bt, context_lens_before=[c - t for c, t in zip(pool.ctx, q_lens)])
    want = oracle.paged_attention(pool.host, hb, q, DT_BF16, q_heads, n_threads=oracle.hw_threads())
    rc, got, _ = pool.G.dev_attention(pool.dev, hb, q, DT_BF16, q_heads, scratch_bytes=96 << 20)
    assert rc == 0
    scale = np.repeat(np.maximum(1.0, np.repeat(pool.v_absmax, q_heads // 2, axis=1)), q_lens, axis=0)
    pool.G.assert_close(got, DT_BF16, want, what=name, scale=scale)
    rc, plain, _ = pool.G.dev_attention(pool.dev, hb, q, DT_BF16, q_heads, scratch_bytes=8 << 20)  # as many chunks as with more, but not the records of the prefix
    assert rc == 0
    # another order of the same sums, unless nothing is shared
    assert (got.tobytes() == plain.tobytes()) == (shared == 0)

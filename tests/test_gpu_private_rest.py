"""The private rest of a verify batch behind a shared prefix, more than 16 query columns per request and kv head: one column tile per
workgroup where it is short, else two, whose sums join the records of the prefix's parts (no counterpart in the reference, which
runs such a batch without any split, op_paged_attn.cu:1399-1415)."""
import numpy as np
import pytest

import oracle
from cases import make_case
from oracle import DT_BF16, FMT_TQ4

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


LONG = 40000         # a bound from which on the shared keys get a pass of their own
WIDE_UNITS = 6144    # units behind the prefix from which on both column tiles go to one workgroup


def _long(block, q_lens, ctx, shared, seed, q_heads=16):
    """Long requests over few pages: their last two and the first behind the shared ones are their own, the others any.  -> pool, batch, queries, scale, units behind the prefix (once per
    column tile pair)"""
    keys = 8192 // block * block
    pool, pages, _, v, _, _, _ = make_case(FMT_TQ4, block, [keys], [1], seed, DT_BF16, q_heads=q_heads)
    pages, rng = pages[0], np.random.default_rng(seed)
    own, common = pages[:3 * len(ctx)].reshape(3, -1), pages[3 * len(ctx):]
    bt = rng.choice(common, (len(ctx), max(ctx) // block + 1)).astype(np.int32)
    bt[:, :shared // block] = bt[0, :shared // block]
    bt[:, shared // block] = own[0]  # (the shared keys end here)
    for r, n in enumerate(ctx):
        last = (n - 1) // block
        bt[r, last - 1:last + 1] = own[1:, r]
    starts = np.concatenate([[0], np.cumsum(q_lens)]).astype(np.int32)
    q = oracle.fill_normal(int(starts[-1]) * q_heads * 256, seed + 2, DT_BF16).reshape(-1, q_heads, 256)
    hb = oracle.HostBatch(starts, ctx, bt, context_lens_before=[n - t for n, t in zip(ctx, q_lens)])
    v_absmax = np.abs(oracle.bits_to_f32(v, DT_BF16)).max(axis=0)
    tok_tile, floor = 64 // q_heads, shared // block * block // 32
    units = sum(-(-t // tok_tile) * ((n - 1) // 32 - floor + 1) for n, t in zip(ctx, q_lens) if t)
    return pool, hb, q, np.repeat(np.maximum(1.0, v_absmax), q_heads // 2, axis=0)[None], units


def _attend(pool, hb, q, dpool=None, **over):
    import gpu_harness as G

    if dpool is None:
        dpool = G.DevPool(pool)
        dpool.upload()
    rc, got, _ = G.dev_attention(dpool, hb, q, DT_BF16, q.shape[1], scratch_bytes=96 << 20, **over)
    assert rc == 0
    return got


@pytest.mark.parametrize("bits", [0x7C00, 0xFFFF])     # an infinite and a NaN scale
@pytest.mark.parametrize("both_slabs", [False, True])  # the value rows, which leave the scores as they are, or the key rows too
@pytest.mark.parametrize("token", [3, 2])              # both in the second column tile of a request, the first one has tokens 0 and 1
def test_scales_of_unseen_rows(token, both_slabs, bits):
    """The scales of a token's rows are not finite: the tokens in front of it, which do not see them, keep their bits."""
    pool, hb, q, _, units = _long(64, (4,) * 8, [29000 + 37 * r for r in range(8)], 4096, 1401)
    assert units >= WIDE_UNITS
    outs = []
    for poisoned in (False, True):
        if poisoned:
            for slab in (pool.k, pool.v) if both_slabs else (pool.v,):
                rows = slab.reshape(-1, pool.kv_heads, pool.block_size, pool.tok).view(np.uint16)
                assert np.shares_memory(rows, slab)
                for r, pos in enumerate(hb.ctx + token):
                    rows[hb.bt[r, pos // 64], :, pos % 64][:, [0, 33]] = bits
        got = _attend(pool, hb, q, max_seq_len=LONG).reshape(8, 4, 16, 256)
        assert both_slabs or np.isnan(oracle.bits_to_f32(got[:, token:], DT_BF16)).all() == poisoned
        outs.append(got[:, :token])
    assert np.isfinite(oracle.bits_to_f32(outs[0], DT_BF16)).all()
    assert np.array_equal(outs[0], outs[1])


@pytest.mark.parametrize("wide", [False, True])
@pytest.mark.parametrize("q_lens,bounds", [((2,) * 8, (2, 3, 4, 16)), ((3, 1, 2, 2, 1, 3, 2, 2), (3, 4, 8)), ((4, 2, 4, 4, 4), (4, 5, 16)),
                                           ((4, 4, 4, 0, 4), (4, 5))])
def test_bytes_do_not_depend_on_the_bounds(q_lens, bounds, wide):
    """A short rest and one of just as many units as two column tiles want."""
    import gpu_harness as G

    tiles = sum(t > 0 for t in q_lens)
    units = (WIDE_UNITS + tiles - 1) // tiles if wide else 30
    pool, hb, q, scale, units = _long(64, q_lens, [4096 + 32 * units - r % 3 for r in range(len(q_lens))], 4096, 1501)
    assert (units >= WIDE_UNITS) == wide
    outs = [_attend(pool, hb, q, max_q_len=tokens, max_seq_len=keys) for tokens in bounds for keys in (LONG + 20000, 200000)]
    want = oracle.paged_attention(pool, hb, q, DT_BF16, 16, n_threads=oracle.hw_threads())
    G.assert_close(outs[0], DT_BF16, want, what="bound %d" % bounds[0], scale=scale)
    assert all(np.array_equal(got, outs[0]) for got in outs)


# pages of 16 keys (two per unit), of 48 (units across their edges) and of 64; the shared keys end inside a page of 48
@pytest.mark.parametrize("block,shared", [(16, 4096), (48, 4176), (64, 4096)])
@pytest.mark.parametrize("q_heads,q_lens,ctx", [(16, (4, 0, 5, 7, 8), (33000, 35001, 34015, 36001, 32912)), (32, (3, 5, 4, 5), (26017, 25002, 26000, 26001)),
                                                (8, (9, 16, 7, 12), (34001, 33000, 37007, 35555))])
def test_two_column_tiles(block, shared, q_heads, q_lens, ctx):
    import gpu_harness as G

    pool, hb, q, scale, units = _long(block, q_lens, ctx, shared, 1601, q_heads)
    assert units >= WIDE_UNITS
    got = _attend(pool, hb, q, max_seq_len=LONG)
    want = oracle.paged_attention(pool, hb, q, DT_BF16, q_heads, n_threads=oracle.hw_threads())
    G.assert_close(got, DT_BF16, want, what="pages of %d" % block, scale=scale)


def test_one_kv_head_gives_the_same_bytes():
    """Whether the rest is for two column tiles does not depend on the kv heads that a rank holds."""
    from test_gpu_head_sharding import _head_layout

    import gpu_harness as G

    for ctx in ((34017, 35001, 34000, 36001, 33912), (15017, 14001, 13015, 16001, 14912)):
        pool, hb, q, _, units = _long(64, (4, 5, 4, 7, 8), ctx, 4096, 1701)
        assert (units >= WIDE_UNITS) == (ctx[0] > 20000)
        full = _attend(pool, hb, q, max_seq_len=LONG)
        dpool = G.DevPool(pool)
        dpool.upload()
        for head in range(2):
            q_h = np.ascontiguousarray(q[:, head * 8:(head + 1) * 8])
            part = _attend(pool, hb, q_h, max_seq_len=LONG, dpool=dpool, layout=_head_layout(dpool, head))
            assert np.array_equal(part, full[:, head * 8:(head + 1) * 8])

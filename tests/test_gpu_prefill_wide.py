"""Chunked prefill in tiles of 256 query rows: every page format, whole tiles and tiles of the last round that are cut in two, more
requests than a wave has lanes, and the TQ4 kernels of both tile sizes against each other byte for byte."""
import numpy as np
import pytest

import oracle
from oracle import DT_BF16, DT_F16, FMT_BF16, FMT_FP16, FMT_FP8, FMT_Q8_0, FMT_TQ4, XF_IDENTITY, XF_WHT256
from cases import make_case

pytestmark = pytest.mark.gpu
SCRATCH = 8 << 20
WIDE = 2  # of the test selector


def _run(fmt, dtype, block, seq_lens, q_lens, seed, xf=None, v_xf=None, q_heads=16, keep=0.2, force=None, mask_mode=0, window=0, excess=0.0):
    """Attention of the tokens that a random mask keeps (the others cost the oracle nothing), held to the contract."""
    import gpu_harness as G

    pool, bt, k, v, q, aq, ctx = make_case(fmt, block, seq_lens, q_lens, seed, dtype, q_heads=q_heads, xf=xf, v_xf=v_xf)
    tmask = (np.random.default_rng(seed).random(aq[-1]) < keep).astype(np.uint8)
    tmask[[0, aq[-1] - 1]] = 1
    hb = oracle.HostBatch(aq, seq_lens, bt, context_lens_before=ctx, valid_token_mask=tmask, mask_mode=mask_mode,
                          sliding_window=window)
    want = oracle.paged_attention(pool, hb, q, dtype, q_heads, n_threads=8)
    dpool = G.DevPool(pool)
    dpool.upload()
    rc, got, _ = G.dev_attention(dpool, hb, q, dtype, q_heads, scratch_bytes=SCRATCH, force_kernel=force)
    assert rc == 0
    live = tmask != 0
    assert (got[~live] == 0x5500).all()
    G.assert_close(got[live], dtype, want[live], what="wide tiles fmt=%d seq=%s q=%s" % (fmt, seq_lens[:4], q_lens[:4]),
                   scale=G.channel_scale(v, dtype, hb, q_heads)[live], plain_excess=excess)
    return dpool, hb, q, got


FORMATS = [(FMT_TQ4, DT_F16, XF_WHT256), (FMT_TQ4, DT_BF16, XF_IDENTITY), (FMT_FP8, DT_F16, XF_IDENTITY), (FMT_FP8, DT_BF16, XF_WHT256),
           (FMT_Q8_0, DT_BF16, XF_IDENTITY), (FMT_Q8_0, DT_F16, XF_WHT256), (FMT_FP16, DT_F16, XF_IDENTITY),
           (FMT_BF16, DT_BF16, XF_IDENTITY)]


@pytest.mark.parametrize("fmt,dtype,xf", FORMATS)
@pytest.mark.parametrize("block,seq_lens,q_lens", [
    (16, [1733, 1100, 905], [1733, 1003, 701]),      # 220 tiles: the longest 36 in halves
    (64, [2100, 1999, 1300], [1900, 1777, 1201]),    # 308 tiles: the last 52 in halves
])
def test_whole_and_cut_tiles(fmt, dtype, xf, block, seq_lens, q_lens):
    # plain TQ4 rows: an element of an outlier row's block is up to the outlier's size times the table's 9.4e-5 off (the allowance
    # of test_tq4_plain_slabs_batched_decode_and_prefill); 128-row tiles are as far off, to the digit
    excess = 2.5e-3 if fmt == FMT_TQ4 and xf == XF_IDENTITY else 0.0
    xf = None if fmt in (FMT_FP16, FMT_BF16) else xf
    _run(fmt, dtype, block, seq_lens, q_lens, 1201, xf=xf, v_xf=xf, keep=0.1, excess=excess)


@pytest.mark.parametrize("fmt,dtype", [(FMT_TQ4, DT_F16), (FMT_Q8_0, DT_F16), (FMT_BF16, DT_BF16)])
def test_more_requests_than_lanes(fmt, dtype):
    n = 70
    q_lens = [33 + (7 * r) % 40 for r in range(n)]
    _run(fmt, dtype, 16, [q + 50 + 3 * r for r, q in enumerate(q_lens)], q_lens, 1301, keep=0.5, force=WIDE if dtype == DT_F16 else None)


@pytest.mark.parametrize("q_heads", [2, 8, 16, 32])
@pytest.mark.parametrize("mask_mode,window", [(0, 0), (0, 100), (1, 0), (1, 64), (0, 1)])
def test_tq4_tile_sizes_agree(q_heads, mask_mode, window):
    """256-row tiles (whole and halves) and 128-row tiles on twelve waves: the same bytes."""
    import gpu_harness as G

    dpool, hb, q, got = _run(FMT_TQ4, DT_F16, 16, [700, 333, 65], [400, 333, 1], 1401, q_heads=q_heads, keep=0.7, force=WIDE,
                             mask_mode=mask_mode, window=window)
    rc, other, _ = G.dev_attention(dpool, hb, q, DT_F16, q_heads, force_kernel=1)
    assert rc == 0 and other.tobytes() == got.tobytes()


def test_tq4_tile_sizes_agree_on_whole_tiles():
    import gpu_harness as G

    dpool, hb, q, got = _run(FMT_TQ4, DT_F16, 64, [2100, 1999, 1300], [1900, 1777, 1201], 1501, keep=0.1, force=WIDE)
    rc, other, _ = G.dev_attention(dpool, hb, q, DT_F16, 16, force_kernel=1)
    assert rc == 0 and other.tobytes() == got.tobytes()


@pytest.mark.parametrize("fmt", [FMT_TQ4, FMT_Q8_0, FMT_FP16])
def test_one_kv_head_gives_the_same_bytes(fmt):
    """Half the heads are half the tiles, of which other ones are cut in two."""
    import gpu_harness as G
    from test_gpu_head_sharding import _head_layout

    dpool, hb, q, full = _run(fmt, DT_F16, 64, [2100, 1999, 1300], [1900, 1777, 1201], 1601, keep=0.1)
    for head in range(2):
        q_h = np.ascontiguousarray(q[:, head * 8:(head + 1) * 8])
        rc, part, _ = G.dev_attention(dpool, hb, q_h, DT_F16, 8, layout=_head_layout(dpool, head))
        assert rc == 0
        assert part.tobytes() == np.ascontiguousarray(full[:, head * 8:(head + 1) * 8]).tobytes()


@pytest.mark.parametrize("bits", [0x7C00, 0xFFFF])  # an infinite and a NaN scale
def test_tq4_scales_of_unseen_rows(bits):
    """The scales of rows behind the sequence and of a token that only the last query token sees are not finite: every other token's
    output has the bits it has without them."""
    import gpu_harness as G

    seq, ql = 333, 333
    pool, bt, k, v, q, aq, ctx = make_case(FMT_TQ4, 64, [seq], [ql], 1701, DT_F16, q_heads=16)
    hb = oracle.HostBatch(aq, [seq], bt, context_lens_before=ctx)
    outs = []
    for poisoned in (False, True):
        if poisoned:
            for slab in (pool.k, pool.v):
                rows = slab.reshape(-1, pool.kv_heads, pool.block_size, pool.tok)[bt[0, (seq - 1) // 64]]
                scales = rows.view(np.uint16) if rows.flags["C_CONTIGUOUS"] else None
                assert scales is not None
                scales[:, (seq - 1) % 64:, [0, 33]] = bits
        dpool = G.DevPool(pool)
        dpool.upload()
        for force in (1, WIDE):
            rc, got, _ = G.dev_attention(dpool, hb, q, DT_F16, 16, force_kernel=force)
            assert rc == 0
            outs.append(got[:-1].tobytes())
    assert all(o == outs[0] for o in outs)


@pytest.mark.parametrize("xf", [XF_WHT256, XF_IDENTITY])
def test_tq4_value_scales_that_leave_no_room_above_one(xf):
    """Value scales of 3 000 in every third token: a probability of more than 21 times such a scale is no fp16 number, so a running maximum
    that lags behind the scores would overflow there.  Tiles of both sizes, the same bytes."""
    import gpu_harness as G

    seq, ql = [700, 333], [300, 333]
    pool, bt, k, v, q, aq, ctx = make_case(FMT_TQ4, 64, seq, ql, 1801, DT_F16, q_heads=16, xf=xf, v_xf=xf)
    rows = pool.v.reshape(-1, pool.kv_heads, pool.block_size, pool.tok).view(np.uint16)
    assert np.shares_memory(rows, pool.v)
    rows[:, :, ::3, [0, 33]] = np.float16(3000.0).view(np.uint16)
    hb = oracle.HostBatch(aq, seq, bt, context_lens_before=ctx)
    want = oracle.paged_attention(pool, hb, q, DT_F16, 16, n_threads=8)
    dpool = G.DevPool(pool)
    dpool.upload()
    outs = []
    for force in (1, WIDE):
        rc, got, _ = G.dev_attention(dpool, hb, q, DT_F16, 16, force_kernel=force)
        assert rc == 0
        outs.append(got)
    assert outs[0].tobytes() == outs[1].tobytes()
    out = oracle.bits_to_f32(outs[0], DT_F16).astype(np.float64)
    assert np.isfinite(out).all()
    # the scores' error, 2e-3 of the largest value scale, and the output's rounding
    assert (np.abs(out - want) <= 1e-2 * np.abs(want) + 2e-3 * 3000.0).all()

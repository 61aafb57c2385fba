"""Contexts and batches of few chunks: shorter chunks, and a merge of one wave per row, against the oracle at the lengths where the number of chunks and
the form of the merge change; and, with a bound on the length under which the merge of several waves runs, the same bytes."""
import ctypes as C

import numpy as np
import pytest

import oracle
from cases import make_case
from oracle import DT_BF16, DT_F16, FMT_BF16, FMT_FP16, FMT_FP8, FMT_Q8_0, FMT_TQ4, XF_IDENTITY, XF_WHT256

pytestmark = pytest.mark.gpu
SCRATCH = 64 << 20
UNIT = 32


@pytest.mark.parametrize("fmt,dtype,head_dim", [(FMT_TQ4, DT_F16, 256), (FMT_TQ4, DT_BF16, 256), (FMT_Q8_0, DT_F16, 256),
                                                (FMT_FP8, DT_BF16, 256), (FMT_BF16, DT_BF16, 128)])
@pytest.mark.parametrize("units", [8, 9, 32, 33, 64, 65, 96, 128, 129, 200, 257])
def test_lengths_at_which_the_chunks_change(fmt, dtype, head_dim, units):
    """One token (rows summed in the order of sixteen waves) and four (of four), a whole last unit and one key in it."""
    import gpu_harness as G

    q_heads, kv_heads = 16, 2 if head_dim == 256 else 4
    for q_len, seq in ((1, units * UNIT), (4, (units - 1) * UNIT + 1)):
        pool, bt, k, v, q, aq, ctx = make_case(fmt, 64, [seq], [q_len], 2300 + units, dtype, kv_heads=kv_heads, q_heads=q_heads,
                                               head_dim=head_dim)
        mask = np.ones(q_len, dtype=np.uint8)
        if q_len > 1:
            mask[1] = 0
        hb = oracle.HostBatch(aq, [seq], bt, context_lens_before=ctx, valid_token_mask=mask)
        want = oracle.paged_attention(pool, hb, q, dtype, q_heads)
        dpool = G.DevPool(pool)
        dpool.upload()
        rc, got, _ = G.dev_attention(dpool, hb, q, dtype, q_heads, scratch_bytes=SCRATCH)
        assert rc == 0
        live = mask != 0
        assert (got[~live] == 0x5500).all()
        G.assert_close(got[live], dtype, want[live], what="fmt=%d seq=%d q=%d" % (fmt, seq, q_len),
                       scale=G.channel_scale(v, dtype, hb, q_heads)[live])
        rc, wide, _ = G.dev_attention(dpool, hb, q, dtype, q_heads, scratch_bytes=SCRATCH, max_seq_len=131072)
        assert rc == 0 and wide.tobytes() == got.tobytes()


@pytest.mark.parametrize("fmt,dtype", [(FMT_TQ4, DT_BF16), (FMT_Q8_0, DT_F16)])
@pytest.mark.parametrize("q_len,seq", [(1, 300), (1, 1200), (4, 1200), (4, 5000), (1, 9000)])
def test_queried_scratch_gives_the_bytes_of_a_large_one(fmt, dtype, q_len, seq):
    import gpu_harness as G

    pool, bt, k, v, q, aq, ctx = make_case(fmt, 64, [seq], [q_len], 2600 + seq, dtype)
    hb = oracle.HostBatch(aq, [seq], bt, context_lens_before=ctx)
    dpool = G.DevPool(pool)
    dpool.upload()
    need = G.lib().warp34_paged_attention_scratch_bytes_for_layout(C.byref(dpool.layout()), q_len, 1, 16, seq)
    outs = []
    for scratch in (need, SCRATCH):
        rc, got, _ = G.dev_attention(dpool, hb, q, dtype, 16, scratch_bytes=scratch, max_seq_len=seq)
        assert rc == 0
        outs.append(got.tobytes())
    assert outs[0] == outs[1]


@pytest.mark.parametrize("fmt,dtype,xf", [(FMT_TQ4, DT_BF16, None), (FMT_Q8_0, DT_F16, XF_IDENTITY), (FMT_Q8_0, DT_F16, XF_WHT256),
                                          (FMT_FP16, DT_F16, None)])
@pytest.mark.parametrize("reqs,longest", [(2, 1024), (2, 1025), (16, 128), (16, 129), (17, 180), (17, 181), (64, 48), (64, 49), (65, 20),
                                            (2, 512), (2, 513), (12, 80), (12, 81), (16, 64), (16, 65), (17, 120), (17, 121), (64, 32), (64, 33)])
def test_decode_batches_on_either_side_of_the_grid_rule(fmt, dtype, xf, reqs, longest):
    """Chunk grid and plan give the same bytes for a batch that the chunk grid may serve: which of them runs follows from the host's bound on
    the lengths (units of the longest request: 8 x (128 / requests); from 17 requests on, times requests, 3 072, row formats 2 048).  A
    masked request among the others."""
    import gpu_harness as G

    rng = np.random.default_rng(reqs * 1000 + longest)
    seq = [int(x) for x in rng.integers(1, longest * UNIT if reqs == 2 else max(2, longest * UNIT // 4), reqs)]
    seq[-1] = longest * UNIT
    q_heads = 16 if reqs < 17 else 8
    pool, bt, k, v, q, aq, ctx = make_case(fmt, 16, seq, [1] * reqs, 2400 + reqs, dtype, q_heads=q_heads, xf=xf)
    mask = np.ones(reqs, dtype=np.uint8)
    if reqs > 2:
        mask[1] = 0
    hb = oracle.HostBatch(aq, seq, bt, context_lens_before=ctx, valid_req_mask=mask)
    want = oracle.paged_attention(pool, hb, q, dtype, q_heads, n_threads=8)
    dpool = G.DevPool(pool)
    dpool.upload()
    outs = []
    for bound in (max(seq), max(seq) + 40 * UNIT, 131072):
        rc, got, _ = G.dev_attention(dpool, hb, q, dtype, q_heads, scratch_bytes=SCRATCH, max_seq_len=bound)
        assert rc == 0
        assert (got[mask == 0] == 0x5500).all()
        outs.append(got.tobytes())
    live = mask != 0
    G.assert_close(got[live], dtype, want[live], what="fmt=%d reqs=%d longest=%d units" % (fmt, reqs, longest),
                   scale=G.channel_scale(v, dtype, hb, q_heads)[live], plain_excess=4e-4 if xf == XF_WHT256 else 0.0)
    assert outs[0] == outs[1] == outs[2]

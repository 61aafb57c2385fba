"""Verify steps and draft blocks: requests with more than 16 query columns per kv head (two column
tiles per workgroup, several tiles per request) on the balanced plan, at the edges of halves, units,
pieces and entry groups; against the oracle at the contract bound."""
import numpy as np
import pytest

import oracle
from oracle import DT_BF16, DT_F16, FMT_BF16, FMT_FP16, FMT_FP8, FMT_Q8_0, FMT_TQ4, XF_IDENTITY, XF_WHT256
from test_gpu_attention import _check

pytestmark = pytest.mark.gpu

SCRATCH = 64 << 20
ROWS = [(FMT_BF16, DT_BF16), (FMT_FP16, DT_F16), (FMT_FP8, DT_F16), (FMT_Q8_0, DT_BF16)]


@pytest.mark.parametrize("fmt,dtype", ROWS)
@pytest.mark.parametrize("seq,q", [([4], [4]), ([16, 17, 33], [4, 3, 4]), ([700, 31, 2500, 48, 900], [4, 4, 3, 1, 2]),
                                   ([5000, 64], [4, 4]), ([130, 900, 70], [9, 16, 5])])
def test_rows_verify_column_tiles(fmt, dtype, seq, q):
    """One to four tiles per request, pieces that end inside a unit, requests shorter than a half."""
    _check(fmt, dtype, 16, seq, q, 411, scratch=SCRATCH, q_heads=16)


@pytest.mark.parametrize("mask_mode", [0, 1])
@pytest.mark.parametrize("seq,q", [([16], [16]), ([300, 41, 1000], [16, 16, 8]), ([2100, 90], [16, 9])])
def test_rows_draft_blocks_head_dim_128(mask_mode, seq, q):
    """Blocks of up to sixteen tokens at head dimension 128, causal and seeing each other both ways."""
    _check(FMT_BF16, DT_BF16, 16, seq, q, 412, scratch=SCRATCH, q_heads=16, kv_heads=4, head_dim=128, mask_mode=mask_mode)


@pytest.mark.parametrize("fmt,dtype", [(FMT_Q8_0, DT_F16), (FMT_BF16, DT_BF16)])
@pytest.mark.parametrize("n", [17, 33, 70])
def test_rows_verify_many_requests(fmt, dtype, n):
    """More entries than are cut into pieces of their own, and more than one group of 64."""
    seq = [20 + 37 * ((i * 7) % 11) for i in range(n)]
    _check(fmt, dtype, 64, seq, [1 + (i % 6) for i in range(n)], 413, scratch=SCRATCH, q_heads=16)


@pytest.mark.parametrize("scratch", [2 << 20, 7 << 20, 8 << 20])
def test_rows_verify_small_scratch(scratch):
    """20 requests in 8 MiB: 106 of the plan's 128 shares.  7 MiB would hold 90: the chunk grid.  Three requests are
    on the grid with any scratch."""
    _check(FMT_FP8, DT_F16, 64, [3000, 900, 2000], [4, 4, 4], 414, scratch=scratch, q_heads=16)
    _check(FMT_FP8, DT_F16, 64, [30 + 61 * ((i * 7) % 20) for i in range(20)], [4] * 20, 419, scratch=scratch, q_heads=16)


@pytest.mark.parametrize("fmt", [FMT_FP8, FMT_Q8_0])
def test_rows_verify_rotated_keys_or_values(fmt):
    """Rotated 8-bit rows: one column tile, several tiles per request; keys alone rotated: two."""
    _check(fmt, DT_F16, 16, [300, 45, 800], [4, 2, 3], 415, scratch=SCRATCH, q_heads=16, xf=XF_WHT256, plain_excess=4e-4)
    _check(fmt, DT_F16, 16, [300, 45, 800], [4, 2, 3], 416, scratch=SCRATCH, q_heads=16, xf=XF_WHT256, v_xf=XF_IDENTITY,
           plain_excess=4e-4)


@pytest.mark.parametrize("fmt,dtype", [(FMT_BF16, DT_BF16), (FMT_Q8_0, DT_F16)])
@pytest.mark.parametrize("n", [4, 5])
def test_rows_verify_either_side_of_the_grid_rule(fmt, dtype, n):
    """Four requests of four tokens (8 tiles per kv head) run on the chunk grid, five on the plan; short and
    longer requests, for which the plan cuts pieces of 4 units and of more."""
    for seq in ([130, 40, 300, 90, 17][:n], [2600, 900, 4000, 31, 1500][:n]):
        _check(fmt, dtype, 16, seq, [4] * n, 417, scratch=SCRATCH, q_heads=16)


@pytest.mark.parametrize("fmt,dtype", [(FMT_Q8_0, DT_F16), (FMT_BF16, DT_BF16)])
@pytest.mark.parametrize("n,q", [(200, 1), (235, 1), (60, 4), (110, 4)])
def test_rows_large_batches_in_8mib_keep_a_workgroup_per_tile(fmt, dtype, n, q):
    """8 MiB hold the records of 52, 17, 66 or 16 shares of these batches: they run as one workgroup per tile, the
    scratch stays untouched and the bits are those of a call without scratch."""
    import gpu_harness as G
    from cases import make_case

    seq = [10 + 23 * ((i * 5) % 7) for i in range(n)]
    pool, bt, k, v, qb, aq, ctx = make_case(fmt, 16, seq, [q] * n, 418, dtype, q_heads=16)
    hb = oracle.HostBatch(aq, seq, bt, context_lens_before=ctx)
    dpool = G.DevPool(pool)
    dpool.upload()
    rc0, plain, _ = G.dev_attention(dpool, hb, qb, dtype, 16)
    rc1, got, ws = G.dev_attention(dpool, hb, qb, dtype, 16, scratch_bytes=8 << 20)
    assert rc0 == 0 and rc1 == 0
    assert bool((ws == 0x5A).all()), "the scratch was used"
    assert got.tobytes() == plain.tobytes()


@pytest.mark.parametrize("fmt,dtype", [(FMT_Q8_0, DT_F16), (FMT_BF16, DT_BF16)])
@pytest.mark.parametrize("lens", [37, 211])
def test_rows_verify_in_8mib_keeps_the_plan_while_it_has_the_workgroups(fmt, dtype, lens):
    """40 requests x 4 tokens: 86 shares for 80 tiles of 16 columns.  Short and longer batches."""
    import gpu_harness as G
    from cases import make_case

    seq = [40 + lens * ((i * 7) % 11) for i in range(40)]
    pool, bt, k, v, qb, aq, ctx = make_case(fmt, 64, seq, [4] * 40, 423, dtype, q_heads=16)
    hb = oracle.HostBatch(aq, seq, bt, context_lens_before=ctx)
    dpool = G.DevPool(pool)
    dpool.upload()
    rc, got, ws = G.dev_attention(dpool, hb, qb, dtype, 16, scratch_bytes=8 << 20)
    assert rc == 0 and not bool((ws == 0x5A).all())
    want = oracle.paged_attention(pool, hb, qb, dtype, 16, n_threads=4)
    G.assert_close(got, dtype, want, what="40 x 4 in 8 MiB", scale=G.channel_scale(v, dtype, hb, 16))


@pytest.mark.parametrize("fmt,dtype", [(FMT_Q8_0, DT_F16), (FMT_BF16, DT_BF16)])
@pytest.mark.parametrize("n,q", [(1, 1), (1, 4), (5, 4), (3, 16), (40, 1), (40, 4)])
def test_rows_scratch_of_the_queried_size_splits_fully(fmt, dtype, n, q):
    """The bits of a call with the scratch the query names are those of a call with 64 MiB."""
    import ctypes as C

    import gpu_harness as G
    from cases import make_case

    seq = [16 + 131 * ((i * 5) % 9) for i in range(n)]
    pool, bt, k, v, qb, aq, ctx = make_case(fmt, 16, seq, [q] * n, 420, dtype, q_heads=16)
    hb = oracle.HostBatch(aq, seq, bt, context_lens_before=ctx)
    dpool = G.DevPool(pool)
    dpool.upload()
    L = dpool.layout()
    need = G.lib().warp34_paged_attention_scratch_bytes_for_layout(C.byref(L), n * q, n, 16, max(seq))
    rc0, want, _ = G.dev_attention(dpool, hb, qb, dtype, 16, scratch_bytes=SCRATCH)
    rc1, got, _ = G.dev_attention(dpool, hb, qb, dtype, 16, scratch_bytes=need)
    assert rc0 == 0 and rc1 == 0
    assert got.tobytes() == want.tobytes()


@pytest.mark.parametrize("fmt,dtype", ROWS)
@pytest.mark.parametrize("seq,q", [([200, 31, 224, 17, 9], [4, 4, 4, 4, 4]), ([40 + 9 * (i % 20) for i in range(20)], [4] * 20),
                                   ([60 + 41 * (i % 5) for i in range(64)], [3] * 64), ([224, 130, 33], [16, 16, 9])])
def test_rows_short_batches_do_not_depend_on_the_sequence_bound(fmt, dtype, seq, q):
    """No request above 224 keys: on the chunk grid where the host's bound says so, as pieces of 16 columns where the
    plan finds it out; the same bits, and the oracle's answer."""
    _short_batch(fmt, dtype, seq, q)


@pytest.mark.parametrize("fmt", [FMT_FP8, FMT_Q8_0])
def test_rows_short_batches_of_rotated_rows(fmt):
    """One column tile, 40 and 60 entries; few enough entries keep the plan with any bound."""
    for seq, q in (([40 + 9 * (i % 20) for i in range(20)], [4] * 20), ([31, 224, 100, 60, 17] * 3, [7] * 15), ([200] * 5, [4] * 5)):
        _short_batch(fmt, DT_F16, seq, q, xf=XF_WHT256, plain_excess=4e-4)
    seq = [16 + 37 * ((i * 7) % 20) for i in range(20)]
    _check(fmt, DT_F16, 16, seq, [4] * 20, 425, scratch=SCRATCH, q_heads=16, xf=XF_WHT256, plain_excess=4e-4)
    _check(fmt, DT_F16, 16, [9 * s for s in seq], [4] * 20, 426, scratch=SCRATCH, q_heads=16, xf=XF_WHT256, plain_excess=4e-4)


def _short_batch(fmt, dtype, seq, q, xf=None, plain_excess=0.0):
    import gpu_harness as G
    from cases import make_case

    pool, bt, k, v, qb, aq, ctx = make_case(fmt, 16, seq, q, 421, dtype, q_heads=16, xf=xf)
    hb = oracle.HostBatch(aq, seq, bt, context_lens_before=ctx)
    dpool = G.DevPool(pool)
    dpool.upload()
    outs = []
    for bound in (None, 224, 225, 4096, 131072):
        rc, out, _ = G.dev_attention(dpool, hb, qb, dtype, 16, scratch_bytes=SCRATCH, max_seq_len=bound)
        assert rc == 0
        outs.append(out)
    assert all(o.tobytes() == outs[0].tobytes() for o in outs[1:])
    want = oracle.paged_attention(pool, hb, qb, dtype, 16, n_threads=4)
    G.assert_close(outs[0], dtype, want, what="short batch", scale=G.channel_scale(v, dtype, hb, 16), plain_excess=plain_excess)


@pytest.mark.parametrize("fmt,dtype", [(FMT_Q8_0, DT_F16), (FMT_BF16, DT_BF16)])
def test_rows_short_batches_with_idle_requests(fmt, dtype):
    """20 requests of up to 900 keys, more than 64 tiles of 16 columns among them, masked requests left untouched;
    and the same lengths eight times over, which is no short batch any more."""
    import gpu_harness as G
    from cases import make_case

    for scale, n, q in ((1, 20, 4), (8, 20, 4), (1, 30, 6), (1, 21, 9)):
        seq = [16 + scale * (37 + 97 * ((i * 7) % 9)) for i in range(n)]
        mask = [0 if i % 6 == 5 else 1 for i in range(n)]
        pool, bt, k, v, qb, aq, ctx = make_case(fmt, 64, seq, [q] * n, 422, dtype, q_heads=16)
        hb = oracle.HostBatch(aq, seq, bt, context_lens_before=ctx, valid_req_mask=mask)
        dpool = G.DevPool(pool)
        dpool.upload()
        rc, got, _ = G.dev_attention(dpool, hb, qb, dtype, 16, scratch_bytes=SCRATCH)
        assert rc == 0
        live = np.repeat(np.array(mask), q) != 0
        assert bool((got[~live] == 0x5500).all()), "masked requests were written"
        want = oracle.paged_attention(pool, hb, qb, dtype, 16, n_threads=4)
        G.assert_close(got[live], dtype, want[live], what="short batch, masked requests x%d" % scale,
                       scale=G.channel_scale(v, dtype, hb, 16)[live])


@pytest.mark.parametrize("n", [2, 3, 4, 7])
def test_rows_decode_head_dim_128_either_side_of_the_grid_rule(n):
    """Up to three requests on the chunk grid, more on the plan."""
    _check(FMT_BF16, DT_BF16, 16, [1500, 37, 4000, 700, 16, 2100, 330][:n], [1] * n, 424, scratch=SCRATCH, q_heads=16, kv_heads=4,
           head_dim=128)


def test_rows_verify_graph_serves_short_and_long_batches():
    """One captured verify step of 20 requests x 4 tokens; the lengths on the device change between replays from
    a short batch to a long one and back.  Every replay gives the bits of an eager call."""
    import torch

    import gpu_harness as G
    from cases import make_case

    n = 20
    long = [1400 - 3 * i for i in range(n)]
    pool, bt, k, v, qb, aq, ctx = make_case(FMT_BF16, 64, long, [4] * n, 427, DT_BF16, q_heads=16)
    hb = oracle.HostBatch(aq, long, bt, context_lens_before=ctx)
    dpool = G.DevPool(pool)
    dpool.upload()
    L = dpool.layout()
    db = G.DevBatch(hb, max_seq_len=8192)
    B = db.struct()
    lens = {"long": long, "short": [90 + 17 * (i % 13) for i in range(n)], "mixed": [90 if i % 2 else s for i, s in enumerate(long)]}
    q = G.to_dev(qb)
    out = torch.zeros((4 * n, 16, 256), dtype=torch.int16, device=G.DEV)
    ws = torch.zeros(SCRATCH, dtype=torch.uint8, device=G.DEV)

    def set_lengths(name):
        s = np.array(lens[name], dtype=np.int32)
        db.t["seq"].copy_(torch.from_numpy(s))
        db.t["ctx"].copy_(torch.from_numpy(s - 4))

    def call():
        import ctypes as C

        from warp34_amd import ffi
        ex = ffi.Warp34Exec(torch.cuda.current_stream().cuda_stream, ws.data_ptr(), ws.numel(), 0)
        assert G.lib().warp34_paged_attention_bf16(C.byref(ex), C.byref(L), C.byref(B), G.ptr(q), G.ptr(out), 16) == 0

    want = {}
    for name in lens:
        set_lengths(name)
        call()
        torch.cuda.synchronize()
        want[name] = out.clone()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        call()
    for name in ("short", "long", "mixed", "short", "long"):
        set_lengths(name)
        out.fill_(0)
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, want[name]), name


@pytest.mark.parametrize("fmt,dtype", [(FMT_Q8_0, DT_F16), (FMT_BF16, DT_BF16)])
@pytest.mark.parametrize("q_heads", [4, 10, 12, 20, 40, 64])
def test_rows_short_batches_other_group_sizes(fmt, dtype, q_heads):
    """2 to 32 q heads per kv head: groups that do not fill a tile of 16 columns, two q subgroups."""
    n = 24
    _check(fmt, dtype, 16, [30 + 53 * ((i * 7) % 12) for i in range(n)], [4 + 5 * (i % 2) for i in range(n)], 428, scratch=SCRATCH,
           q_heads=q_heads)
    _check(fmt, dtype, 16, [100 + 9 * (i % 14) for i in range(n)], [9] * n, 429, scratch=SCRATCH, q_heads=q_heads)


@pytest.mark.parametrize("fmt,dtype,heads,head_dim", [(FMT_TQ4, DT_F16, 2, 256), (FMT_Q8_0, DT_F16, 2, 256), (FMT_BF16, DT_BF16, 4, 128)])
@pytest.mark.parametrize("seq,q", [([900, 900, 900], [16, 16, 16]), ([900, 60, 1500], [1, 3, 16]), ([40, 2500, 300], [16, 1, 2]),
                                   ([700, 33], [5, 5]), ([1800], [16]), ([64, 900, 500, 200], [0, 7, 0, 7]),
                                   ([30 + 11 * (i % 17) for i in range(70)], [1 + (i * 5) % 6 for i in range(70)])])
def test_grid_of_several_tiles_per_request(fmt, dtype, heads, head_dim, seq, q):
    """The grid's bound (as many tiles for every request as the longest has, or one more per request than the tokens
    fill): all requests full, only the first or only the last, none; and the request guessed from the tile number right,
    wrong, and behind the last; more requests than a wave looks up at a time."""
    _check(fmt, dtype, 16, seq, q, 431, scratch=SCRATCH, q_heads=16, kv_heads=heads, head_dim=head_dim)


@pytest.mark.parametrize("fmt,dtype,q_heads,kv_heads,head_dim,seq,q", [
    # 7 chunks x 4 heads, 9 requests of two tiles; 3 x 3; 1 x 4 (no split)
    (FMT_BF16, DT_BF16, 16, 4, 128, [2000 + 131 * i for i in range(9)], [8] * 9),
    (FMT_BF16, DT_BF16, 12, 3, 128, [900 + 257 * i for i in range(9)], [16] * 9),
    (FMT_FP16, DT_F16, 16, 4, 128, [20 + 31 * (i % 7) for i in range(30)], [16] * 30),
    # requests with fewer tiles than the longest, none at all; two q subgroups (20 q heads per kv head)
    (FMT_BF16, DT_BF16, 16, 4, 128, [1500] * 8 + [70], [16, 16, 9, 16, 16, 0, 16, 16, 13]),
    (FMT_BF16, DT_BF16, 40, 2, 128, [900, 40, 1300, 700, 2100], [5] * 5),
    # by length, eight requests in the first round (launch order, 8 a tile; equal lengths, a request without tokens) and ten (by keys)
    (FMT_BF16, DT_BF16, 16, 4, 128, [2100, 300, 2100, 90, 1500, 16, 700, 2100, 40, 1100, 1900, 333], [16] * 12),
    (FMT_FP16, DT_F16, 16, 4, 128, [2001 - 170 * i for i in range(11)], [16, 3, 16, 16, 0, 16, 16, 16, 16, 9, 16]),
    (FMT_BF16, DT_BF16, 12, 3, 128, [90, 4000, 3100, 16, 800, 2222, 60, 4000, 1000], [16] * 9),
    # head dimension 256: 21 chunks x 2 heads, 63 x 2
    (FMT_Q8_0, DT_F16, 16, 2, 256, [6000, 900, 6000], [4] * 3),
    (FMT_FP8, DT_F16, 16, 2, 256, [16000], [4]),
    (FMT_BF16, DT_BF16, 8, 1, 256, [9000, 40, 9000], [4, 3, 4]),
])
def test_chunk_grid_by_groups_of_keys(fmt, dtype, q_heads, kv_heads, head_dim, seq, q):
    """Workgroups that are not a multiple of eight a tile go by the keys they share, long requests at head dimension 128 by length; the
    bits are those of launch order, where a batch without a bound on its requests' tokens stays."""
    import gpu_harness as G
    from cases import make_case

    pool, bt, k, v, qb, aq, ctx = make_case(fmt, 16, seq, q, 432, dtype, kv_heads=kv_heads, q_heads=q_heads, head_dim=head_dim)
    hb = oracle.HostBatch(aq, seq, bt, context_lens_before=ctx, mask_mode=1 if head_dim == 128 else 0)
    dpool = G.DevPool(pool)
    dpool.upload()
    outs = []
    for bound in (None, 0):
        rc, out, _ = G.dev_attention(dpool, hb, qb, dtype, q_heads, scratch_bytes=SCRATCH, max_q_len=bound)
        assert rc == 0
        outs.append(out)
    assert outs[0].tobytes() == outs[1].tobytes()
    want = oracle.paged_attention(pool, hb, qb, dtype, q_heads, n_threads=4)
    G.assert_close(outs[0], dtype, want, what="groups of keys", scale=G.channel_scale(v, dtype, hb, q_heads))

"""Batches whose requests differ: what the kernels pay for them, as ratios of times of two batches on the same card, and the results of
the routes that only such batches take."""
import ctypes as C

import numpy as np
import pytest

import oracle
from oracle import DT_BF16, DT_F16, FMT_BF16, FMT_FP16, FMT_FP8, FMT_Q8_0, FMT_TQ4

pytestmark = pytest.mark.gpu

ROW_BYTES = {FMT_TQ4: lambda hd: 132, FMT_FP8: lambda hd: 264, FMT_Q8_0: lambda hd: 272, FMT_FP16: lambda hd: 2 * hd,
             FMT_BF16: lambda hd: 2 * hd}


class Batch:
    """One attention call over empty pages, which take as long as full ones."""

    def __init__(self, fmt, seqs, news, q_heads=16, kv_heads=2, head_dim=256, both_ways=False, block=64):
        import torch

        from warp34_amd import ffi

        dev = "cuda:0"
        self.lib = ffi.load()
        tok = ROW_BYTES[fmt](head_dim)
        pages = [(s + block - 1) // block for s in seqs]
        table = np.zeros((len(seqs), max(pages)), np.int32)
        order = np.random.default_rng(7).permutation(sum(pages)).astype(np.int32)
        at = 0
        for r, n in enumerate(pages):
            table[r, :n] = order[at:at + n]
            at += n
        starts = np.concatenate([[0], np.cumsum(news)]).astype(np.int32)
        n = int(starts[-1])
        keep = [torch.zeros(sum(pages) * kv_heads * block * tok, dtype=torch.uint8, device=dev) for _ in range(2)]
        keep += [torch.from_numpy(a).to(dev) for a in (table, starts, np.array(seqs, np.int32),
                                                       np.array(seqs, np.int32) - np.array(news, np.int32))]
        k, v, tab, qsl, seq, ctx = keep
        dtype = torch.bfloat16 if fmt == FMT_BF16 else torch.float16
        q, out = (torch.zeros((n, q_heads, head_dim), dtype=dtype, device=dev) for _ in range(2))
        strides = (kv_heads * block * tok, block * tok, tok)
        xf = oracle.XF_WHT256 if fmt == FMT_TQ4 else oracle.XF_IDENTITY
        layout = ffi.Warp34KvLayerLayout(k.data_ptr(), v.data_ptr(), *strides, *strides, 0, 0, kv_heads, head_dim, block, fmt, fmt,
                                         xf, xf, 0)
        mask = ffi.WARP34_ATTN_MASK_NONCAUSAL_WINDOW if both_ways else ffi.WARP34_ATTN_MASK_CAUSAL
        batch = ffi.Warp34AttentionBatch(qsl.data_ptr(), ctx.data_ptr(), seq.data_ptr(), tab.data_ptr(), None, None, None, len(seqs), n,
                                         table.shape[1], max(news), max(seqs), mask, 0, head_dim ** -0.5, 0)
        need = self.lib.warp34_paged_attention_scratch_bytes_for_layout(C.byref(layout), n, len(seqs), q_heads, max(seqs))
        scratch = torch.zeros(max(need, 8 << 20), dtype=torch.uint8, device=dev)
        ex = ffi.Warp34Exec(torch.cuda.current_stream().cuda_stream, scratch.data_ptr(), scratch.numel(), 0)
        self.keep = (keep, q, out, layout, batch, scratch, ex)
        call = self.lib.warp34_paged_attention_bf16 if fmt == FMT_BF16 else self.lib.warp34_paged_attention_f16
        self.args = (call, C.byref(ex), C.byref(layout), C.byref(batch), q.data_ptr(), out.data_ptr(), q_heads)

    def __call__(self):
        assert self.args[0](*self.args[1:]) == 0


def times(*batches, rounds=15, calls=10):
    """Least microseconds a call of each, measured in turn."""
    import torch

    best = [float("inf")] * len(batches)
    start, end = (torch.cuda.Event(enable_timing=True) for _ in range(2))
    for _ in range(rounds):
        for i, b in enumerate(batches):
            b()
            start.record()
            for _ in range(calls):
                b()
            end.record()
            torch.cuda.synchronize()
            best[i] = min(best[i], start.elapsed_time(end) / calls * 1e3)
    print("us a call:", ["%.1f" % t for t in best], flush=True)
    return best


@pytest.mark.parametrize("fmt", [FMT_TQ4, FMT_FP8, FMT_Q8_0, FMT_FP16, FMT_BF16])
def test_tile_of_few_rows_costs_less_than_a_whole_one(fmt):
    """Requests of 80 and of 256 query rows, one tile of 256 each: 0.75 of the time."""
    short, whole = times(Batch(fmt, [400] * 64, [40] * 64, kv_heads=8), Batch(fmt, [400] * 64, [128] * 64, kv_heads=8))
    assert short < 0.88 * whole


@pytest.mark.parametrize("fmt", [FMT_FP8, FMT_Q8_0, FMT_FP16, FMT_BF16])
def test_short_last_tiles_of_many_requests(fmt):
    """A whole tile and one of a few rows each, more requests than a wave has lanes: less than two whole tiles on every part of the chip."""
    ragged, whole = times(Batch(fmt, [1000] * 150, [33] * 150), Batch(fmt, [1000] * 150, [64] * 150))
    assert ragged < 0.94 * whole


@pytest.mark.parametrize("n,q,more", [(12, 8, 13), (9, 16, 11)])
def test_draft_blocks_in_an_odd_number_of_chunks(n, q, more):
    """Draft blocks cut into 5 (3) chunks, and more requests cut into 4 (2) of them: the tiles of a request, which read the same keys, are
    on one XCD with either number, and the time goes with the keys (0.88 and 0.75; on two XCDs 1.5 and 0.98)."""
    odd, even = times(*(Batch(FMT_BF16, [8000] * r, [q] * r, kv_heads=4, head_dim=128, both_ways=True) for r in (n, more)))
    assert odd < 0.95 * even


def test_long_draft_blocks_do_not_share_a_cu():
    """Twelve draft blocks, 384 workgroups: the long requests at the places whose workgroups would share CUs, and none of them there."""
    long, short = 12000, 2000
    apart = [long] * 4 + [short] * 4 + [short] * 4
    meet = [long] * 2 + [short] * 6 + [long] * 2 + [short] * 2
    a, b = times(*(Batch(FMT_BF16, s, [16] * 12, kv_heads=4, head_dim=128, both_ways=True) for s in (apart, meet)))
    assert max(a, b) < 1.08 * min(a, b)


@pytest.mark.parametrize("fmt", [FMT_BF16, FMT_Q8_0])
def test_one_request_of_many_tiles_uses_the_whole_chip(fmt):
    """One request with the tiles of eight: the same products (1.0; on one XCD 6)."""
    one, eight = times(Batch(fmt, [4473], [952], q_heads=8, kv_heads=1), Batch(fmt, [4473] * 8, [119] * 8, q_heads=8, kv_heads=1))
    assert one < 1.5 * eight


@pytest.mark.parametrize("fmt", [FMT_FP8, FMT_Q8_0, FMT_FP16, FMT_BF16])
def test_tiles_of_a_request_much_longer_than_the_others(fmt):
    """As many tiles as CUs, a quarter of them on eight times the keys: the long ones do not run whole (0.71 to 0.82;
    whole 0.97)."""
    mixed, long = times(Batch(fmt, [16000] + [2000] * 3, [1024] * 4), Batch(fmt, [16000] * 4, [1024] * 4))
    assert mixed < 0.9 * long


@pytest.mark.parametrize("fmt,dtype", [(FMT_TQ4, DT_F16), (FMT_Q8_0, DT_F16), (FMT_FP8, DT_F16), (FMT_BF16, DT_BF16)])
@pytest.mark.parametrize("n,q_heads,longest", [(9, 4, 128), (70, 4, 129), (66, 16, 33), (70, 16, 64)])
def test_many_short_requests(fmt, dtype, n, q_heads, longest):
    """Tiles of one row up to whole ones, one or two a request, at most and more than 64 requests."""
    from test_gpu_prefill_wide import WIDE, _run

    q_lens = [1 + (r * 37) % longest for r in range(n - 2)] + [longest, longest // 2]
    _run(fmt, dtype, 16, [q + 30 + 5 * r for r, q in enumerate(q_lens)], q_lens, 1901 + longest, q_heads=q_heads, keep=0.3,
         force=WIDE if dtype == DT_F16 else None)


@pytest.mark.parametrize("fmt", [FMT_Q8_0, FMT_FP8])
@pytest.mark.parametrize("reqs,idle", [(2, 2), (5, 5), (64, 64), (70, 64), (70, 70)])
def test_idle_requests_over_rotated_8bit_values_and_many_query_heads(fmt, reqs, idle):
    """32 query heads on one kv head, decode: the first requests (all that the plan looks at first, or all there are) masked, then without keys.
    Masked rows stay as they were, rows without keys are zero, the others are the oracle's."""
    import gpu_harness as G
    from cases import make_case

    seq = [20 + 37 * (r % 5) for r in range(reqs)]
    pool, bt, k, v, q, aq, ctx = make_case(fmt, 16, seq, [1] * reqs, 2500 + reqs, DT_F16, kv_heads=1, q_heads=32, xf=oracle.XF_WHT256)
    dpool = G.DevPool(pool)
    dpool.upload()
    live = np.arange(reqs) >= idle
    for masked in (True, False):
        lens = seq if masked else [s if on else 0 for s, on in zip(seq, live)]
        hb = oracle.HostBatch(aq, lens, bt, context_lens_before=[max(0, s - 1) for s in lens],
                              valid_req_mask=live.astype(np.uint8) if masked else None)
        want = oracle.paged_attention(pool, hb, q, DT_F16, 32)
        rc, got, _ = G.dev_attention(dpool, hb, q, DT_F16, 32, scratch_bytes=64 << 20, max_seq_len=max(seq))
        assert rc == 0
        assert (got[~live] == (0x5500 if masked else 0)).all()
        if live.any():
            full = oracle.HostBatch(aq, seq, bt, context_lens_before=ctx)
            G.assert_close(got[live], DT_F16, want[live], what="fmt=%d reqs=%d idle=%d" % (fmt, reqs, idle),
                           scale=G.channel_scale(v, DT_F16, full, 32)[live], plain_excess=4e-4)

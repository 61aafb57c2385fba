"""The running maximum of the TQ4 kernels, on rows that are made for it: every key is one row with a scale of its own, every query is that
row, so a key's score is what its scale says.  A wave of a decode kernel works on units 8, 16, ... units behind its first one."""
import numpy as np
import pytest

import oracle
from oracle import DT_F16, FMT_TQ4, XF_WHT256

pytestmark = pytest.mark.gpu

HEADS = 8  # query heads, one kv head
LOG2E = 1.4426950408889634


def _pool(block, seqs, q_lens, score, shared=0, seed=1):
    """score(position): of the keys at these positions, log2 domain; value rows of N(0, 1) numbers."""
    pages = [(s + block - 1) // block for s in seqs]
    pool = oracle.HostPool(sum(pages), 1, 256, block, FMT_TQ4, XF_WHT256)
    perm = oracle.permutation(sum(pages), seed)
    bt = np.zeros((len(seqs), max(pages)), dtype=np.int32)
    k = pool.k.reshape(-1, block, pool.tok)
    v = pool.v.reshape(-1, block, pool.tok)
    rng = np.random.default_rng(seed)
    codes = oracle.encode_row(rng.standard_normal(256).astype(np.float32))
    values = np.stack([oracle.encode_row(x) for x in rng.standard_normal((509, 256)).astype(np.float32)])
    query = oracle.f32_to_f16_bits(oracle.unrotate_row(oracle.dequant_row(codes)))
    codes.view(np.uint16)[[0, 33]] = np.float16(1.0).view(np.uint16)
    unit = 0.0625 * LOG2E * float(oracle.bits_to_f32(query, DT_F16) @ oracle.unrotate_row(oracle.dequant_row(codes)))
    at = 0
    for r, n in enumerate(pages):
        bt[r, :n] = perm[at:at + n]
        if r > 0:
            bt[r, :shared // block] = bt[0, :shared // block]
        at += n
        pos = np.arange(n * block)
        rows = np.tile(codes, (len(pos), 1))
        rows.view(np.uint16)[:, [0, 33]] = (score(pos) / unit).astype(np.float16).view(np.uint16)[:, None]
        k[bt[r, :n]] = rows.reshape(n, block, -1)
        v[bt[r, :n]] = values[(pos // 100 * 7 + 13 * r) % 509].reshape(n, block, -1)
    qsl = np.concatenate([[0], np.cumsum(q_lens)]).astype(np.int32)
    hb = oracle.HostBatch(qsl, seqs, bt, context_lens_before=[s - n for s, n in zip(seqs, q_lens)])
    return pool, hb, np.ascontiguousarray(np.broadcast_to(query, (int(qsl[-1]), HEADS, 256)))


# name: tokens and keys per request, shared keys, bound on the keys (0: exact), scratch
FORMS = {
    "decode": ((1,), (1300,), 0, 0, 0),
    "four tokens": ((4,), (1300,), 0, 0, 0),
    "balanced": ((1, 1, 1, 1), (16384, 9000, 12000, 300), 0, 0, 64 << 20),
    # two column tiles, whose eight chunks are of six units a wave
    "private rest": ((4,) * 16, (16384,) * 16, 4096, 40000, 96 << 20),
}


def _attend(pool, hb, q, form):
    import gpu_harness as G

    bound, scratch = FORMS[form][3:]
    dpool = G.DevPool(pool)
    dpool.upload()
    rc, got, _ = G.dev_attention(dpool, hb, q, DT_F16, HEADS, scratch_bytes=scratch, max_seq_len=bound or None)
    assert rc == 0
    return got


@pytest.mark.parametrize("form", ["decode", "four tokens", "private rest"])
def test_units_without_weight_before_low_scores(form):
    """The first unit of every wave has scores of minus infinity, the others -300: the keys of the former count for nothing, as with a score of -2 000."""
    import gpu_harness as G

    q_lens, seqs, shared, _, _ = FORMS[form]
    outs = []
    for none in (-2000.0, -np.inf):
        score = lambda pos: np.where((pos >= shared) & ((pos - shared) % 1536 < 256), none, -300.0 - 0.1 * (pos % 7))
        pool, hb, q = _pool(64, seqs, q_lens, score, shared)
        outs.append(_attend(pool, hb, q, form))
        if none > -np.inf:
            want = oracle.paged_attention(pool, hb, q, DT_F16, HEADS, n_threads=oracle.hw_threads())
    for got in outs:
        G.assert_close(got, DT_F16, want, what=form)


@pytest.mark.parametrize("force", [1, 2])  # tiles of 128 rows and of 256
def test_prefill_units_without_weight_before_low_scores(force):
    """The same for the tile kernels, whose waves work on all units of the request: the first two have scores of minus infinity."""
    import gpu_harness as G

    outs = []
    for none in (-2000.0, -np.inf):
        pool, hb, q = _pool(64, (400,), (200,), lambda pos: np.where(pos < 64, none, -300.0 - 0.1 * (pos % 7)))
        dpool = G.DevPool(pool)
        dpool.upload()
        rc, got, _ = G.dev_attention(dpool, hb, q, DT_F16, HEADS, force_kernel=force)
        assert rc == 0
        outs.append(got)
        if none > -np.inf:
            want = oracle.paged_attention(pool, hb, q, DT_F16, HEADS, n_threads=oracle.hw_threads())
    for got in outs:
        G.assert_close(got, DT_F16, want, what="tiles %d" % force)


@pytest.mark.parametrize("form", sorted(FORMS))
@pytest.mark.parametrize("lengths_before", [True, False])
def test_value_scales_that_leave_no_room_above_one(form, lengths_before):
    """Value scales of 3 000 in every third token and scores that rise by 6 from one unit of a wave to its next: with a maximum that stays where it
    is, as it does for ordinary scales up to a rise of 8, a weight would be 64 x 3 000, which is no fp16 number."""
    q_lens, seqs, shared, _, _ = FORMS[form]
    pool, hb, q = _pool(64, seqs, q_lens, lambda pos: 6.0 * (pos // 256 + 1), shared)
    rows = pool.v.reshape(-1, 64, pool.tok).view(np.uint16)
    assert np.shares_memory(rows, pool.v)
    rows[:, ::3, [0, 33]] = np.float16(3000.0).view(np.uint16)
    want = oracle.paged_attention(pool, hb, q, DT_F16, HEADS, n_threads=oracle.hw_threads())
    if not lengths_before:  # decode: the kernel that does not work ahead of them; a verify batch has no pass for shared keys
        hb = oracle.HostBatch(hb.qsl, hb.seq, hb.bt)
    out = oracle.bits_to_f32(_attend(pool, hb, q, form), DT_F16).astype(np.float64)
    assert np.isfinite(out).all()
    # the scores' error, 2e-3 of the largest value scale, and the output's rounding
    assert (np.abs(out - want) <= 1e-2 * np.abs(want) + 2e-3 * 3000.0).all()

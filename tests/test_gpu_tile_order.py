"""The 128-row tile kernel hands out a batch's tiles longest first.  A tile's rows do not depend on the
rest of the batch, so a batch must give, byte for byte, what each of its requests gives alone: every
tile of every request taken once, none of a masked request."""
import numpy as np
import pytest

import oracle
from cases import make_case
from oracle import DT_F16, FMT_FP16, FMT_Q8_0, FMT_TQ4

pytestmark = pytest.mark.gpu

TILE_KERNEL = 2  # the test selector's value


def _batch_equals_requests(fmt, seq, q_lens, masked=()):
    import gpu_harness as G

    pool, bt, _, _, q, aq, ctx = make_case(fmt, 16, seq, q_lens, 511, DT_F16, q_heads=16)
    dpool = G.DevPool(pool)
    dpool.upload()

    def run(qsl, seqs, tables, before, rows, mask=None):
        hb = oracle.HostBatch(qsl, seqs, tables, context_lens_before=before, valid_req_mask=mask)
        rc, got, _ = G.dev_attention(dpool, hb, rows, DT_F16, 16, force_kernel=TILE_KERNEL)
        assert rc == 0
        return got

    mask = None if not masked else np.array([0 if r in masked else 1 for r in range(len(seq))], dtype=np.uint8)
    got = run(aq, seq, bt, ctx, q, mask)
    for r in range(len(seq)):
        rows = slice(aq[r], aq[r + 1])
        if r in masked:
            assert (got[rows].view(np.uint16) == 0x5500).all()
        elif q_lens[r]:
            alone = run([0, q_lens[r]], [seq[r]], bt[r:r + 1], [ctx[r]], q[rows])
            assert got[rows].tobytes() == alone.tobytes(), "request %d" % r


@pytest.mark.parametrize("fmt", [FMT_TQ4, FMT_Q8_0, FMT_FP16])
@pytest.mark.parametrize("seq,q", [
    ([455, 738, 514, 33], [365, 722, 514, 33]),  # no context, tiles of equal length, a last one of one token
    ([640, 640, 640, 640], [448, 448, 448, 448]),  # all tiles of a rank alike
    ([1500, 40, 1100], [1300, 1, 700]),  # a decode token between prompts
])
def test_ragged_batches(fmt, seq, q):
    _batch_equals_requests(fmt, seq, q)


def test_masked_requests():
    _batch_equals_requests(FMT_TQ4, [300, 200, 400, 90], [200, 200, 150, 60], masked=(0, 2))


@pytest.mark.parametrize("n", [63, 64, 65])
def test_number_of_requests(n):
    """One request per lane up to 64, grid order beyond."""
    q = [32 + (7 * i) % 23 for i in range(n)]
    _batch_equals_requests(FMT_TQ4, [x + 5 * (i % 9) for i, x in enumerate(q)], q)

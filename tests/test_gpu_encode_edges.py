"""TQ4 codes around every boundary of the code book and past its ends, rows at the ends of the energy
range, and the Q/K producer on both sides of the number of tokens from which it gives a token one
workgroup: byte for byte against the oracle."""
import numpy as np
import pytest

import oracle
from oracle import DT_BF16, DT_F16, FMT_Q8_0, FMT_TQ4, XF_IDENTITY, XF_WHT256

pytestmark = pytest.mark.gpu


def _append_equals_oracle(rows, dtype, xf):
    import gpu_harness as G

    n = rows.shape[0]
    pages = (n + 63) // 64
    bits = (oracle.f32_to_bf16_bits if dtype == DT_BF16 else oracle.f32_to_f16_bits)(rows.reshape(n, 1, 256))
    v = bits[::-1].copy()
    pool = oracle.HostPool(pages, 1, 256, 64, FMT_TQ4, xf)
    bt = np.arange(pages, dtype=np.int32).reshape(1, -1)
    hb = oracle.HostBatch([0, n], [n], bt, context_lens_before=[0],
                          write_slot_mapping=oracle.slot_mapping(bt[0], 0, n, 64))
    oracle.kv_cache_write(pool, hb, bits, v, dtype)
    dev = G.DevPool(pool)
    assert G.dev_write(dev, hb, bits, v, dtype) == 0
    gk, gv = dev.download()
    assert gk.tobytes() == pool.k.tobytes() and gv.tobytes() == pool.v.tobytes()


def _boundary_rows(half_energy):
    """Rows whose normalised values (energy `half_energy` in each half) lie on both sides of the boundaries, up to 2^-9
    from them, each row at another scale; and rows that reach past the ends of the code book, up to a single
    element that holds all of the energy."""
    rng = np.random.default_rng(5)
    b = oracle.boundaries().astype(np.float64)
    rows = np.zeros((192, 2, 128))
    for r in range(160):
        near = b[rng.integers(0, 15, (2, 24))] * (1.0 + rng.integers(-4, 5, (2, 24)) * 2.0 ** -11)
        rest = half_energy - np.sum(near ** 2, axis=1, keepdims=True)
        rows[r, :, :24] = near
        rows[r, :, 24:] = np.sqrt(np.maximum(rest, 0.0) / 104) * rng.choice([-1.0, 1.0], (2, 104))
        rows[r] = rng.permuted(rows[r], axis=1) * 2.0 ** rng.integers(-6, 7)
    for r in range(160, 192):
        rows[r, :, (r * 37) % 128] = (-1.0) ** r * 2.0 ** (r % 9)
        if r % 3 == 0:
            rows[r] += np.linspace(-0.25, 0.25, 128)
    return rows.reshape(192, 256).astype(np.float32)


@pytest.mark.parametrize("dtype", [DT_BF16, DT_F16])
@pytest.mark.parametrize("xf", [XF_IDENTITY, XF_WHT256])
def test_codes_around_every_boundary(dtype, xf):
    rows = _boundary_rows(0.5 if xf == XF_IDENTITY else 0.25)
    if xf == XF_WHT256:  # the rows that the sign diagonal and the rotation bring there (both are their own inverse)
        rows = np.stack([oracle.signs() * oracle.wht256(r) for r in rows])
    _append_equals_oracle(rows, dtype, xf)


@pytest.mark.parametrize("xf", [XF_IDENTITY, XF_WHT256])
def test_rows_at_the_ends_of_the_energy_range(xf):
    """Energies around the 1e-20 below which a row has no codes, and bf16 rows up to the largest finite energy."""
    rng = np.random.default_rng(7)
    rows = [rng.standard_normal(256) * 10.0 ** e for e in (-18, -12, -11.5, -11.2, -11, -10.8, -10, 0, 10, 17, 17.5)]
    spike = np.zeros(256)
    spike[3] = 1e-10
    rows += [spike, -spike, 1.0000001 * spike, spike * 1.5, np.full(256, 6.25e-12), np.full(256, 1e17)]
    _append_equals_oracle(np.stack(rows).astype(np.float32), DT_BF16, xf)


@pytest.mark.parametrize("n,qh,kh", [(1, 16, 2), (2, 1, 1), (3, 5, 3), (255, 6, 1), (256, 3, 2), (257, 3, 2), (258, 6, 1),
                                     (512, 3, 2), (513, 6, 1)])
@pytest.mark.parametrize("fmt", [FMT_TQ4, FMT_Q8_0])
def test_producer_on_both_sides_of_the_token_limit(n, qh, kh, fmt):
    import gpu_harness as G
    from test_gpu_fused_qk_norm import EPS, MROPE, THETA, _dev_fused_write, _inputs, _positions

    hd, rot, bs = 256, 64, 64
    qg, k, qw, kw = _inputs(n, qh, kh, hd, 61)
    k[0, :] = 0  # mean = eps
    v = oracle.fill_normal(n * kh * hd, 65, DT_F16).reshape(n, kh * hd)
    pos = _positions(n, 66)
    pages = (n + bs - 1) // bs
    bt = np.arange(pages, dtype=np.int32)[::-1].copy()
    slots = oracle.slot_mapping(bt, 0, n, bs)
    mask = np.ones(n, np.uint8)
    mask[n // 2 + 1:n // 2 + 2] = 0
    fill = 0x7E7E
    want_q, want_k, want_g = oracle.fused_qk_rmsnorm_rope_gate_f16(
        qg, k, qw, kw, pos, qh, kh, hd, rot, MROPE, THETA, EPS, valid_token_mask=mask,
        q_out=np.full((n, qh, hd), fill, np.uint16), k_out=np.full((n, kh, hd), fill, np.uint16),
        gate_out=np.full((n, qh, hd), fill, np.uint16))
    pool = oracle.HostPool(pages, kh, hd, bs, fmt, XF_WHT256)
    pool.k[:], pool.v[:] = 0x7E, 0x7E
    hb = oracle.HostBatch([0, n], [n], bt.reshape(1, -1), context_lens_before=[0], write_slot_mapping=slots,
                          valid_token_mask=mask)
    oracle.kv_cache_write(pool, hb, want_k.reshape(n, kh * hd), v, DT_F16, kh * hd, kh * hd)
    dev = G.DevPool(pool, fill=0x7E)
    rc, (q, ko, g) = _dev_fused_write(dev, qg, k, v, qw, kw, pos, slots, qh, kh, hd, rot, mask=mask)
    assert rc == 0
    assert q.tobytes() == want_q.tobytes() and ko.tobytes() == want_k.tobytes() and g.tobytes() == want_g.tobytes()
    gk, gv = dev.download()
    assert gk.tobytes() == pool.k.tobytes() and gv.tobytes() == pool.v.tobytes()


def test_rows_on_both_sides_of_the_short_transform():
    """Rows whose sum of squares sends a wave to the exact transform beside rows that stay on the short one: energies around 1e-15 / 256 and
    around the largest finite sum of 16-fold values, zeros, subnormal elements, single elements."""
    rng = np.random.default_rng(11)
    rows = [rng.standard_normal(256) * 10.0 ** e for e in np.concatenate([np.arange(-10.6, -9.2, 0.05), np.arange(16.4, 18.4, 0.1)])]
    for e in (-38, -30, -20, 0):
        row = rng.standard_normal(256)
        row[rng.permutation(256)[:200]] *= 10.0 ** e
        rows += [row, np.where(np.arange(256) < 128, row, 0.0)]
    for i in range(16):
        spike = np.zeros(256)
        spike[17 * i] = 2.0 ** (i - 8)
        rows.append(spike)
    rows.append(np.zeros(256))
    _append_equals_oracle(rng.permutation(np.stack(rows)).astype(np.float32), DT_BF16, XF_WHT256)

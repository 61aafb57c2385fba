"""Performance cases of the KV-cache path: what a serving engine has the library do, through the C ABI.

A case is a dict of plain values; its "kind" says which calls one pass makes:

  step       the target model's layers of one engine step, layer after layer: Gemma RMSNorm + mRoPE + gate split fused with
             the append of the new tokens, then gated paged attention over prefix + new tokens (fp16 activations)
  attention  paged attention alone, bf16 activations
  chunk      append of a bf16 chunk, then causal attention over prefix + chunk (bf16 activations)
  append     quantize-on-append of bf16 rows alone
  producer   the fused producer of `step` alone, over a prefill chunk
  qsa        sparse attention: each query token over its own list of selected 4-token groups
  draft      the draft model's layers: RMSNorm + RoPE fused with the append, then attention in which the tokens of a
             draft block see each other both ways (bf16 rows and pages, head dimension 128)

A pass goes through `layers` layers, each with pages and activations of its own, as a model's step does: a layer's pages are
not in the caches any more when its turn comes again.  Context lengths are drawn uniformly from [ctx_min, ctx_max] and the
numbers of new tokens from [q_min, q_max] by a generator seeded with "lens", so they belong to the case; the values, the
page order and the selected groups come from the seed.
"""
import ctypes as C
import math
import random

import torch

from warp34_amd import ffi

DEV = "cuda:0"
FORMATS = {"fp16": ffi.WARP34_KV_FORMAT_FP16, "bf16": ffi.WARP34_KV_FORMAT_BF16, "tq4": ffi.WARP34_KV_FORMAT_TQ4,
           "q8_0": ffi.WARP34_KV_FORMAT_Q8_0, "fp8": ffi.WARP34_KV_FORMAT_FP8_E4M3}
ROTARY_DIM, MROPE, ROPE_THETA, RMS_EPS = 64, (11, 11, 10), 1.0e7, 1.0e-6


def row_bytes(fmt, head_dim):
    return {"fp16": 2 * head_dim, "bf16": 2 * head_dim, "tq4": 66 * head_dim // 128, "q8_0": 68 * head_dim // 64,
            "fp8": 264 * head_dim // 256}[fmt]


def _case(kind, fmt, requests, ctx_min, ctx_max, q_min, q_max, layers, *, block=64, q_heads=16, kv_heads=2, head_dim=256,
          shared=0, groups=0, lens=1):
    return {"kind": kind, "fmt": fmt, "requests": requests, "ctx_min": ctx_min, "ctx_max": ctx_max, "q_min": q_min,
            "q_max": q_max, "layers": layers, "block": block, "q_heads": q_heads, "kv_heads": kv_heads, "head_dim": head_dim,
            "shared": shared, "groups": groups, "lens": lens}


def listed():
    named = [
        # one user, a short chat, a model of eight full-attention layers: nothing but latency and launches
        ("step_tq4_1x1200", _case("step", "tq4", 1, 1200, 1200, 1, 1, 8, block=16)),
        # one user at 128K context
        ("decode_tq4_1x131072", _case("attention", "tq4", 1, 131072, 131072, 1, 1, 4)),
        # a full decode batch of users with contexts of any length
        ("step_tq4_32x1k_64k", _case("step", "tq4", 32, 1024, 65536, 1, 1, 1)),
        # unquantised pages, one long document
        ("decode_bf16_1x32768", _case("attention", "bf16", 1, 32768, 32768, 1, 1, 4)),
        # a few users, one token and three drafted ones verified, over the 8-bit pages the policy keeps for the last layers
        ("step_q8_0_5x4_3k_21k", _case("step", "q8_0", 5, 3000, 21000, 4, 4, 4, block=16)),
        # verification over a long prefix (a repository, a book) that all requests share
        ("verify_tq4_16x4_262144", _case("attention", "tq4", 16, 262144, 262144, 4, 4, 1, shared=200000)),
        # chunked prefill in full swing
        ("chunk_tq4_8x2048_16384", _case("chunk", "tq4", 8, 18432, 18432, 2048, 2048, 1)),
        # prompts and follow-up turns of odd lengths
        ("step_q8_0_3x200_1900", _case("step", "q8_0", 3, 1900, 7000, 200, 1900, 2, block=16)),
        # the producer of a long prefill chunk
        ("producer_tq4_8192", _case("producer", "tq4", 1, 8192, 8192, 8192, 8192, 1)),
        # the append alone
        ("append_tq4_4096", _case("append", "tq4", 1, 4096, 4096, 4096, 4096, 4)),
        # sparse attention of a small decode batch over a long context
        ("qsa_tq4_16x513", _case("qsa", "tq4", 1, 131072, 131072, 16, 16, 2, groups=513)),
        # four users' draft blocks of sixteen tokens
        ("draft_bf16_4x16_1k_9k", _case("draft", "bf16", 4, 1000, 9000, 16, 16, 5, block=16, kv_heads=4, head_dim=128)),
    ]
    return [dict(c, name=n) for n, c in named]


def _log_int(rng, lo, hi):
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    """A case of the ranges the listed ones stand for; never more bytes or operations than the largest of those."""
    kind = rng.choice(["step"] * 4 + ["attention"] * 4 + ["chunk"] * 2 + ["prefill", "append", "producer", "qsa", "draft"])
    lens = rng.randrange(1 << 20)
    block = rng.choice([16, 64, 64, 128])
    q_heads, kv_heads = rng.choice([(16, 2), (16, 2), (8, 1), (8, 2), (32, 4)])
    while True:
        if kind in ("step", "attention"):
            fmt = rng.choice(["tq4"] * 4 + ["q8_0", "fp8", "fp16" if kind == "step" else "bf16"])
            ctx_max = _log_int(rng, 300, 131072)
            q = rng.choice([1, 1, 1, 2, 4])
            c = _case(kind, fmt, _log_int(rng, 1, 32), max(32, int(ctx_max * rng.uniform(0.02, 1.0))), ctx_max, q, q, 1,
                      block=block, q_heads=q_heads, kv_heads=kv_heads, lens=lens)
        elif kind in ("chunk", "prefill"):
            fmt = rng.choice(["tq4", "tq4", "q8_0", "fp8", "fp16" if kind == "prefill" else "bf16"])
            q_max = _log_int(rng, 40, 2048)
            c = _case("step" if kind == "prefill" else kind, fmt, _log_int(rng, 1, 8), q_max, q_max + rng.randrange(16384),
                      max(17, int(q_max * rng.uniform(0.2, 1.0))), q_max, 1, block=block, q_heads=q_heads, kv_heads=kv_heads,
                      lens=lens)
        elif kind in ("append", "producer"):
            n = _log_int(rng, 1, 8192)
            c = _case(kind, rng.choice(["tq4", "tq4", "q8_0", "fp8", "bf16" if kind == "append" else "fp16"]), 1, n, n, n, n, 1,
                      block=block, q_heads=q_heads, kv_heads=kv_heads, lens=lens)
        elif kind == "qsa":
            groups, n = _log_int(rng, 16, 513), _log_int(rng, 1, 64)
            ctx = _log_int(rng, 4 * groups + 64, 131072)
            c = _case(kind, rng.choice(["tq4", "tq4", "fp8", "q8_0"]), 1, ctx, ctx, n, n, 1, block=block, groups=groups,
                      lens=lens)
        else:
            ctx_max = _log_int(rng, 300, 16384)
            q = rng.choice([8, 16])
            c = _case(kind, "bf16", _log_int(rng, 1, 16), max(32, ctx_max // 8), ctx_max, q, q, 1, block=16, q_heads=16,
                      kv_heads=4, head_dim=128, lens=lens)
        w = work(c)
        if w["bytes"] > 5.0e8 or w["flops"] > 2.0e12:
            continue
        # several layers where one is little work
        c["layers"] = max(1, min(8, int(6.0e7 / max(w["bytes"], w["flops"] / 300))))
        return c


def _lengths(case):
    """Per request: tokens after the step, new tokens."""
    rng = random.Random(case["lens"])
    seqs, news = [], []
    for _ in range(case["requests"]):
        s = rng.randint(case["ctx_min"], case["ctx_max"])
        seqs.append(s)
        news.append(min(rng.randint(case["q_min"], case["q_max"]), s))
    return seqs, news


def _normal(gen, shape, dtype, scale=1.0, shift=0.0):
    return (torch.randn(shape, generator=gen, device=DEV, dtype=torch.float32) * scale + shift).to(dtype)


def _kv_rows(gen, case, n):
    """K or V rows: N(0, 1) with three channels of every head twenty times as large, as real caches show them."""
    kvh, hd = case["kv_heads"], case["head_dim"]
    rows = torch.randn((n, kvh, hd), generator=gen, device=DEV, dtype=torch.float32)
    rows[:, :, [7, hd // 2 + 13, hd - 30]] *= 20.0
    return rows.to(torch.float16 if case["fmt"] == "fp16" else torch.bfloat16).reshape(n, kvh * hd)


class _Layer:
    """One layer's pages, filled through the append entry point, and the descriptors of its step."""

    def __init__(self, case, gen, lib, stream, seqs, news, fill):
        kvh, hd, bs, fmt = case["kv_heads"], case["head_dim"], case["block"], case["fmt"]
        tok = row_bytes(fmt, hd)
        pages_per = [(s + bs - 1) // bs for s in seqs]
        mb, shared = max(pages_per), case["shared"] // bs
        pool = sum(pages_per) - shared * (len(seqs) - 1) + 3
        order = torch.randperm(pool, generator=gen, device=DEV).to(torch.int32)
        self.block_tables = torch.zeros((len(seqs), mb), dtype=torch.int32, device=DEV)
        at = 0
        for r, n in enumerate(pages_per):
            own = shared if r else 0
            if own:
                self.block_tables[r, :own] = self.block_tables[0, :own]
            self.block_tables[r, own:n] = order[at:at + n - own]
            at += n - own
        self.k = torch.zeros(pool * kvh * bs * tok, dtype=torch.uint8, device=DEV)
        self.v = torch.zeros_like(self.k)
        xf = ffi.WARP34_KV_TRANSFORM_RADEMACHER_WHT256 if fmt == "tq4" else ffi.WARP34_KV_TRANSFORM_IDENTITY
        strides = (kvh * bs * tok, bs * tok, tok)
        self.layout = ffi.Warp34KvLayerLayout(self.k.data_ptr(), self.v.data_ptr(), *strides, *strides, 0, 0, kvh, hd, bs,
                                              FORMATS[fmt], FORMATS[fmt], xf, xf, 0)
        slots, new_slots, positions = [], [], []
        for r, (s, n) in enumerate(zip(seqs, news)):
            pos = torch.arange(s, device=DEV)
            slot = (self.block_tables[r][pos // bs] * bs + pos % bs).to(torch.int32)
            new_slots.append(slot[s - n:])
            positions.append(pos[s - n:])
            slots.append(slot[shared * bs if r else 0:])
        self.slots = torch.cat(new_slots)
        self.positions = torch.cat(positions).to(torch.int32)
        starts = [0]
        for n in news:
            starts.append(starts[-1] + n)
        self.qsl = torch.tensor(starts, dtype=torch.int32, device=DEV)
        self.seq = torch.tensor(seqs, dtype=torch.int32, device=DEV)
        self.ctx = torch.tensor([s - n for s, n in zip(seqs, news)], dtype=torch.int32, device=DEV)
        mask = ffi.WARP34_ATTN_MASK_NONCAUSAL_WINDOW if case["kind"] == "draft" else ffi.WARP34_ATTN_MASK_CAUSAL
        self.batch = ffi.Warp34AttentionBatch(
            self.qsl.data_ptr(), self.ctx.data_ptr(), self.seq.data_ptr(), self.block_tables.data_ptr(), self.slots.data_ptr(),
            None, None, len(seqs), starts[-1], mb, max(news), max(seqs), mask, 0, hd ** -0.5, 0)
        if fill:
            write = lib.warp34_kv_cache_write if fmt == "fp16" else lib.warp34_kv_cache_write_bf16
            ex = ffi.Warp34Exec(stream, 0, 0, 0)
            for part in torch.cat(slots).split(65536):
                n = part.numel()
                k, v = _kv_rows(gen, case, n), _kv_rows(gen, case, n)
                ends = torch.tensor([0, n], dtype=torch.int32, device=DEV)
                b = ffi.Warp34AttentionBatch(ends.data_ptr(), None, ends[1:].data_ptr(), self.block_tables.data_ptr(),
                                             part.data_ptr(), None, None, 1, n, mb, n, n, 0, 0, 1.0, 0)
                ffi.check_rc(write(C.byref(ex), C.byref(self.layout), C.byref(b), k.data_ptr(), v.data_ptr()), "append")


class _State:
    """calls: [(function, arguments)] of one pass in order; outputs: what they write."""

    def __init__(self):
        self.calls, self.outputs, self.keep = [], [], []


def prepare(case, seed):
    lib = ffi.load()
    gen = torch.Generator(device=DEV)
    gen.manual_seed(seed)
    stream = torch.cuda.current_stream().cuda_stream
    kind, fmt = case["kind"], case["fmt"]
    qh, kvh, hd = case["q_heads"], case["kv_heads"], case["head_dim"]
    seqs, news = _lengths(case)
    if kind == "qsa":
        n, news = case["q_max"], [1]
    else:
        n = sum(news)
    st = _State()
    # one workspace for all layers, as an engine keeps it
    scratch = None
    for _ in range(case["layers"]):
        layer = _Layer(case, gen, lib, stream, seqs, news, fill=kind not in ("append", "producer"))
        if scratch is None:
            need = lib.warp34_paged_attention_scratch_bytes_for_layout(C.byref(layer.layout), n, len(seqs), qh, max(seqs))
            scratch = torch.zeros(max(need, 8 << 20), dtype=torch.uint8, device=DEV)
            ex = C.pointer(ffi.Warp34Exec(stream, scratch.data_ptr(), scratch.numel(), 0))
        lay, bat = C.pointer(layer.layout), C.pointer(layer.batch)
        keep, outs = [layer], []
        if kind in ("step", "producer"):
            qg, kv = qh * 2 * hd, kvh * hd
            row = qg + 2 * kv
            proj = _normal(gen, (n, row), torch.float16)
            qw, kw = (_normal(gen, (hd,), torch.float16, 0.1) for _ in range(2))
            pos = layer.positions.repeat(3, 1).contiguous()
            q, gate = (torch.empty((n, qh, hd), dtype=torch.float16, device=DEV) for _ in range(2))
            at = proj.data_ptr()
            st.calls.append((lib.warp34_fused_qk_rmsnorm_rope_gate_kv_write_f16, (
                ex, at, at + 2 * qg, at + 2 * (qg + kv), qw.data_ptr(), kw.data_ptr(), pos.data_ptr(), None, q.data_ptr(), None,
                gate.data_ptr(), lay, layer.slots.data_ptr(), n, n, qh, kvh, hd, ROTARY_DIM, *MROPE, row, row, row, ROPE_THETA,
                RMS_EPS)))
            keep += [proj, qw, kw, pos]
            outs += [q, gate, layer.k, layer.v]
        if kind == "step":
            out = torch.zeros((n, qh, hd), dtype=torch.float16, device=DEV)
            st.calls.append((lib.warp34_paged_attention_gated_f16, (ex, lay, bat, q.data_ptr(), gate.data_ptr(), out.data_ptr(),
                                                                    qh)))
            outs.append(out)
        if kind in ("append", "chunk"):
            k, v = (_normal(gen, (n, kvh * hd), torch.bfloat16) for _ in range(2))
            st.calls.append((lib.warp34_kv_cache_write_bf16, (ex, lay, bat, k.data_ptr(), v.data_ptr())))
            keep += [k, v]
            outs += [layer.k, layer.v]
        if kind in ("attention", "chunk"):
            q = _normal(gen, (n, qh, hd), torch.bfloat16)
            out = torch.zeros_like(q)
            st.calls.append((lib.warp34_paged_attention_bf16, (ex, lay, bat, q.data_ptr(), out.data_ptr(), qh)))
            keep.append(q)
            outs.append(out)
        if kind == "qsa":
            total, take, per_page = (seqs[0] + 3) // 4, case["groups"], case["block"] // 4
            # the newest group is always selected
            logical = torch.stack([torch.randperm(total - 1, generator=gen, device=DEV)[:take] for _ in range(n)])
            logical[:, -1] = total - 1
            physical = layer.block_tables[0][logical // per_page] * per_page + logical % per_page
            logical, physical = (t.to(torch.int32).contiguous() for t in (logical, physical))
            count = torch.full((n,), take, dtype=torch.int32, device=DEV)
            last = torch.full((n,), seqs[0] - 1, dtype=torch.int32, device=DEV)
            q, gate = (_normal(gen, (n, qh, hd), torch.float16) for _ in range(2))
            out = torch.zeros_like(q)
            st.calls.append((lib.warp34_qsa_sparse_paged_attn_f16, (
                ex, q.data_ptr(), gate.data_ptr(), lay, physical.data_ptr(), logical.data_ptr(), count.data_ptr(),
                last.data_ptr(), None, out.data_ptr(), n, qh, take, hd ** -0.5)))
            keep += [logical, physical, count, last, q, gate]
            outs.append(out)
        if kind == "draft":
            qkv = _normal(gen, (n, (qh + 2 * kvh) * hd), torch.bfloat16)
            qw, kw = (_normal(gen, (hd,), torch.bfloat16, 0.1, 1.0) for _ in range(2))
            angle = torch.arange(max(seqs), device=DEV)[:, None] * (
                1.0e4 ** (-torch.arange(hd // 2, device=DEV) / (hd // 2)))[None, :]
            table = torch.cat([torch.cos(angle), torch.sin(angle)], dim=1).float().contiguous()
            q, out = (torch.empty((n, qh, hd), dtype=torch.bfloat16, device=DEV) for _ in range(2))
            st.calls.append((lib.warp34_dflash_qk_norm_rope_kv_write_bf16_f32_table, (
                ex, qkv.data_ptr(), q.data_ptr(), layer.positions.data_ptr(), qw.data_ptr(), kw.data_ptr(), table.data_ptr(),
                lay, layer.slots.data_ptr(), n, qh, kvh, hd, max(seqs), RMS_EPS)))
            st.calls.append((lib.warp34_paged_attention_bf16, (ex, lay, bat, q.data_ptr(), out.data_ptr(), qh)))
            keep += [qkv, qw, kw, table]
            outs += [q, layer.k, layer.v, out]
        st.keep.append(keep)
        st.outputs.append(outs)
    st.keep += [scratch, ex]
    return st


def run(state):
    for call, args in state.calls:
        rc = call(*args)
        if rc:
            raise ffi.Warp34Error(rc, call.__name__)
    return state.outputs


def work(case):
    kind, qh, kvh, hd = case["kind"], case["q_heads"], case["kv_heads"], case["head_dim"]
    kv_row = 2 * kvh * row_bytes(case["fmt"], hd)  # K and V of one token
    seqs, news = _lengths(case)
    n = sum(news)
    flops = bytes_ = 0.0
    if kind == "qsa":
        n, total, take = case["q_max"], (seqs[0] + 3) // 4, case["groups"]
        touched = total * (1.0 - (1.0 - take / total) ** n)  # groups that at least one token selects
        bytes_ = 4 * touched * kv_row + n * qh * hd * 2 * 3 + n * take * 8
        flops = 4.0 * hd * qh * n * take * 4
    else:
        pairs = keys = 0.0
        for r, (s, q) in enumerate(zip(seqs, news)):
            pairs += float(q) * s if kind == "draft" else float(q) * (s - q) + q * (q + 1) / 2
            keys += s - (case["shared"] // case["block"] * case["block"] if r else 0)
        if kind not in ("append", "producer"):
            bytes_ += keys * kv_row + n * qh * hd * 2 * 2  # pages, queries, output
            flops += 4.0 * hd * qh * pairs
        if kind in ("append", "chunk"):
            bytes_ += n * (2 * kvh * hd * 2 + kv_row + 4)
        if kind in ("step", "producer"):
            # projection rows; queries and gates written; encoded rows (a step's attention has counted those and its queries)
            bytes_ += n * ((2 * qh + 2 * kvh) * hd * 2 + qh * hd * 2 + 16)
            bytes_ += n * (qh * hd * 2 + kv_row) if kind == "producer" else 0
        if kind == "draft":
            bytes_ += n * ((qh + 2 * kvh) * hd * 2 + hd * 4 + 8)
    return {"bytes": bytes_ * case["layers"], "flops": flops * case["layers"]}


def tolerance(case):
    """Encoded pages are bytes and stay the same.  Attention multiplies 16-bit operands and rounds its result to 16 bits."""
    if case["kind"] == "append":
        return "exact"
    if case["kind"] == "producer":
        return {"rel": 5e-4, "max": 4e-3}  # fp16 rows, computed in fp32
    return {"rel": 1e-2, "max": 0.1} if case["kind"] in ("attention", "chunk", "draft") else {"rel": 4e-3, "max": 0.05}

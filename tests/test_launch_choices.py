"""Which kernels the attention entry points launch, and with which numbers of chunks and shares, on the CPU: the library's host code runs over a
recorder in the place of the HIP runtime, in a child process."""
import json
import os
import re
import subprocess
import sys

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CHILD = """
import ctypes as C, json, re, sys
rec = C.CDLL(sys.argv[1], mode=C.RTLD_GLOBAL)  # before the library: its symbols are the ones that are found
rec.rec_name.restype = C.c_char_p
from warp34_amd import ffi
lib = ffi.load()
FMT = {"tq4": 2, "q8_0": 3, "fp8": 4, "bf16": 1}
out = []
for c in json.load(open(sys.argv[2])):
    kvh, hd, bs = c["kv_heads"], c["head_dim"], 64
    tok = {"tq4": 66 * hd // 128, "q8_0": 272, "fp8": 264, "bf16": 2 * hd}[c["fmt"]]
    strides = (kvh * bs * tok, bs * tok, tok)
    f, xf = FMT[c["fmt"]], c["xf"]
    L = ffi.Warp34KvLayerLayout(1 << 20, 1 << 30, *strides, *strides, 0, 0, kvh, hd, bs, f, f, xf, xf, 0)
    n = c["reqs"] * c["q_len"]
    B = ffi.Warp34AttentionBatch(4096, 4096, 4096, 4096, 4096, None, None, c["reqs"], n, (c["max_seq"] + bs - 1) // bs, c["q_len"], c["max_seq"],
                                 0, 0, 0.0625, 0)
    need = lib.warp34_paged_attention_scratch_bytes_for_layout(C.byref(L), n, c["reqs"], c["q_heads"], c["max_seq"])
    runs = []
    for scratch in c["scratch"]:
        rec.rec_clear()
        ex = ffi.Warp34Exec(0, 1 << 40, need if scratch == "queried" else scratch, 0)
        assert lib.warp34_paged_attention_bf16(C.byref(ex), C.byref(L), C.byref(B), 4096, 4096, c["q_heads"]) == 0
        run = []
        for i in range(rec.rec_count()):
            shape, choice = (C.c_uint32 * 5)(), (C.c_int * 6)()
            rec.rec_shape(i, shape)
            rec.rec_choice(i, choice)
            run.append([rec.rec_name(i).decode(), list(shape), list(choice)])
        runs.append(run)
    out.append([need, runs])
print(json.dumps(out))
"""


@pytest.fixture(scope="module")
def recorder(tmp_path_factory):
    tmp = str(tmp_path_factory.mktemp("recorder"))
    with open(os.path.join(ROOT, "warp34_amd", "csrc", "paged_attn.hip")) as f:
        block = re.search(r"^struct AttnParams \{.*?^\};", f.read(), re.M | re.S).group(0)
    with open(os.path.join(tmp, "attn_params.inc"), "w") as f:
        f.write(block)
    so = os.path.join(tmp, "launch_recorder.so")
    subprocess.run(["g++", "-std=c++17", "-O1", "-shared", "-fPIC", "-I", os.path.join(ROOT, "include"), "-I", tmp, "-o", so,
                    os.path.join(ROOT, "tests", "host", "launch_recorder.cpp")], check=True)

    def launches(cases):
        path = os.path.join(tmp, "cases.json")
        with open(path, "w") as f:
            json.dump(cases, f)
        p = subprocess.run([sys.executable, "-c", CHILD, so, path], cwd=ROOT, stdout=subprocess.PIPE, stderr=subprocess.PIPE, text=True)
        assert p.returncode == 0, p.stderr
        return json.loads(p.stdout)

    return launches


def case(fmt, reqs, q_len, max_seq, q_heads=16, kv_heads=2, head_dim=256, xf=None, scratch=(64 << 20,)):
    return dict(fmt=fmt, reqs=reqs, q_len=q_len, max_seq=max_seq, q_heads=q_heads, kv_heads=kv_heads, head_dim=head_dim,
                xf=(1 if fmt == "tq4" else 0) if xf is None else xf, scratch=list(scratch))


def test_kernels_of_the_plan_get_the_numbers_that_they_read(recorder):
    """Kernels that leave a short batch to its own plan (two column tiles; rotated 8-bit values without streaming loads) get a line below every batch
    or the tiles that go with it; the others the chunk grid's cap, from which no batch has more chunks than workgroups."""
    cases = [case(fmt, reqs, q_len, max_seq, q_heads, kv_heads, xf=xf)
             for fmt, xf in (("q8_0", 0), ("q8_0", 1), ("fp8", 1), ("bf16", 0), ("tq4", 1))
             for q_heads, kv_heads in ((16, 2), (8, 1), (32, 1), (48, 2), (40, 1), (4, 4))
             for reqs, q_len in ((2, 1), (7, 1), (64, 1), (65, 1), (100, 1), (2, 2), (5, 4), (20, 4), (3, 16))
             for max_seq in (200, 4000, 131072)]
    seen = set()
    for c, (_, (run,)) in zip(cases, recorder(cases)):
        for name, (grid, *_), (_, grid_chunks, short_units, short_tiles, short_tok_tile, q_subgroups) in run:
            if "balanced_kernel" not in name:
                continue
            short = False
            if "rows" in name:
                nt, vres, stream = re.search(r"Li(\d)ELi\d+ELb(\d)ELb(\d)E", name).groups()
                short = nt == "2" or (vres == "1" and stream == "0")
            seen.add((short, q_subgroups > 1))
            if short:
                assert short_units == -1 or (short_units > 0 and short_tok_tile > 0 and 0 < short_tiles * c["reqs"] <= 128), (c, name)
            else:
                assert grid_chunks == 0 or (q_subgroups == 1 and 1 < grid_chunks and grid_chunks * c["reqs"] <= grid), (c, name)
    assert len(seen) == 4


def test_short_decode_batches_on_the_grid_keep_the_chunks_of_the_plan(recorder):
    """Up to 16 requests a batch runs on the chunk grid only where the cap leaves the longest request chunks of eight units, the plan's least; with more
    requests up to 3 072 units (row formats: 2 048) for all of them at the longest one's length."""
    units = (1, 8, 40, 42, 43, 48, 49, 62, 63, 64, 65, 72, 73, 80, 81, 120, 121, 180, 181, 256, 257, 512, 513, 1024)
    cases = [case(fmt, reqs, 1, 32 * u, xf=xf) for fmt, xf in (("tq4", 1), ("q8_0", 0), ("fp8", 1), ("bf16", 0))
             for reqs in (2, 4, 12, 13, 14, 16, 17, 33, 48, 64, 65) for u in units]
    for c, (_, (run,)) in zip(cases, recorder(cases)):
        u = c["max_seq"] // 32
        if c["reqs"] <= 16:
            grid = u <= 8 * (128 // c["reqs"])
        else:
            grid = c["reqs"] <= 64 and u * c["reqs"] <= (3072 if c["fmt"] == "tq4" else 2048)
        assert ("balanced_kernel" not in run[0][0]) == grid, c
        if grid and c["reqs"] <= 16:
            shape = run[0][1]
            assert shape[0] * 8 >= u, c


def test_queried_scratch_gives_the_launches_of_a_large_one(recorder):
    """What the size query answers is what the launchers want: same kernels, grids and numbers of chunks as with 64 MiB."""
    cases = [case(fmt, reqs, q_len, max_seq, q_heads, kv_heads, head_dim, xf, scratch=("queried", 64 << 20))
             for fmt, xf, q_heads, kv_heads, head_dim in (("tq4", 1, 16, 2, 256), ("tq4", 1, 32, 4, 256), ("q8_0", 0, 16, 2, 256), ("q8_0", 1, 8, 1, 256),
                                                          ("fp8", 0, 32, 1, 256), ("bf16", 0, 16, 2, 256), ("bf16", 0, 16, 4, 128))
             for reqs, q_len in ((1, 1), (1, 2), (1, 4), (1, 7), (1, 16), (2, 1), (3, 4), (16, 1), (40, 1))
             for max_seq in (1, 100, 224, 257, 600, 768, 769, 1000, 1200, 2500, 5000, 6144, 8192, 8193, 10000, 32000, 131072)]
    for c, (need, (queried, large)) in zip(cases, recorder(cases)):
        assert queried == large, (c, need)


def test_merge_of_one_wave(recorder):
    """In the place of sixteen waves up to 16 chunks, of four (from 32 rows per kv head on) up to 32."""
    cases = [case(fmt, 1, q_len, 32 * units) for fmt in ("tq4", "q8_0", "bf16") for q_len in (1, 2, 3, 4, 8) for units in range(8, 300, 7)]
    forms = set()
    for c, (_, (run,)) in zip(cases, recorder(cases)):
        if len(run) == 2:
            name, (_, _, _, _, slots), _ = run[1]
            few = 32 if c["q_len"] * 8 >= 32 else 16
            assert ("split_merge_few_kernel" in name) == (slots <= few), (c, name, slots)
            forms.add((few, slots <= few))
    assert len(forms) == 4


def test_shorter_chunks_take_no_second_round(recorder):
    """A call that fits the chip (256 workgroups) with chunks of eight units does so with shorter ones, up to four kv heads; at one kv head as at
    four the same number of chunks."""
    cases = [case(fmt, 1, q_len, 32 * units, 8 * kv_heads, kv_heads, head_dim, xf)
             for fmt, xf, head_dim in (("tq4", 1, 256), ("q8_0", 0, 256), ("bf16", 0, 128)) for q_len in (1, 2, 4, 6, 8, 12, 16)
             for units in (9, 15, 19, 30, 47, 63, 94, 120, 188) for kv_heads in (1, 2, 4)]
    chunks = {}
    for c, (_, (run,)) in zip(cases, recorder(cases)):
        n, whole, tiles = run[0][2][0], (c["max_seq"] // 32 + 1 + 7) // 8, (c["q_len"] * 8 + 15) // 16
        assert n * tiles * c["kv_heads"] <= max(256, min(whole, 128 // tiles) * tiles * c["kv_heads"]), c
        assert chunks.setdefault((c["fmt"], c["q_len"], c["max_seq"]), n) == n, c


def test_batches_of_the_plain_kernels(recorder):
    """The batches of several requests whose bytes are compared with the general kernels' run in the plain ones."""
    from oracle import FMT_FP8, FMT_Q8_0
    from test_gpu_plain_decode import ON_GRID

    names = {FMT_Q8_0: "q8_0", FMT_FP8: "fp8"}
    cases = [case(names.get(fmt, "tq4"), len(seqs), max(q_lens), bound or max(seqs), q_heads, kv_heads)
             for fmt, _, _, kv_heads, q_heads, seqs, q_lens, bound in ON_GRID]
    for c, (_, (run,)) in zip(cases, recorder(cases)):
        assert ("paged_attn_tq4_plain_kernel" if c["fmt"] == "tq4" else "paged_attn_rows_plain_kernel") in run[0][0], (c, run[0][0])
        if c["fmt"] != "tq4":  # one tile per request
            assert re.search(r"plain_kernelI.*Lb1E", run[0][0]), run[0][0]

"""warp34_paged_attention_scratch_bytes[_for_layout] on the CPU: a pure function of its numbers.  The calls run
in a child process, so that one that ends the process fails its test and not the test run."""
import json
import os
import subprocess
import sys

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
RECORD = 260 * 4  # a partial record: 256 fp32 channels, maximum, sum, two unused

CHILD = """
import ctypes as C, json, sys
from warp34_amd import ffi
lib = ffi.load()
out = []
for c in json.loads(sys.argv[1]):
    xf = {"tq4": (1, 1), "q8_0 rotated values": (0, 1)}.get(c["fmt"], (0, 0))
    fmt = {"tq4": ffi.WARP34_KV_FORMAT_TQ4, "fp8": ffi.WARP34_KV_FORMAT_FP8_E4M3, "bf16": ffi.WARP34_KV_FORMAT_BF16,
           "fp16": ffi.WARP34_KV_FORMAT_FP16}.get(c["fmt"], ffi.WARP34_KV_FORMAT_Q8_0)
    L = ffi.Warp34KvLayerLayout(0, 0, *([0] * 6), 0, 0, c["kv_heads"], c["head_dim"], 64, fmt, fmt, *xf, 0)
    out.append(lib.warp34_paged_attention_scratch_bytes_for_layout(C.byref(L), c["tokens"], c["reqs"], c["q_heads"],
                                                                   c["max_seq"]))
print(json.dumps(out))
"""


def query(tokens, reqs, max_seq, fmt="tq4", q_heads=16, kv_heads=2, head_dim=256):
    case = dict(tokens=tokens, reqs=reqs, max_seq=max_seq, fmt=fmt, q_heads=q_heads, kv_heads=kv_heads, head_dim=head_dim)
    p = subprocess.run([sys.executable, "-c", CHILD, json.dumps([case])], cwd=ROOT, stdout=subprocess.PIPE,
                       stderr=subprocess.PIPE, text=True)
    assert p.returncode == 0, "the query ended its process: %s %s" % (p.returncode, p.stderr)
    return json.loads(p.stdout)[0]


@pytest.mark.parametrize("fmt", ["tq4", "q8_0"])
def test_request_counts_outside_the_batch(fmt):
    """4 tokens, 16 query rows per kv head: a request of 1000 keys (33 units counted) has nine chunks of four units, no
    request means no plan; a negative count and one above the tokens stand for one token per request."""
    assert query(4, 0, 1000, fmt) == 4 * 16 * 9 * RECORD
    assert query(4, -1, 1000, fmt) == query(4, 4, 1000, fmt) == query(4, 9, 1000, fmt)


def chunks(tokens, n, q_heads=16):
    return tokens * q_heads * n * RECORD


def plan(tokens, entries, columns=16, kv_heads=2):
    return (128 + entries) * kv_heads * columns * RECORD + 16 * tokens


@pytest.mark.parametrize("fmt", ["tq4", "q8_0", "fp8", "bf16", "fp16", "q8_0 rotated values"])
def test_batches_on_the_chunk_grid_are_not_sized_for_the_plan(fmt):
    """One request's decode step, and up to eight 16-column tiles per kv head: the records of the chunks."""
    assert query(1, 1, 131072, fmt) == chunks(1, 128)
    assert query(4, 1, 131072, fmt) == chunks(4, 64)
    assert query(16, 1, 131072, fmt) == chunks(16, 16)
    assert query(16, 4, 21000, fmt) == chunks(16, 16)


def test_decode_batches_of_every_format_and_verify_batches_of_row_formats():
    """Shares + entries.  A verify batch of TQ4 pages has no entries wider than a tile: chunks, or the parts of a
    shared prefix (16 requests x 4 tokens, group 8: 4 tiles of 128 rows, 32 parts behind 4 chunks)."""
    for fmt in ("tq4", "q8_0", "bf16"):
        assert query(32, 32, 30000, fmt) == plan(32, 32)
        assert query(32, 16, 30000, fmt) == max(plan(32, 16), chunks(32, 8))
    assert query(4, 4, 2000, "bf16", q_heads=4, kv_heads=2, head_dim=128) == max(plan(4, 4), chunks(4, 16, 4))
    assert query(3, 3, 2000, "bf16", q_heads=4, kv_heads=2, head_dim=128) == chunks(3, 16, 4)
    for fmt in ("q8_0", "fp8", "bf16", "fp16"):
        assert query(20, 5, 21000, fmt) == plan(20, 5, 32)
        assert query(64, 16, 262144, fmt) == plan(64, 16, 32)
        assert query(32, 2, 21000, fmt) == plan(32, 2 * 4, 32)
    assert query(20, 5, 21000, "q8_0 rotated values") == plan(20, 5 * 2, 16)
    assert query(20, 5, 21000, "tq4") == chunks(20, 12)
    assert query(64, 16, 262144, "tq4") == chunks(64, 4 + 32) + 32
    assert query(64, 16, 3000, "tq4") == chunks(64, 4)
    assert query(64, 4, 9000, "bf16", kv_heads=4, head_dim=128) == chunks(64, 8)


def test_the_plan_does_not_take_batches_above_its_limits():
    """More than 16 tiles per request, more than 65 535 tokens: neither plan nor, with so many tiles, chunks."""
    assert query(5 * 65, 5, 9000, "q8_0") == 0
    assert query(1 << 17, 1 << 16, 100, "bf16") == 0
    assert query(2**31 - 1, 2, 100, "bf16") == 0

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
    """4 tokens, 16 query rows per kv head: five chunks of a request of 1000 keys fit their minimum of 8 units, no
    request means no plan; a negative count and one above the tokens stand for one token per request."""
    assert query(4, 0, 1000, fmt) == 4 * 16 * 5 * RECORD
    assert query(4, -1, 1000, fmt) == query(4, 4, 1000, fmt) == query(4, 9, 1000, fmt)

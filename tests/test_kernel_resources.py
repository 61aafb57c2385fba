"""What the built library's kernel descriptors say: the row-format attention and the prefill kernels keep everything in registers.
A reload from scratch memory waits for the row loads in flight as well, which the kernels place their own waits for.  And what the
compiler makes of device helpers whose instructions have waiting times."""
import os
import re
import shutil
import struct
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
READELF = "/opt/rocm/llvm/bin/llvm-readelf"


def code_objects(tmp_path):
    """Paths of the gfx950 code objects inside the library."""
    from warp34_amd import ffi

    data = open(ffi.LIB_PATH, "rb").read()
    paths, at = [], data.find(b"__CLANG_OFFLOAD_BUNDLE__")
    while at >= 0:
        pos = at + 32
        for _ in range(struct.unpack_from("<Q", data, at + 24)[0]):
            offset, size, name_len = struct.unpack_from("<QQQ", data, pos)
            triple = data[pos + 24:pos + 24 + name_len]
            pos += 24 + name_len
            if b"gfx950" not in triple or not size:
                continue
            paths.append(os.path.join(str(tmp_path), "%d.o" % len(paths)))
            with open(paths[-1], "wb") as f:
                f.write(data[at + offset:at + offset + size])
        at = data.find(b"__CLANG_OFFLOAD_BUNDLE__", at + 24)
    return paths


def readelf(*args):
    return subprocess.run([READELF, *args], stdout=subprocess.PIPE, text=True, check=True).stdout


def kernel_scratch_bytes(tmp_path):
    """{kernel name: bytes of scratch memory per lane}"""
    found = {}
    for path in code_objects(tmp_path):
        for name, scratch in re.findall(r"\.name: +(_Z\S+)\n(?:.*\n)*?.*\.private_segment_fixed_size: (\d+)", readelf("--notes", path)):
            found[name] = int(scratch)
    return found


def kernel_scalar_spills(tmp_path):
    """{kernel name: scalar registers that are kept in lanes of vector registers}"""
    found = {}
    for path in code_objects(tmp_path):
        for name, spills in re.findall(r"\.name: +(_Z\S+)\n(?:.*\n)*?.*\.sgpr_spill_count: (\d+)", readelf("--notes", path)):
            found[name] = int(spills)
    return found


def kernel_preload_dwords(tmp_path):
    """{kernel name: dwords of its arguments that are in scalar registers when a wave starts}"""
    found = {}
    for path in code_objects(tmp_path):
        data = open(path, "rb").read()
        text = readelf("--sections", "--symbols", "--wide", path)
        addr, offset = (int(x, 16) for x in re.search(r"\.rodata +PROGBITS +(\w+) +(\w+)", text).groups())
        for value, name in re.findall(r"^ *\d+: (\w+) +64 OBJECT .* (\S+)\.kd$", text, re.M):
            found[name] = struct.unpack_from("<H", data, int(value, 16) - addr + offset + 58)[0] & 127  # kernarg_preload_spec_length
    return found


@pytest.mark.skipif(not os.path.exists(READELF), reason="no llvm-readelf")
def test_row_format_kernels_do_not_spill(tmp_path):
    kernels = {k: v for k, v in kernel_scratch_bytes(tmp_path).items() if "paged_attn_rows" in k}
    assert len(kernels) >= 20, sorted(kernels)
    assert {k: v for k, v in kernels.items() if v} == {}


@pytest.mark.skipif(not os.path.exists(READELF), reason="no llvm-readelf")
def test_prefill_kernels_do_not_spill(tmp_path):
    kernels = {k: v for k, v in kernel_scratch_bytes(tmp_path).items() if "paged_prefill" in k}
    assert len(kernels) >= 16, sorted(kernels)
    assert {k: v for k, v in kernels.items() if v} == {}


@pytest.mark.skipif(not os.path.exists(READELF), reason="no llvm-readelf")
def test_wide_pieces_of_8bit_rows_keep_their_scalars(tmp_path):
    """Two column tiles: a kernel that has to bring 110 scalars and more back starts a microsecond later."""
    kernels = {k: v for k, v in kernel_scalar_spills(tmp_path).items() if re.search(r"rows_balanced_kernel.*Li2ELi[34]E", k)}
    assert len(kernels) == 8, sorted(kernels)
    assert {k: v for k, v in kernels.items() if v >= 100} == {}


@pytest.mark.skipif(not os.path.exists(READELF), reason="no llvm-readelf")
def test_sparse_kernels_do_not_spill(tmp_path):
    """Two registers of the Q8_0 form with rotated values excepted, which is faster with them there."""
    kernels = {k: v for k, v in kernel_scratch_bytes(tmp_path).items() if "qsa_sparse" in k}
    assert len(kernels) == 7, sorted(kernels)
    assert {k: v for k, v in kernels.items() if v > (12 if "rows_kernelILi3ELb1E" in k else 0)} == {}


@pytest.mark.skipif(not os.path.exists(READELF), reason="no llvm-readelf")
@pytest.mark.parametrize("part,dwords", [("kv_append_kernel", 14), ("fused_qk_norm_rope_gate_kernel", 13), ("qk_norm_rope_kernel", 14),
                                         ("balanced_merge_kernel", 10), ("split_merge_few_kernel", 6), ("qsa_sparse_", 11)])
def test_leading_arguments_are_preloaded(tmp_path, part, dwords):
    """Kernels whose first requests wait for nothing but their arguments."""
    kernels = {k: v for k, v in kernel_preload_dwords(tmp_path).items() if part in k and (part != "qk_norm_rope_kernel" or "fused" not in k)}
    assert kernels
    assert {k: v for k, v in kernels.items() if v < dwords} == {}


@pytest.mark.skipif(not os.path.exists(READELF), reason="no llvm-readelf")
@pytest.mark.parametrize("part,dwords", [("balanced_merge_kernel", 12), ("split_merge_few_kernel", 11), ("split_merge_kernel", 11)])
def test_merges_have_all_of_their_leading_arguments(tmp_path, part, dwords):
    """The requests' token ranges and the gate among them, which are asked for together with the slices."""
    kernels = {k: v for k, v in kernel_preload_dwords(tmp_path).items() if re.search(r"w34\d+" + part + "I", k)}
    assert len(kernels) >= 8, sorted(kernels)
    assert {k: v for k, v in kernels.items() if v < dwords} == {}


@pytest.mark.skipif(not os.path.exists(READELF), reason="no llvm-readelf")
def test_tq4_decode_kernels_do_not_spill(tmp_path):
    """Two column tiles hold 128 accumulators per lane; their stores must not turn into an address inside the array either."""
    kernels = {k: v for k, v in kernel_scratch_bytes(tmp_path).items() if "paged_attn_tq4" in k}
    assert len(kernels) == 10, sorted(kernels)
    assert {k: v for k, v in kernels.items() if v} == {}


def assembly(tmp_path, source):
    path = os.path.join(str(tmp_path), "probe.hip")
    with open(path, "w") as f:
        f.write('#include "%s"\n%s' % (os.path.join(ROOT, "warp34_amd", "csrc", "kv_common.h"), source))
    cmd = ["hipcc", "-O3", "-std=c++17", "--offload-arch=gfx950", "--cuda-device-only", "-S", "-o", "-", path]
    text = subprocess.run(cmd, stdout=subprocess.PIPE, text=True, check=True).stdout
    lines = [line.split(";")[0].strip() for line in text.splitlines()]
    return [line for line in lines if re.match(r"[a-z]+_", line)]


@pytest.mark.skipif(shutil.which("hipcc") is None, reason="no hipcc")
def test_product_of_a_weight_waits_for_its_exponential(tmp_path):
    code = assembly(tmp_path, """
        __global__ void weight(float* p, const float* d) {
            const int i = threadIdx.x;
            const float scale = d[i], score = p[i] * scale;
            p[i] = w34::mul_legacy(__builtin_amdgcn_exp2f(score), scale);
        }""")
    at = next(i for i, line in enumerate(code) if line.startswith("v_exp_f32"))
    use = next(i for i, line in enumerate(code) if line.startswith("v_mul_legacy_f32"))
    assert use > at + 1, code[at:use + 1]


@pytest.mark.skipif(shutil.which("hipcc") is None, reason="no hipcc")
@pytest.mark.parametrize("cells_per_unit,holds", [("120.25f", True), ("121.0f", False), ("118.0f", False), ("208.0f", False)])
def test_code_cells_keep_the_boundaries_from_their_edges(tmp_path, cells_per_unit, holds):
    """Sizes of the encoders' cells with every boundary in a cell of its own, but some nearer than a quarter of a cell to its edge (with
    208 also in the first cell), do not compile."""
    csrc = os.path.join(ROOT, "warp34_amd", "csrc")
    with open(os.path.join(csrc, "kv_encode.h")) as f:
        text, n = re.subn(r"kCellsPerUnit = [0-9.]+f", "kCellsPerUnit = " + cells_per_unit, f.read())
    assert n == 1
    path = os.path.join(str(tmp_path), "probe.hip")
    with open(path, "w") as f:
        f.write(text.replace("#pragma once", ""))
    cmd = ["hipcc", "-std=c++17", "--offload-arch=gfx950", "--cuda-device-only", "-fsyntax-only", "-I", csrc, path]
    p = subprocess.run(cmd, stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True)
    assert (p.returncode == 0) == holds, p.stdout
    assert holds or "away from its edges" in p.stdout

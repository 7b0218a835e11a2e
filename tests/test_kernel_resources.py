"""Registers and private memory of the operator kernels, from the metadata of the
library's own code objects: the stage kernel of the 7-site chain in FP64 keeps six
wavefronts per SIMD (80 vector registers), and only matrix-core kernels, which trade
registers for tiles, may spill to private memory."""
import os
import re
import struct
import subprocess
import tempfile

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
LIB = os.path.join(ROOT, "libheom_amd", "_lib", "libheom_amd.so")
LLVM = os.path.join(os.environ.get("ROCM_PATH", "/opt/rocm"), "llvm", "bin")
MAGIC = b"__CLANG_OFFLOAD_BUNDLE__"


def code_objects(data):
    """Device ELF images of the offload bundles in a host library."""
    at = data.find(MAGIC)
    while at >= 0:
        n = struct.unpack_from("<Q", data, at + len(MAGIC))[0]
        p = at + len(MAGIC) + 8
        for _ in range(n):
            off, size, ln = struct.unpack_from("<QQQ", data, p)
            name = data[p + 24:p + 24 + ln].decode()
            p += 24 + ln
            if "gfx950" in name and size:
                yield data[at + off:at + off + size]
        at = data.find(MAGIC, at + 1)


@pytest.fixture(scope="module")
def kernels():
    if not os.path.exists(LIB):
        pytest.skip("library not built")
    out = {}
    for elf in code_objects(open(LIB, "rb").read()):
        with tempfile.NamedTemporaryFile(suffix=".elf") as f:
            f.write(elf)
            f.flush()
            notes = subprocess.run([os.path.join(LLVM, "llvm-readelf"), "--notes", f.name],
                                   capture_output=True, text=True, check=True).stdout
        for k in notes.split("  - .agpr_count:")[1:]:
            get = lambda key: int(re.search(r"\.%s:\s*(\d+)" % key, k).group(1))  # noqa: E731
            name = re.search(r"\.name:\s*(\S+)", k).group(1)
            out[name] = {"vgprs": get("vgpr_count"), "private": get("private_segment_fixed_size"),
                         "spills": get("vgpr_spill_count")}
    names = subprocess.run(["c++filt"], input="\n".join(out), capture_output=True, text=True,
                           check=True).stdout.split("\n")
    return {re.sub(r"\(hamd::Epi\)|hamd::|\(anonymous namespace\)::|^void ", "", n): v
            for n, v in zip(names, out.values())}


def test_operator_kernels_found(kernels):
    for name in ("hilb_fast_kernel<7, double", "hilb_kernel<2, double", "batch_kernel<float"):
        assert any(k.startswith(name) for k in kernels), sorted(kernels)[:5]


@pytest.mark.parametrize("N", [7, 8, 9, 11])
def test_fast_kernel_keeps_six_waves(kernels, N):
    ks = {k: v for k, v in kernels.items()
          if re.match(r"hilb_fast_kernel<%d, double, true, true, [46]" % N, k)}
    assert len(ks) >= 2
    assert {k: v for k, v in ks.items() if v["vgprs"] > 80 or v["private"]} == {}


def test_no_private_memory_outside_matrix_core_kernels(kernels):
    ops = {k: v for k, v in kernels.items() if "StageArgs" in k}  # the operator kernels
    assert len(ops) > 500
    assert {k: v for k, v in ops.items() if v["private"] and "mfma" not in k} == {}
    # there, only what does not fit the registers
    assert {k: v for k, v in ops.items() if v["private"] and not v["spills"]} == {}

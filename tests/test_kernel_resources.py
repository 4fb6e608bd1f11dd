"""Private (scratch) memory of the compiled kernels, from the metadata of the built library.

A kernel that calls a function the compiler did not inline, or that indexes a per-thread array at
run time, keeps a stack in device memory: every hardware queue it runs on then gets its own scratch
allocation, and the call takes the registers of the calling convention.  None of the stencil,
obstacle, swimmer and adjoint kernels needs one.  (The FFT passes are held to 128 registers, where
a few instances spill.)"""
import os
import re
import struct
import subprocess
import tempfile

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
LIB = os.path.join(ROOT, "cubismup_2d_amd", "libcup2d_hip.so")
READELF = "/opt/rocm/llvm/bin/llvm-readelf"
MAGIC = b"__CLANG_OFFLOAD_BUNDLE__"


def device_images(data):
    """The device code objects of the library's offload bundles (one per source file)."""
    for m in re.finditer(MAGIC, data):
        pos = m.start() + len(MAGIC)
        (n,) = struct.unpack_from("<Q", data, pos)
        pos += 8
        for _ in range(n):
            off, size, tlen = struct.unpack_from("<QQQ", data, pos)
            triple = data[pos + 24:pos + 24 + tlen]
            pos += 24 + tlen
            if b"gfx950" in triple and size:
                yield data[m.start() + off:m.start() + off + size]


@pytest.mark.skipif(not os.path.exists(LIB) or not os.path.exists(READELF),
                    reason="needs the built library and ROCm's readelf")
def test_no_private_memory_outside_fft():
    with open(LIB, "rb") as f:
        images = list(device_images(f.read()))
    assert images
    seen, private = 0, {}
    for img in images:
        with tempfile.NamedTemporaryFile(suffix=".elf") as t:
            t.write(img)
            t.flush()
            notes = subprocess.run([READELF, "--notes", t.name], check=True, capture_output=True,
                                   text=True).stdout
        names = re.findall(r"^\s+\.name:\s+(_Z\w+)$", notes, re.M)
        sizes = re.findall(r"\.private_segment_fixed_size:\s+(\d+)", notes)
        assert len(names) == len(sizes)
        for name, size in zip(names, sizes):
            if "k_rows_" in name or "k_cols" in name:
                continue
            seen += 1
            if int(size):
                private[name] = int(size)
    assert seen > 20 and not private, private

"""Registers of the kernels whose blocks fill the register file: none of them
may keep values in scratch memory beyond what is listed. A spill costs no
result, only time (the fp32 GEMM over [K][N] operands ran at a quarter of its
speed, ResNet-50's 128-channel 3x3 layers at 0.94), so no other test sees it. Read from the metadata of the library built
here; CPU only."""
import os
import re
import shutil
import struct
import subprocess

import pytest

from nnr_amd import _lib

READELF = next((p for p in (shutil.which("llvm-readelf"), "/opt/rocm/llvm/bin/llvm-readelf") if p and os.path.exists(p)),
               None)
MAGIC = b"__CLANG_OFFLOAD_BUNDLE__"


def code_objects(data):
    """The gfx950 ELF images of the library's offload bundles."""
    at = data.find(MAGIC)
    while at >= 0:
        n, p = struct.unpack_from("<Q", data, at + len(MAGIC))[0], at + len(MAGIC) + 8
        for _ in range(n):
            off, size, idlen = struct.unpack_from("<QQQ", data, p)
            ident = data[p + 24:p + 24 + idlen]
            p += 24 + idlen
            if b"gfx950" in ident and size:
                yield data[at + off:at + off + size]
        at = data.find(MAGIC, p)


@pytest.fixture(scope="module")
def scratch(tmp_path_factory):
    """{mangled kernel name: scratch bytes a lane}"""
    if READELF is None:
        pytest.skip("llvm-readelf is not here")
    with open(_lib.LIB_PATH, "rb") as f:
        data = f.read()
    path, out = tmp_path_factory.mktemp("co") / "co.elf", {}
    for image in code_objects(data):
        path.write_bytes(image)
        notes = subprocess.run([READELF, "--notes", str(path)], check=True, capture_output=True, text=True).stdout
        for kernel in notes.split("- .agpr_count")[1:]:
            name = re.findall(r"^ {4}\.name: +(\S+)", kernel, re.M)
            out[name[-1].strip("'\"")] = int(re.search(r"\.private_segment_fixed_size:\s+(\d+)", kernel).group(1))
    assert len(out) > 100, "no kernels found in the library"
    return out


# (name pattern, scratch bytes a lane that it may use)
LIMITS = [
    (r"gemm_f32_mfma_kernel", 0),
    # pipelined, K split over two waves (8 waves, 128 registers): dense, uniform taps
    (r"qgemm_dma_kernelILi128ELi128ELi2ELi0ELi\d+ELi0ELi128ELi0ELi2E", 0),
    (r"qgemm_dma_kernelILi128ELi128ELi2ELi3ELi\d+ELi0ELi128ELi0ELi2E", 12),
]


@pytest.mark.parametrize("pattern,limit", LIMITS)
def test_scratch(scratch, pattern, limit):
    found = {n: b for n, b in scratch.items() if re.search(pattern, n)}
    assert found
    assert max(found.values()) <= limit, found

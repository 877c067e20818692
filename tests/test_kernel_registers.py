"""Registers of the LDS-staged bf16 kernels with f32 x, from the code objects of the built library: three blocks of 8 waves
have to fit on a CU (512 registers a lane and SIMD, in eights, six waves a SIMD), two for the pair with two row tiles."""
import os
import re
import struct
import subprocess

import pytest

from sharplight_amd import build, native

READELF = "/opt/rocm/llvm/bin/llvm-readelf"
MAGIC = b"__CLANG_OFFLOAD_BUNDLE__"


def _code_objects(lib):
    """The gfx950 code objects of each translation unit."""
    at = lib.find(MAGIC)
    while at >= 0:
        n, p = struct.unpack_from("<Q", lib, at + 24)[0], at + 32
        for _ in range(n):
            off, size, name = struct.unpack_from("<QQQ", lib, p)
            if lib[p + 24:p + 24 + name].endswith(b"gfx950") and size:
                yield lib[at + off:at + off + size]
            p += 24 + name
        at = lib.find(MAGIC, at + 1)


def test_lds_staged_kernels_keep_their_blocks(tmp_path):
    if not os.path.exists(READELF):
        pytest.skip("llvm-readelf not available")
    native.lib()
    used = {}
    for obj in _code_objects(open(build.LIB, "rb").read()):
        if b"matvec_mfma_lds" not in obj:
            continue
        f = tmp_path / "object"
        f.write_bytes(obj)
        notes = subprocess.run([READELF, "--notes", str(f)], check=True, capture_output=True, text=True, timeout=60).stdout
        for m in re.finditer(r"\.name:\s+_ZN5slhip15matvec_mfma_ldsILb(\d)ELb1ELi256ELi(\d)E.*?\.vgpr_count:\s+(\d+)\s+\.vgpr_spill_count:\s+(\d+)",
                             notes, re.S):
            used[m[1] == "1", int(m[2])] = (int(m[3]), int(m[4]))
    assert set(used) == {(False, 1), (False, 2), (True, 1), (True, 2)}
    for (pair, tiles), (n, spilled) in used.items():
        assert n <= (128 if pair and tiles == 2 else 80) and spilled == 0, (pair, tiles, n, spilled)

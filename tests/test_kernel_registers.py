"""Kernels of the built library that must hold their values in registers: their gfx950 code
objects' metadata (scratch bytes, spilled registers), read without a GPU."""
import os
import re
import struct
import subprocess

import pytest

from exl3_amd import build

READELF = "/opt/rocm/llvm/bin/llvm-readelf"


def kernels(path, tmp_path):
    """{kernel symbol: (scratch bytes, spilled VGPRs)} over the library's offload bundles."""
    data = open(path, "rb").read()
    out, at = {}, data.find(b"__CLANG_OFFLOAD_BUNDLE__")
    while at >= 0:
        n, = struct.unpack_from("<Q", data, at + 24)
        p = at + 32
        for _ in range(n):
            off, size, length = struct.unpack_from("<QQQ", data, p)
            target, p = data[p + 24:p + 24 + length], p + 24 + length
            if b"gfx950" not in target or not size:
                continue
            obj = tmp_path / "code_object"
            obj.write_bytes(data[at + off:at + off + size])
            notes = subprocess.run([READELF, "--notes", str(obj)], capture_output=True, text=True, check=True).stdout
            for k in re.findall(r"- \.agpr_count.*?\.wavefront_size", notes, re.S):
                name, scratch, spill = (re.search(rf"\.{f}:\s+(\S+)", k).group(1) for f in
                                        ("name", "private_segment_fixed_size", "vgpr_spill_count"))
                out[name] = int(scratch), int(spill)
        at = data.find(b"__CLANG_OFFLOAD_BUNDLE__", at + 24)
    return out


@pytest.mark.skipif(not os.path.exists(READELF), reason="no llvm-readelf")
@pytest.mark.parametrize("pattern,least,spilling", [
    # the linear of many rows: 8 widths x 3 codebooks x 3 tiles
    (r"10k_qmv_rowsI", 72, r"(?!)"),
    # the long-run expert kernels in the reference form, two steps in flight (the default): 2
    # projections x 8 widths x 3 codebooks; two instances are faster with 6 and 8 spilled
    # registers than with a wave less
    (r"k_moe_(gate_up|down)_longILi\dELi[012]ELi2E", 48, r"k_moe_gate_up_longILi[23]ELi1E"),
])
def test_no_spills(pattern, least, spilling, tmp_path):
    found = {k: v for k, v in kernels(build.LIB_PATH, tmp_path).items() if re.search(pattern, k)}
    assert len(found) >= least
    assert not {k: v for k, v in found.items() if v[1] > (8 if re.search(spilling, k) else 0)}

"""Registers of the built kernels, from the metadata of the library's gfx950 code objects: the random-candidate
encoders keep everything in registers and LDS, none in scratch memory (but for up to 76 bytes a lane of the batch kernel
with three row blocks in registers, which costs it less than the waves that it would give up)."""
import os
import re
import struct
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
LIB = os.path.join(ROOT, "s2tc_amd", "libtxc_dxtn.so")
READELF = "/opt/rocm/llvm/bin/llvm-readelf"
MAGIC = b"__CLANG_OFFLOAD_BUNDLE__"


def _code_objects():
    data = open(LIB, "rb").read()
    at = data.find(MAGIC)
    while at >= 0:
        n, = struct.unpack_from("<Q", data, at + len(MAGIC))
        p = at + len(MAGIC) + 8
        for _ in range(n):
            off, size, idlen = struct.unpack_from("<QQQ", data, p)
            if b"gfx950" in data[p + 24:p + 24 + idlen] and size:
                yield data[at + off:at + off + size]
            p += 24 + idlen
        at = data.find(MAGIC, at + 1)


def _kernels(tmp_path):
    """{mangled name: bytes of scratch per lane}"""
    out = {}
    for i, obj in enumerate(_code_objects()):
        f = tmp_path / f"{i}.co"
        f.write_bytes(obj)
        notes = subprocess.run([READELF, "--notes", str(f)], capture_output=True, text=True, check=True).stdout
        for k in re.split(r"\n\s*- \.a", notes)[1:]:
            name, scratch = re.search(r"\.name:\s+(\S+)", k), re.search(r"\.private_segment_fixed_size:\s+(\d+)", k)
            if name and scratch:
                out[name.group(1)] = int(scratch.group(1))
    return out


def test_random_candidate_kernels_use_no_scratch(tmp_path):
    if not os.path.exists(LIB) or not os.path.exists(READELF):
        pytest.skip("library or llvm-readelf not here")
    kernels = {k: v for k, v in _kernels(tmp_path).items() if "k_normal" in k}
    assert sum("14k_normal_batchI" in k for k in kernels) >= 8 and sum("8k_normalI" in k for k in kernels) >= 16
    over = {k: v for k, v in kernels.items() if v > (76 if re.search("14k_normal_batchILi.ELi3E", k) else 0)}
    assert over == {}

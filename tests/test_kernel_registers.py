"""Registers of the built kernels, from the metadata of the code objects in
libbluecrunch.so: the strided passes that run between points (k_fwd, k_inv of
transforms and of whole middle passes) and those of few tiles keep everything in
registers. Private memory there is a scratch allocation per launch and a memory
access per twiddle."""
import os
import re
import shutil
import struct
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
LIB = os.path.join(ROOT, "bluecrunch_amd", "libbluecrunch.so")
READELF = "/opt/rocm/llvm/bin/llvm-readelf"
MAGIC = b"__CLANG_OFFLOAD_BUNDLE__"


def _code_objects(lib):
    data = open(lib, "rb").read()
    for m in re.finditer(MAGIC, data):
        at = m.start() + len(MAGIC)
        (n,) = struct.unpack_from("<Q", data, at)
        at += 8
        for _ in range(n):
            off, size, tl = struct.unpack_from("<QQQ", data, at)
            triple = data[at + 24:at + 24 + tl].decode()
            at += 24 + tl
            if "gfx950" in triple and size:
                yield data[m.start() + off:m.start() + off + size]


def test_strided_passes_use_no_private_memory(tmp_path):
    readelf = READELF if os.path.exists(READELF) else shutil.which("llvm-readelf")
    if not readelf:
        pytest.skip("llvm-readelf not available")
    if not os.path.exists(LIB):
        pytest.fail("libbluecrunch.so is not built")
    seen, bad = 0, []
    for i, obj in enumerate(_code_objects(LIB)):
        p = tmp_path / f"{i}.co"
        p.write_bytes(obj)
        notes = subprocess.run([readelf, "--notes", str(p)], check=True, capture_output=True, text=True).stdout
        for name, private in re.findall(r"\.name:\s+(\S+).*?\.private_segment_fixed_size:\s+(\d+)", notes, re.S):
            # k_fwd<L, C, PACK = false, ..>, k_inv<L, C, MODE = 0, ..>, k_fwd8, k_inv8
            if re.search(r"k_fwdILi\d+ELi\d+ELb0E|k_invILi\d+ELi\d+ELi0E|k_(fwd|inv)8I", name):
                seen += 1
                if int(private):
                    bad.append((name, int(private)))
    assert seen > 40
    assert not bad, bad

"""The outermost stage of a strided pass (first_stage), compiled with g++ from the
kernels' own source: two to four radix-2 levels in registers, forward and inverse,
against the same butterflies in long double with exact twiddles. With every twiddle a
table entry or i times one, an output carries the rounding of one addition and, in
half of the cases, one complex product per level: at most sqrt(levels) times
sqrt(1/2 + 5/2) 2^-53 of the norm, and no more than with twiddles that are products."""
import math
import os
import shutil
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
SRC = os.path.join(os.path.dirname(HERE), "bluecrunch_amd", "csrc", "fft_device.h")


def _cut(src, a, b):
    i = src.index(a)
    return src[i:src.index(b, i)]


def test_first_stage_error(tmp_path):
    if not shutil.which("g++"):
        pytest.skip("g++ not available")
    src = open(SRC).read()
    body = (_cut(src, "__device__ __forceinline__ cd cadd", "// Streaming (nontemporal)")
            + _cut(src, "// e^{+2 pi i j / 16}", "constexpr int ilog2c")
            + _cut(src, "// Level twiddle bases of dif_levels", "// 3-point DFT, natural order"))
    with open(tmp_path / "stages_cpu.h", "w") as f:
        f.write('#include "emu.h"\n#define __restrict__\nstruct double2 { double x, y; };\n'
                "inline double2 make_double2(double x, double y) { return {x, y}; }\ntypedef double2 cd;\n" + body)
    exe = tmp_path / "stages"
    subprocess.run(["g++", "-std=c++20", "-O1", "-pthread", "-w", f"-I{HERE}/emu", f"-I{tmp_path}",
                    os.path.join(HERE, "emu", "stages.cpp"), "-o", str(exe)], check=True)
    rows = [r.split() for r in subprocess.run([str(exe)], check=True, capture_output=True, text=True).stdout.splitlines()]
    assert len(rows) == 10
    for L, rb, inv, fine, prod in rows:
        rb, fine, prod = int(rb), float(fine), float(prod)
        assert fine <= math.sqrt(3 * rb) * 2.0 ** -53, (L, rb, inv, fine)
        assert fine <= prod * (1 if rb == 2 else 0.99), (L, rb, inv, fine, prod)

"""The carry from group sums (k_carry_groups), run on the CPU from the kernel's own
source against a thread-per-lane stand-in for the HIP built-ins (tests/emu): its
words equal Python integers for outputs as long as the digits reach, one, two and
thousands of words longer, with and without an addend that goes on there, for
group starts on whole words and between them. LDS beyond the staged group sums
holds a pattern, so a word taken from there shows."""
import os
import random
import shutil
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
SRC = os.path.join(os.path.dirname(HERE), "bluecrunch_amd", "csrc", "kernels.h")
GCT, GWPT, GCOV = 256, 8, 4

STAND_IN = """
#include "emu.h"
#include <algorithm>
#include <cstdlib>
using std::min;
struct uint4 { uint32_t x, y, z, w; };
inline uint4 make_uint4(uint32_t x, uint32_t y, uint32_t z, uint32_t w) { return {x, y, z, w}; }
std::vector<uint32_t> g_lds;
struct Lds {
  uint32_t &operator[](size_t i) const {
    if (i >= g_lds.size()) std::abort();
    return g_lds[i];
  }
};
unsigned g_lanes[1024];
inline unsigned __shfl_up(unsigned v, int off, int) {
  const unsigned t = threadIdx.x;
  g_lanes[t] = v;
  __syncthreads();
  const unsigned r = (int)(t & 63) >= off ? g_lanes[t - off] : v;
  __syncthreads();
  return r;
}
struct HostResult { unsigned margin, open_carry; };
inline void host_store(unsigned *p, unsigned v) { *p = v; }
struct MulDesc { uint32_t *c; const uint32_t *d; unsigned long long cl, dl; int bits, cbits, gk; };
constexpr int MARGIN_SLOTS = 64, MARGIN_STRIDE = 32;
inline unsigned margin_of_slots(const unsigned *, int) { return 0; }
"""


def _cut(src, a, b):
    i = src.index(a)
    return src[i:src.index(b, i)]


@pytest.fixture(scope="module")
def drv(tmp_path_factory):
    if not shutil.which("g++"):
        pytest.skip("g++ not available")
    d = tmp_path_factory.mktemp("emu")
    src = open(SRC).read()
    body = (_cut(src, "// Carry functions of single-bit carry chains", "__device__ __forceinline__ long long coef_at")
            + _cut(src, "// Batched carries: product p's", "// Coefficient window of one carry block")
            + _cut(src, "// floor(x / b) for 0 <= x < 2^40", "// x / b for 0 <= x < 2^24")
            + _cut(src, "struct BlockCarry {", "// Words of one block from coefficients")
            + _cut(src, "constexpr int GCT = 256;", "// The blocks whose carry-in the block itself left open"))
    body = body.replace("extern __shared__ uint32_t gl_w[];", "const Lds gl_w;")
    with open(d / "carry_cpu.h", "w") as f:
        f.write(STAND_IN + body)
    exe = d / "drv"
    subprocess.run(["g++", "-std=c++20", "-O1", "-pthread", "-w", f"-I{HERE}/emu", f"-I{d}",
                    os.path.join(HERE, "emu", "carry.cpp"), "-o", str(exe)], check=True)
    return str(exe), d


def _words(x, n):
    return [(x >> (32 * t)) & 0xffffffff for t in range(n)]


# digits a group and bits a digit: groups on whole words (16 x 16, 8 x 16, 8 x 12, 8 x 20,
# 16 x 4), between them (16 x 15, 8 x 14)
@pytest.mark.parametrize("C,b", [(16, 16), (8, 16), (8, 12), (8, 20), (16, 4), (16, 15), (8, 14)])
@pytest.mark.parametrize("more,addend", [(0, True), (1, False), (1, True), (2, True), (5000, False), (5000, True)])
def test_words_past_the_last_group_sum(drv, C, b, more, addend):
    exe, d = drv
    n2 = 768                                  # digits of the product (2 N)
    cb = 2 * b + 11                           # its coefficients lie below 2^cb
    off = max((C * b * g) & 31 for g in range(32))
    K = (off + b * (C - 1) + cb + 31) // 32
    gb = C * b
    cover = (K + gb // 32 - 1) // (gb // 32) if gb % 32 == 0 else (32 * K + gb - 1) // gb + 1
    assert cover <= GCOV
    rng = random.Random(1000 * C + 10 * b + more + addend)
    coef = [rng.getrandbits(cb) for _ in range(n2)]
    stride, sums = (K + 3) & ~3, []
    for g in range(n2 // C):
        s = sum(coef[C * g + i] << (b * i) for i in range(C)) << (gb * g & 31)
        sums += _words(s, stride)
    CL = n2 * b // 32 + more
    D = rng.getrandbits(32 * (CL - 1)) if addend else 0
    lds = (32 * GCT * GWPT // gb + GCOV + 4) * stride
    lds += lds // 32 + 4
    inp, out = d / "in", d / "out"
    with open(inp, "w") as f:
        f.write(f"{C} {b} {K} {n2 // C} {CL} {CL - 1 if addend else 0} {cover} {lds}\n")
        f.write(" ".join(map(str, sums)) + "\n" + " ".join(map(str, _words(D, CL - 1 if addend else 0))) + "\n")
    subprocess.run([exe, str(inp), str(out)], check=True)
    got = list(map(int, open(out).read().split()))
    assert not any(got[CL:])                  # no block here waits for the one below
    want = _words((sum(c << (b * j) for j, c in enumerate(coef)) + D) % (1 << (32 * CL)), CL)
    assert not [i for i in range(CL) if got[i] != want[i]][:3]

"""Host arrays through the staging ring: sizes around one piece (512 KiB), around
all sixteen of a region (8 MiB) and beyond, in and out, and a product whose
output array is one of its operands."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

PIECE = 131072  # words


@pytest.mark.parametrize("n", [PIECE - 1, PIECE, PIECE + 1, 2 * PIECE, 2 * PIECE + 3, 3 * PIECE - 1, 16 * PIECE - 1,
                               16 * PIECE, 16 * PIECE + 5])
def test_words_in_and_out(bc, n):
    a = np.random.default_rng(n).integers(0, 1 << 32, n, dtype=np.uint64).astype(np.uint32)
    c, _ = bc.mul(a, np.array([3], dtype=np.uint32))
    t = a.astype(np.uint64) * 3
    want = np.append(t & 0xFFFFFFFF, np.uint64(0))
    want[1:] += t >> 32
    while (want >> 32).any():
        carry = want >> 32
        want &= 0xFFFFFFFF
        want[1:] += carry[:-1]
    assert np.array_equal(c, want.astype(np.uint32))


def test_output_is_an_operand(bc):
    n = 2 * PIECE + 7
    rng = np.random.default_rng(1)
    a = rng.integers(0, 1 << 32, n, dtype=np.uint64).astype(np.uint32)
    b = rng.integers(0, 1 << 32, n, dtype=np.uint64).astype(np.uint32)
    want = bc.mul(a, b, cl=n)[0]
    c = a.copy()
    bc.check(bc.lib().bcg_mul_host(c.ctypes.data, n, c.ctypes.data, n, b.ctypes.data, n, None), "mul")
    assert np.array_equal(c, want)

"""Sums and differences of device bigfloats around the workgroup size (2048
words) and the 64 blocks one look covers: carries and borrows through runs of
whole blocks, cancellation down to one word, equal operands, either order."""
import numpy as np
import pytest

from helpers import words_to_int

pytestmark = pytest.mark.gpu

SIZES = [1, 2, 2047, 2048, 2049, 4096, 64 * 2048, 64 * 2048 + 1, 66 * 2048 + 5, 131 * 2048 + 7]


def _value(t):
    w, e, s = t
    v = words_to_int(w) << (32 * e) if e >= 0 else words_to_int(w)
    return v if s else -v


def _op(bc, name, a, b):
    x, y, t = bc.DeviceBigfloat((a, 0, 1)), bc.DeviceBigfloat((b, 0, 1)), bc.DeviceBigfloat()
    bc.bf_op(name, t, x, y, 0)
    w, e, s = t.triple()
    assert w.size == 0 or w[-1] != 0 or name == "add"
    return _value((w, e, s))


@pytest.mark.parametrize("n", SIZES)
def test_carry_and_borrow_runs(bc, n):
    ones = np.full(n, 0xFFFFFFFF, dtype=np.uint32)
    one = np.ones(1, dtype=np.uint32)
    power = np.zeros(n + 1, dtype=np.uint32)
    power[n] = 1  # 2^(32 n)
    rng = np.random.default_rng(n)
    r = rng.integers(1, 1 << 32, n, dtype=np.uint64).astype(np.uint32)
    low = r.copy()
    low[0] ^= 1  # differs from r in the lowest word only
    pairs = [(ones, one), (power, one), (power, ones), (ones, ones), (r, low), (low, r), (r, r), (power, r), (r, one)]
    for a, b in pairs:
        x, y = words_to_int(a), words_to_int(b)
        assert _op(bc, "add", a, b) == x + y
        assert _op(bc, "sub", a, b) == x - y
        assert _op(bc, "sub", b, a) == y - x


@pytest.mark.parametrize("n", [2048, 64 * 2048 + 1])
def test_target_is_an_operand(bc, n):
    rng = np.random.default_rng(n)
    a = rng.integers(0, 1 << 32, n, dtype=np.uint64).astype(np.uint32)
    b = rng.integers(0, 1 << 32, n - 3, dtype=np.uint64).astype(np.uint32)
    a[-1] |= 1
    b[-1] |= 1
    x, y = bc.DeviceBigfloat((a, 0, 1)), bc.DeviceBigfloat((b, 0, 1))
    bc.bf_op("sub", x, x, y, 0)
    assert _value(x.triple()) == words_to_int(a) - words_to_int(b)
    bc.bf_op("add", y, x, y, 0)
    assert _value(y.triple()) == words_to_int(a)


@pytest.mark.parametrize("n", [8192 * 17 - 1, 8192 * 64 + 1, 8192 * 66 + 5])
def test_runs_in_long_blocks(bc, n):
    # above 2^17 words a workgroup takes 8192 of them
    test_carry_and_borrow_runs(bc, n)

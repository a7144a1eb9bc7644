"""Carry blocks that cannot know their own carry-in: the word below a block is
all ones, so the carry into it decides (single products, products in place,
batches and fft_to_int), for runs that start and end one word around block
boundaries, with and without a carry entering them."""
import numpy as np
import pytest

from helpers import int_to_words, words_to_int

pytestmark = pytest.mark.gpu

BLOCK = 2048  # words per carry block of a product (1024 in fft_to_int)


def _operands(first, last, n=12 * BLOCK + 77, shift=3 * BLOCK + 5):
    """A: zeros but words [first, last) all ones; B = 2^(32 shift): the product
    is A moved up by shift words."""
    a = np.zeros(n, dtype=np.uint32)
    a[-1] = 5
    a[first:last] = 0xFFFFFFFF
    b = np.zeros(shift + 1, dtype=np.uint32)
    b[shift] = 1
    return a, b, shift


@pytest.mark.parametrize("start", [-2, -1, 0, 1])
@pytest.mark.parametrize("length", [1, 2, 3, BLOCK, BLOCK + 1, 5 * BLOCK + 1])
def test_open_block_of_a_product(bc, start, length):
    shift = 3 * BLOCK + 5
    first = 5 * BLOCK + start - shift  # the run starts at product word 5 BLOCK + start
    a, b, shift = _operands(first, first + length)
    n = a.size + b.size
    for carry in (0, 1):
        d = np.zeros(first + shift + 1, dtype=np.uint32)
        d[first + shift] = carry
        want = (words_to_int(a) << (32 * shift)) + words_to_int(d)
        c, info = bc.muladd(a, b, d, n)
        assert info["passes"] > 1
        assert words_to_int(c) == want
        if length <= BLOCK + 1:
            out, _ = bc.mul_batch([(a, b), (a, b)], cls=[n, n], adds=[d, np.zeros(1, np.uint32)])
            assert words_to_int(out[0]) == want
            assert words_to_int(out[1]) == words_to_int(a) << (32 * shift)


@pytest.mark.parametrize("start", [-2, -1, 0, 1])
@pytest.mark.parametrize("length", [1, 2, 1024, 3 * 1024 + 1])
def test_open_block_of_fft_to_int(bc, start, length):
    # 16-bit digits: all ones is 0xffff twice a word; a digit of 0x10000 at the
    # run's start carries into it
    words, first = 8 * 1024 + 13, 2 * 1024 + start
    for carry in (0, 1):
        digits = np.zeros(2 * words)
        digits[2 * first:2 * (first + length)] = 0xFFFF
        digits[2 * first] += carry
        z = (digits * words * 2).astype(np.complex128)
        got = bc.fft_to_int(z, 2 * words, words, 16)
        want = ((1 << (32 * length)) - 1 + carry) << (32 * first)
        assert np.array_equal(got, int_to_words(want, words))


@pytest.mark.parametrize("off", [0.3, 0.45, -0.45])
@pytest.mark.parametrize("carry", [0, 1])
def test_open_block_of_fft_to_int_between_whole_numbers(bc, oracle, off, carry):
    # the points are rounded whatever their distance; the carry through words of
    # ones runs on all the same
    words = 3 * 1024 + 13
    digits = np.full(2 * words, 65535.0)
    digits[0] += carry
    length = 8192
    z = np.zeros(length, dtype=np.complex128)
    z[:2 * words] = (digits + off) * length
    want, margin = oracle.fft_to_int(z, length, words, 16)
    got = bc.fft_to_int(z, length, words, 16)
    assert margin > 0.25
    assert np.array_equal(want, np.zeros(words) if carry else np.full(words, 0xFFFFFFFF, dtype=np.uint32))
    assert np.array_equal(got, want)

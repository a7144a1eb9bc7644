"""One workgroup per contiguous block of points: every one-pass product length
(64 to 8192 points, 2^k and 3 * 2^k) at the longest and the shortest operands
of its class, ragged pairs, squares and operands of all ones, and every middle
pass length in a two-pass split, each product exact."""
import numpy as np
import pytest

from helpers import exact_product, reference_order
from bluecrunch_amd.workload import operands

pytestmark = pytest.mark.gpu

LENGTHS = [64, 96, 128, 192, 256, 384, 512, 768, 1024, 1536, 2048, 3072, 4096, 6144, 8192]


def _pairs(bc, n):
    """(al, bl) on both edges of the class of n points, balanced and 1 to 3."""
    out = []
    for num in (2, 4):  # bl = al, bl = al / 3
        on = [t for t in range(100, 2 * n) if bc.plan(t - t // num, t // num)["points"] == n]
        if on:
            out += [(t - t // num, t // num) for t in (on[0], on[-1])]
    return out


@pytest.mark.parametrize("n", LENGTHS)
def test_one_pass_lengths(bc, n):
    pairs = _pairs(bc, n)
    if not pairs:
        pytest.skip("no product of at least 100 words has this length")
    for al, bl in pairs:
        a, b = operands(al * 31 + bl, al, bl)
        c, info = bc.mul(a, b)
        assert (info["points"], info["passes"]) == (n, 1)
        assert np.array_equal(c, exact_product(a, b)), (al, bl)
        s, sinfo = bc.mul(a, a)
        assert np.array_equal(s, exact_product(a, a)), (al, sinfo)
        ones = np.full(al, 0xFFFFFFFF, dtype=np.uint32)
        m, _ = bc.mul(ones, b)
        assert np.array_equal(m, exact_product(ones, b)), (al, bl)
    out, worst = bc.mul_batch([operands(k, al, bl) for k, (al, bl) in enumerate(pairs * 3)])
    for k, (c, (al, bl)) in enumerate(zip(out, pairs * 3)):
        assert np.array_equal(c, exact_product(*operands(k, al, bl))), (al, bl)
    assert worst < 0.25


@pytest.mark.parametrize("inner", [x for x in LENGTHS if x >= 128])
def test_middle_pass_lengths(bc, inner):
    n = 64 * inner
    if n < 12288:
        pytest.skip("shorter lengths run as one pass")
    lo, hi = 100, n
    while hi - lo > 1:  # the longest balanced product of n points
        mid = (lo + hi) // 2
        lo, hi = (mid, hi) if bc.plan(mid, mid)["points"] <= n else (lo, mid)
    assert bc.plan(lo, lo)["points"] == n
    a, b = operands(inner, lo, lo - 7)
    want = exact_product(a, b), exact_product(a, a)
    cands = bc.plan_candidates(n)
    picks = [i for i, (P, L, C) in enumerate(cands) if P == 2 and L == [64, inner]]
    assert picks
    try:
        for i in picks:
            bc.plan_force(n, i)
            c, info = bc.mul(a, b)
            assert info["passes"] == 2 and np.array_equal(c, want[0]), cands[i]
            s, _ = bc.mul(a, a)
            assert np.array_equal(s, want[1]), cands[i]
    finally:
        bc.plan_force(n, -1)


def test_margins_are_each_products_own(bc):
    # a margin raised by digits far above the bound must not stay in any slot:
    # the same product reads the same margin before and after it, alone and batched
    a, b = operands(7, 3000, 2500)
    own = bc.mul(a, b)[1]["margin"]
    _, batch = bc.mul_batch([(a, b), (a[:700], b[:600])])
    bc.plan_digit_bias(6)
    try:
        assert bc.mul(*operands(8, 5000, 5000))[1]["retries"] >= 1
        bc.mul_batch([operands(9, 5000, 5000), operands(10, 5000, 5000), operands(11, 40000, 40000)])
    finally:
        bc.plan_digit_bias(0)
    assert bc.mul(a, b)[1]["margin"] == own
    assert bc.mul_batch([(a, b), (a[:700], b[:600])])[1] == batch
    small = bc.mul(a[:700], b[:600])[1]["margin"]
    assert batch == max(own, small) and small < own


@pytest.mark.parametrize("inner", LENGTHS)
def test_innermost_pass_of_transforms(bc, inner):
    # alone (one block), and under 128 rows (several blocks per workgroup)
    for n in (inner, 128 * inner):
        rng = np.random.default_rng(n)
        x = rng.standard_normal(n) + 1j * rng.standard_normal(n)
        want = (np.fft.ifft(x) * n)[reference_order(n)]
        picks = [i for i, (P, L, C) in enumerate(bc.plan_candidates(n)) if n == inner or L == [128, inner]][:1]
        try:
            for i in picks:
                bc.plan_force(n, i)
                z = x.copy()
                bc.fft_forward(z)
                assert np.abs(z - want).max() <= 1e-13 * np.abs(want).max() * np.log2(n)
                back = want.copy()
                bc.fft_inverse(back)
                assert np.abs(back / n - x).max() <= 1e-13 * np.abs(x).max() * np.log2(n)
        finally:
            bc.plan_force(n, -1)


@pytest.mark.parametrize("rows", [64, 128, 256])
@pytest.mark.parametrize("inner", [192, 256])
def test_packing_and_unpacking_of_few_tiles(bc, rows, inner):
    # eight columns: balanced, and with words in the upper digit half (4 to 1)
    n = rows * inner
    if n < 12288:
        pytest.skip("shorter lengths run as one pass")
    total = max(t for t in range(2, 2 * n, 2) if bc.plan(t // 2, t // 2)["points"] <= n)
    picks = [i for i, (P, L, C) in enumerate(bc.plan_candidates(n)) if P == 2 and L == [rows, inner] and C[0] == 8]
    assert picks
    try:
        bc.plan_force(n, picks[0])
        for al in (total // 2, total * 4 // 5):
            bl = total - al
            a, b = operands(rows + al, al, bl)
            c, info = bc.mul(a, b)
            assert info["passes"] == 2
            assert np.array_equal(c, exact_product(a, b)), (al, bl)
            ones = np.full(al, 0xFFFFFFFF, dtype=np.uint32)
            c, _ = bc.mul(ones, b)
            assert np.array_equal(c, exact_product(ones, b)), (al, bl)
    finally:
        bc.plan_force(n, -1)


@pytest.mark.parametrize("n", [12288, 16384, 24576, 32768, 49152])
def test_group_sums_of_nine_to_twelve_words(bc, n):
    # sixteen columns with 15- and 16-bit digits: the longest operands of the class,
    # random and all ones (the largest coefficients), odd lengths below them
    total = max(t for t in range(2, 2 * n, 2) if bc.plan(t // 2, t // 2)["points"] <= n)
    picks = [i for i, (P, L, C) in enumerate(bc.plan_candidates(n)) if P == 2 and C[0] == 16][:2]
    assert picks
    try:
        for i in picks:
            bc.plan_force(n, i)
            for al, bl in ((total // 2, total // 2), (total // 2 - 5, total // 2 - 26)):
                a, b = operands(n + al, al, bl)
                c, info = bc.mul(a, b)
                assert (info["group_digits"], info["group_stride"]) == (16, 12), info
                assert np.array_equal(c, exact_product(a, b))
                ones = np.full(al, 0xFFFFFFFF, dtype=np.uint32)
                c, _ = bc.mul(ones, np.full(bl, 0xFFFFFFFF, dtype=np.uint32))
                assert np.array_equal(c, exact_product(ones, ones[:bl]))
    finally:
        bc.plan_force(n, -1)

"""Products whose digits fill their transform length exactly (32 (AL + BL) = 2 N b),
with outputs one, two and thousands of words longer than AL + BL and an addend that
goes on there: the words past the last group sum come from the addend and the
carries alone, single and batched, exact."""
import numpy as np
import pytest

from helpers import exact_product, int_to_words, words_to_int
from bluecrunch_amd.workload import operands

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("al,bl", [(6144, 6144), (8192, 8192), (9000, 7384), (12288, 12288), (14336, 14336),
                                   (30000, 19152), (106496, 106496), (3 << 19, 3 << 19)])
def test_outputs_past_a_full_class(bc, al, bl):
    plan = bc.plan(al, bl)
    assert 2 * plan["points"] * plan["bits"] == 32 * (al + bl), plan
    a, b = operands(al + 5 * bl, al, bl)
    a[-1] = b[-1] = 0xFFFFFFFF
    # the longest: against the product at its own length, which other tests pin
    prod = words_to_int(exact_product(a, b) if al < 200000 else bc.mul(a, b)[0])
    cls = [al + bl + more for more in (1, 2, 5000)]
    adds, want = [], []
    for n in cls:
        d = np.random.default_rng(n).integers(0, 2**32, n - 1, dtype=np.uint64).astype(np.uint32)
        d[al + bl - 3:] = 0xFFFFFFFF  # a carry out of the product's top word runs to the end
        adds.append(d)
        want.append(int_to_words((prod + words_to_int(d)) % (1 << (32 * n)), n))
    for n, d, w in zip(cls, adds, want):
        c, info = bc.muladd(a, b, d, n)
        assert info["passes"] > 1 and np.array_equal(c, w), n
        c, _ = bc.mul(a, b, cl=n)
        assert np.array_equal(c, int_to_words(prod, n)), n
    if al + bl < 100000:
        out, _ = bc.mul_batch([(a, b)] * 3, cls=cls, adds=adds)
        for c, w in zip(out, want):
            assert np.array_equal(c, w)

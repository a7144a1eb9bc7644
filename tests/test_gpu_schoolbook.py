"""Schoolbook products: one wave's and one workgroup's columns, operands staged
in LDS or not, outputs cut short and running past the product, long addends,
carries through every word, and outputs in place, each exact."""
import ctypes

import numpy as np
import pytest

from helpers import int_to_words, words_to_int
from bluecrunch_amd.workload import operands

pytestmark = pytest.mark.gpu

PAIRS = [(1, 1), (1, 98), (31, 33), (49, 50), (64, 35), (98, 1)]


@pytest.mark.parametrize("al,bl", PAIRS)
@pytest.mark.parametrize("extra", [-1, 0, 1, 29, 5000])
def test_short_products(bc, al, bl, extra):
    cl = max(1, al + bl + extra)
    ones = np.full(max(al, bl), 0xFFFFFFFF, dtype=np.uint32)
    for a, b in (operands(al * 100 + bl, al, bl), (ones[:al], ones[:bl])):
        x = words_to_int(a) * words_to_int(b)
        for dl in (0, 1, al, cl):
            d = np.full(dl, 0xFFFFFFFF, dtype=np.uint32)
            want = int_to_words((x + words_to_int(d)) % (1 << (32 * cl)), cl)
            assert np.array_equal(bc.muladd(a, b, d, cl)[0], want), dl
            out, _ = bc.mul_batch([(a, b)], cls=[cl], adds=[d])
            assert np.array_equal(out[0], want), dl


@pytest.mark.parametrize("al,bl", PAIRS + [(60, 68), (60, 69), (512, 512), (1000, 25), (2000, 2000), (1, 3999)])
def test_entry_point_and_in_place(bc, al, bl):
    a, b = operands(al * 7 + bl, al, bl)
    want = int_to_words(words_to_int(a) * words_to_int(b), al + bl)
    assert np.array_equal(bc.basecase(a, b), want)
    L = bc.lib()
    for first in (True, False):  # C == A, C == B
        dC = bc.DeviceWords(al + bl)
        own, other = (a, b) if first else (b, a)
        bc.check(L.bcg_memcpy_h2d(dC.ptr, own.ctypes.data, own.nbytes), "h2d")
        dO = bc.DeviceWords.from_host(other)
        pa, pb = (dC.ptr, dO.ptr) if first else (dO.ptr, dC.ptr)
        bc.check(L.bcg_basecase_dev(dC.ptr, al + bl, pa, al, pb, bl, None), "bcg_basecase_dev")
        assert np.array_equal(dC.to_host(), want)

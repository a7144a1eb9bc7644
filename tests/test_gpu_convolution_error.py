"""Error of a convolution through the transform calls (int_to_fft, two fft_forward,
fft_pointwise, fft_inverse) against the exact coefficients: root mean square over the
points, of the coefficients' own, mean of forty pairs of operands. The limits are the
means of the kernels with sixteen points per thread and passes of 64 rows, measured
over forty other pairs, and three of their standard errors."""
import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,bits,mean,err", [(3072, 12, 1.158e-16, 2.2e-18), (12288, 12, 1.255e-16, 2.1e-18),
                                             (24576, 12, 1.323e-16, 3.3e-18), (49152, 12, 1.348e-16, 1.8e-18),
                                             (98304, 11, 1.461e-16, 2.1e-18), (65536, 12, 2.011e-16, 5.5e-18)])
def test_convolution_error(bc, n, bits, mean, err):
    L = bc.lib()
    za, zb = bc.DeviceWords(4 * n), bc.DeviceWords(4 * n)
    pts = ctypes.c_size_t()
    w = n * bits // 64
    got = []
    for seed in range(40):
        rng = np.random.default_rng([n, seed])
        a, b = (rng.integers(0, 2**32, w, dtype=np.uint64).astype(np.uint32) for _ in range(2))
        digits = []
        for z, x in ((za, a), (zb, b)):
            d = bc.DeviceWords.from_host(x)
            bc.check(L.bcg_int_to_fft_dev(z.ptr, n, d.ptr, w, bits, ctypes.byref(pts), None), "int_to_fft")
            digits.append(z.to_host().view(np.float64)[::2].astype(np.longdouble))
        exact = np.rint(np.fft.irfft(np.fft.rfft(digits[0]) * np.fft.rfft(digits[1]), n)) * n
        bc.check(L.bcg_fft_forward_dev(za.ptr, n, None), "fft_forward")
        bc.check(L.bcg_fft_forward_dev(zb.ptr, n, None), "fft_forward")
        bc.check(L.bcg_fft_pointwise_dev(za.ptr, zb.ptr, n, None), "fft_pointwise")
        bc.check(L.bcg_fft_inverse_dev(za.ptr, n, None), "fft_inverse")
        z = za.to_host().view(np.float64).astype(np.longdouble)
        z[::2] -= exact
        got.append(float(np.sqrt(np.sum(z * z) / np.sum(exact * exact))))
    assert np.mean(got) <= mean + 3 * err, (n, np.mean(got))

"""Transforms whose values grow as far as the lazily reduced arithmetic inside
a pass lets them: inputs at the modulus (all r - 1, whose sums are the largest
a stage can form, and alternating 0 and r - 1, whose differences are), at every
size up to a full workgroup tile and the first ones of two passes, under each
tile size and register radix.  Exact against the oracle."""
import numpy as np
import pytest

import nkr_g16 as N
import pyoracle as O

pytestmark = pytest.mark.gpu

R_MINUS_1 = np.array([0x43E1F593F0000000, 0x2833E84879B97091, 0xB85045B68181585D, 0x30644E72E131A029], dtype=np.uint64)
LOGS = list(range(1, 14)) + [15]


def inputs(log_n):
    n = 1 << log_n
    top = np.tile(R_MINUS_1, (n, 1))
    alternating = top.copy()
    alternating[::2] = 0
    halves = top.copy()
    halves[n // 2 :] = 0
    return {"random": O.fr_random(7700 + log_n, n), "top": top, "alternating": alternating, "halves": halves}


@pytest.mark.parametrize("lds_log,radix_log", [(10, 2), (11, 2), (10, 3), (11, 3)])
def test_transforms_at_the_modulus(lds_log, radix_log):
    N._check(N.lib().nkr_ntt_set_shape(lds_log, radix_log, 1))
    try:
        for log_n in LOGS:
            for name, a in inputs(log_n).items():
                for kind in (N.FFT, N.IFFT, N.COSET_FFT, N.ICOSET_FFT):
                    assert np.array_equal(N.ntt(a, kind), O.fft(a, kind)), (log_n, name, kind)
    finally:
        N._check(N.lib().nkr_ntt_set_shape(11, 2, 1))


@pytest.mark.parametrize("log_n", [1, 2, 5, 10, 11, 12, 14])
@pytest.mark.parametrize("lds_log,radix_log", [(10, 3), (11, 2)])
def test_quotient_at_the_modulus(log_n, lds_log, radix_log):
    """The quotient chain runs the transposed (DIT) passes as well."""
    x = inputs(log_n)
    N._check(N.lib().nkr_ntt_set_shape(lds_log, radix_log, 1))
    try:
        for names in (("top", "top", "top"), ("alternating", "top", "halves"), ("random", "halves", "top")):
            a, b, c = (x[k] for k in names)
            assert np.array_equal(N.quotient(a, b, c), O.quotient(a, b, c)), names
    finally:
        N._check(N.lib().nkr_ntt_set_shape(11, 2, 1))

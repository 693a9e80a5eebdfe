"""The first transforms of a size (nkr_fr_ntt_dev builds and caches the size's
tables then) issued one right after the other on two streams: both equal the
oracle's.  The second stream is not ordered after the first, so the tables
have to be whole before either transform starts."""
import ctypes

import numpy as np
import pytest

import nkr_g16 as N
import pyoracle as O

pytestmark = pytest.mark.gpu

NON_BLOCKING = 1


def hip(name, *args):
    # the runtime the library itself is linked with
    assert getattr(N.lib(), name)(*args) == 0, name


@pytest.mark.parametrize("log_n", [3, 11, 13, 17])
@pytest.mark.parametrize("kind", [N.FFT, N.ICOSET_FFT])
def test_first_calls_on_two_streams(log_n, kind):
    L = N.lib()
    n_bytes = 32 << log_n
    inputs = [O.fr_random(60 + i, 1 << log_n) for i in range(2)]
    data = [ctypes.c_void_p() for _ in inputs]
    streams = [ctypes.c_void_p() for _ in inputs]
    try:
        for a, d, s in zip(inputs, data, streams):
            N._check(L.nkr_dev_alloc(n_bytes, ctypes.byref(d)))
            N._check(L.nkr_memcpy_htod(d, N._p(a), n_bytes))
            hip("hipStreamCreateWithFlags", ctypes.byref(s), ctypes.c_uint(NON_BLOCKING))
        N._check(L.nkr_ntt_set_shape(11, 2, 1))  # drops the cached sizes
        for d, s in zip(data, streams):
            N._check(L.nkr_fr_ntt_dev(d, log_n, kind, s))
        N._check(L.nkr_device_synchronize())
        for a, d in zip(inputs, data):
            got = np.empty_like(a)
            N._check(L.nkr_memcpy_dtoh(N._p(got), d, n_bytes))
            assert np.array_equal(got, O.fft(a, kind)), (log_n, kind)
    finally:
        for d, s in zip(data, streams):
            if s:
                hip("hipStreamDestroy", s)
            if d:
                N._check(L.nkr_dev_free(d))

"""The first transforms of a size (nkr_fr_ntt_dev builds and caches the size's
tables then) issued one right after the other on two streams: both equal the
oracle's.  The second stream is not ordered after the first, so the tables
have to be whole before either transform starts."""
import numpy as np
import pytest

import nkr_g16 as N
import pyoracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("log_n", [3, 11, 13, 17])
@pytest.mark.parametrize("kind", [N.FFT, N.ICOSET_FFT])
def test_first_calls_on_two_streams(log_n, kind):
    import torch

    L = N.lib()
    inputs = [O.fr_random(60 + i, 1 << log_n) for i in range(2)]
    data = [torch.from_numpy(a.view(np.int64)).cuda() for a in inputs]
    streams = [torch.cuda.Stream() for _ in inputs]
    torch.cuda.synchronize()
    N._check(L.nkr_ntt_set_shape(11, 2, 1))  # drops the cached sizes
    for d, s in zip(data, streams):
        N._check(L.nkr_fr_ntt_dev(d.data_ptr(), log_n, kind, s.cuda_stream))
    torch.cuda.synchronize()
    for a, d in zip(inputs, data):
        assert np.array_equal(d.cpu().numpy().view(np.uint64), O.fft(a, kind)), (log_n, kind)

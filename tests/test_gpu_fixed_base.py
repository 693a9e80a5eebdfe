"""Fixed-base multiplication around the sizes where the number of threads per
scalar changes and where a workgroup's shared inversion has idle or zero
members, against the oracle's scalar multiplication (exact equality)."""
import numpy as np
import pytest

import nkr_g16 as N
import pyoracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("g2,n", [(False, 1), (False, 63), (False, 64), (False, 16384), (False, 16385), (False, 32769),
                                  (False, 65537), (True, 1), (True, 33), (True, 8192), (True, 8193), (True, 32769)])
def test_fixed_base_mul_sizes(g2, n):
    base = O.g2_generator() if g2 else O.g1_generator()
    k = O.fr_random(9000 + n, n)
    edge = [0, 1, 255, 256, O.R - 1, 1 << 248, (1 << 253) + 1]
    k[: min(n, len(edge))] = O.fr_array(edge[:n])
    k[n // 2] = 0
    k[n - 1] = O.fr_array([O.R - 2])[0] if n > 1 else k[0]
    got = N.fixed_base_mul(base, k, g2=g2)
    pick = np.unique(np.concatenate([np.arange(min(n, 40)), np.arange(max(0, n - 40), n),
                                     np.random.default_rng(n).integers(0, n, 60)]))
    mul, affine = (O.g2_mul, O.g2_to_affine) if g2 else (O.g1_mul, O.g1_to_affine)
    assert np.array_equal(got[pick], affine(mul(base, np.ascontiguousarray(k[pick]))))
    assert np.array_equal(got[n // 2], affine(mul(base, k[n // 2: n // 2 + 1]))[0])

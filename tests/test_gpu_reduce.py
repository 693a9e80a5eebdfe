"""The MSM bucket reduction (fold, completion, bit-plane tree), whose additions
are shared by groups of lanes: buckets whose partial sums are equal, opposite
or infinite, so that its additions double, cancel and pass operands through,
at entry counts around the fold limit and with several fold launches.  Every
term is +-k B for one base B, so the sum is (k times the signs' sum) B; the bar
is equality of the normalised point."""
import numpy as np
import pytest

import nkr_g16 as N
import pyoracle as O

pytestmark = pytest.mark.gpu


def words(x):
    return np.array(O.int_to_words(O.to_mont_int(x % O.R, O.R)), dtype=np.uint64)


@pytest.mark.parametrize("g2", [False, True], ids=["g1", "g2"])
@pytest.mark.parametrize("n,signs", [(1, "same"), (2, "same"), (2, "halves"), (63, "same"), (64, "halves"),
                                     (65, "same"), (257, "random"), (4096, "halves"), (4097, "same"),
                                     (70001, "random"), (300000, "same")])
def test_equal_and_opposite_partial_sums(g2, n, signs):
    mul = O.g2_mul if g2 else O.g1_mul
    affine = O.g2_to_affine if g2 else O.g1_to_affine
    base = affine(mul(O.g2_generator() if g2 else O.g1_generator(), words(0xB15E).reshape(1, 4)))[0]
    neg = affine(mul(base, words(-1).reshape(1, 4)))[0]
    s = np.ones(n, dtype=np.int64)
    if signs == "halves":
        s[n // 2:] = -1
    elif signs == "random":
        s = np.random.default_rng(n).choice([-1, 1], n)
    bases = np.where((s > 0)[:, None], base[None, :], neg[None, :])
    m = N.Msm(bases, g2=g2)
    for k in (1, 3, O.R - 2):  # one bucket; another; one bucket per window
        got = m.run(np.tile(words(k), (n, 1)))
        want = affine(mul(base, words(k * int(s.sum())).reshape(1, 4)))[0]
        assert np.array_equal(got, want), (n, signs, k)
    m.close()

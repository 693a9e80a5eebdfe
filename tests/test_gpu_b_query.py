"""bs1 and bs2 over the finite points of the B query: a schedule of their own
where at most three quarters of the variables occur in B, the witness schedule
otherwise.  Plain and batched proofs against the oracle for a B with few
variables, with all of them (A and B exchanged), and with none."""
import numpy as np
import pytest

import circuits as C
import nkr_g16 as N
import pyoracle as O

pytestmark = pytest.mark.gpu


def no_b(circ):
    return np.zeros(circ.rows + 1, dtype=np.uint32), np.zeros(0, dtype=np.uint32), np.zeros((0, 4), dtype=np.uint64)


@pytest.mark.parametrize("kind", ["few", "all", "none"])
@pytest.mark.parametrize("size", [2, 15])  # 15: 4051 of 4096 columns in use, 3601 of them in A
def test_b_query_schedules(size, kind):
    circ = C.matmul(size, 77 + size, wide=True)
    if kind == "all":
        circ.a, circ.b = circ.b, circ.a
    elif kind == "none":
        circ.b = no_b(circ)
    keys = N.setup(circ, C.random_scalars(5, 99))
    finite = int((keys.b_g1_query.reshape(-1, 12)[:, 8:] != 0).any(axis=1).sum())
    assert (finite > circ.cols - circ.cols // 4) == (kind == "all" and size == 15)
    pv = N.Prover(circ, keys)
    rs = C.random_scalars(2, 5)
    want = O.prove_mt(circ, keys, circ.witness)
    want = np.concatenate([O.g1_to_affine(want[:48].reshape(4, 12)).reshape(-1), O.g2_to_affine(want[48:])[0]])
    raw, proof = pv.prove_blind(circ.witness, rs[0], rs[1])
    assert np.array_equal(raw, want)
    batch = N.Batch()
    for _ in range(3):  # eager, captured, replayed
        for got_raw, got_proof in batch.prove([(pv, circ.witness, rs[0], rs[1])] * 2):
            assert np.array_equal(got_raw, want) and np.array_equal(got_proof, proof)
    batch.close()
    pv.close()

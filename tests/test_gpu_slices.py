"""Column slices per XCD (slices_for in csrc/tf_rows.h) on a graph with a few rows of more than 32 entries: the short rows keep the
oracle's bits, the long ones' chunks, a workgroup each beside them, agree with float64."""
import numpy as np
import pytest
import scipy.sparse as sp

from test_gpu_parity import oracle_spmm_spmm, say

pytestmark = pytest.mark.gpu


# rows: the fewest that are cut into slices for the width; long: rows of one chunk, of one entry more than 32, of several chunks
@pytest.mark.parametrize("rows,N", [(16000, 128), (16003, 100), (16003, 97), (24001, 64), (24001, 49)])
def test_slices_beside_long_rows(gpu, tf, orc, rows, N):
    say(f"slices beside long rows, {rows} rows, N={N}")
    rng = np.random.default_rng(41)
    long = {5: 33, 4000: 1024, 9001: 1025, 15999: 5000}
    count = rng.integers(0, 20, rows)
    for r, n in long.items():
        count[r] = n
    ptr = np.concatenate([[0], np.cumsum(count)]).astype(np.int32)
    idx = np.concatenate([np.sort(rng.choice(rows, n, replace=False)) for n in count]).astype(np.int32)
    A = sp.csr_matrix((rng.uniform(-1, 1, len(idx)).astype(np.float32), idx, ptr), shape=(rows, rows))
    Ah = tf.CsrMatrix.from_scipy(A)
    Cd = tf.workloads.uniform((rows, N), 42)
    D0 = tf.workloads.uniform((rows, N), 43)
    S = tf.inspector(Ah, 1, op=tf.OP_SPMM_SPMM, N=N, inner=Ah)
    S.validate()
    assert S.info()["marched"] == 0 and S.info()["windowed"] == 0
    A64 = A.astype(np.float64)
    T = A64 @ Cd.astype(np.float64)
    want = A64 @ T
    size = abs(A64) @ (abs(A64) @ abs(Cd.astype(np.float64)))
    for acc in (False, True):
        D = tf.DenseMatrix(rows, N, D0) if acc else tf.DenseMatrix(rows, N)
        tf.spmm_spmm(Ah, Ah, tf.DenseMatrix.from_numpy(Cd), D, S, accumulate=acc)
        tf.device_synchronize()
        got = D.to_numpy().astype(np.float64) - (D0 if acc else 0)
        # two sums of up to 5,000 terms in fp32, in any order: 2 x 5,000 roundings of 2^-24 of the magnitudes, and the added D0's own
        assert (abs(got - want) <= 2 * 5000 * 2.0 ** -24 * size + 2.0 ** -23 * (1 + abs(want))).all(), (rows, N, acc)
    # rows whose own and whose columns' sums are of 32 entries and less: the oracle's bits
    D = tf.DenseMatrix(rows, N)
    tf.spmm_spmm(Ah, Ah, tf.DenseMatrix.from_numpy(Cd), D, S)
    tf.device_synchronize()
    short = np.ones(rows, bool)
    short[list(long)] = False
    bad = np.zeros(rows, bool)
    bad[list(long)] = True
    short &= np.asarray((abs(A) @ bad.astype(np.float32)) == 0).ravel()
    assert short.sum() > rows // 2
    assert np.array_equal(D.to_numpy()[short], oracle_spmm_spmm(orc, A, A, Cd)[short])

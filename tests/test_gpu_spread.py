"""Row products of graphs whose entries are spread over all columns (sweep_rows_kernel, sweep_for in csrc/tf_rows.h): the sums are added in the row's
order whatever the limit lets through, so both products of a two-hop call have the oracle's bits."""
import numpy as np
import pytest
import scipy.sparse as sp

from test_gpu_parity import oracle_spmm_spmm, say

pytestmark = pytest.mark.gpu


# rows: a little more than 15 MB of X for the width (20 for 128), at the edges of a workgroup's rows; N: every number of lanes, slices of 32 and of 64 columns, rows
# that do not start at a line, a last lane that reaches back (97: into the slice before it).  Row lengths around the 16 entries that
# are kept in LDS, none, and as many as a row in one piece may have; one row reads one column many times, one reads the last columns only.
@pytest.mark.parametrize("rows,N", [(39104, 128), (84001, 128), (38703, 97), (37502, 100), (58602, 64), (76531, 49), (113641, 33), (117249, 32),
                                    (220601, 17), (234385, 16), (340910, 11), (140001, 128)])
def test_spread_rows(gpu, tf, orc, rows, N):
    say(f"spread rows, {rows} rows, N={N}")
    rng = np.random.default_rng(51)
    count = rng.poisson(6, rows).clip(0, 30)
    special = {0: 128, 1: 0, 2: 16, 3: 17, 40: 15, 41: 32, 42: 33, 1000: 127, rows - 1: 48, rows - 2: 0}
    for r, n in special.items():
        count[r] = n
    ptr = np.concatenate([[0], np.cumsum(count)]).astype(np.int32)
    idx = rng.integers(0, rows, ptr[-1]).astype(np.int64)
    idx[ptr[2]:ptr[3]] = rows - 1 - np.arange(16)
    key = np.repeat(np.arange(rows, dtype=np.int64), count) * rows + idx
    idx = (np.sort(key) % rows).astype(np.int32)
    idx[ptr[41]:ptr[42]] = 7
    idx[ptr[42]:ptr[43]] = idx[ptr[42]:ptr[43]][::-1]  # (columns that fall: slower, the same sums)
    val = rng.uniform(-1, 1, len(idx)).astype(np.float32)
    A = sp.csr_matrix((val, idx, ptr), shape=(rows, rows))
    Ah = tf.CsrMatrix(rows, rows, ptr, idx, val)
    S = tf.inspector(Ah, 1, op=tf.OP_SPMM_SPMM, N=N, inner=Ah)
    S.validate()
    assert S.info()["n_long_rows"] == 0
    Cd = tf.workloads.uniform((rows, N), 52)
    want = oracle_spmm_spmm(orc, A, A, Cd)
    Ch = tf.DenseMatrix.from_numpy(Cd)
    D = tf.DenseMatrix(rows, N)
    S.set_profiling(True)
    tf.spmm_spmm(Ah, Ah, Ch, D, S)
    tf.device_synchronize()
    assert np.array_equal(D.to_numpy(), want)
    assert [n for n, _ in S.profile()] == ["sweep_rows_kernel"] * 2
    D0 = tf.workloads.uniform((rows, N), 53)
    D = tf.DenseMatrix(rows, N, D0)
    tf.spmm_spmm(Ah, Ah, Ch, D, S, accumulate=True)
    tf.device_synchronize()
    # the sum starts at D0 instead of at zero: a row's roundings, each of 2^-24 of a partial sum below |D0| and the magnitudes
    size = abs(A) @ abs(A @ Cd.astype(np.float64)) + abs(D0)
    assert (abs(D.to_numpy() - (want + D0.astype(np.float64))) <= 2 * 129 * 2.0 ** -24 * size).all()


def test_infinities_of_other_rows_stay_out(gpu, tf):
    """A row's gather that the limit holds back reads nothing: an infinity in X or among the values is in the sums of the rows it belongs to."""
    rows, N = 60001, 64
    rng = np.random.default_rng(54)
    count = rng.integers(4, 10, rows)
    ptr = np.concatenate([[0], np.cumsum(count)]).astype(np.int32)
    key = np.repeat(np.arange(rows, dtype=np.int64), count) * rows + rng.integers(0, rows, ptr[-1])
    idx = (np.sort(key) % rows).astype(np.int32)
    val = rng.uniform(0.5, 1, len(idx)).astype(np.float32)
    val[ptr[100]] = np.inf
    X = rng.uniform(0.5, 1, (rows, N)).astype(np.float32)
    X[0, 3], X[rows - 1, 60], X[777] = np.inf, np.nan, -np.inf
    Ah = tf.CsrMatrix(rows, rows, ptr, idx, val)
    S = tf.inspector(Ah, 1, op=tf.OP_SPMM_SPMM, N=N, inner=Ah)
    D = tf.DenseMatrix(rows, N)
    tf.spmm_spmm(Ah, Ah, tf.DenseMatrix.from_numpy(X), D, S)
    tf.device_synchronize()
    A = sp.csr_matrix((val.astype(np.float64), idx, ptr), shape=(rows, rows))
    with np.errstate(invalid="ignore"):
        want = A @ (A @ X.astype(np.float64))
    got = D.to_numpy()
    assert np.array_equal(np.isnan(got), np.isnan(want)) and np.array_equal(np.isposinf(got), np.isposinf(want)) and np.array_equal(np.isneginf(got), np.isneginf(want))
    fine = np.isfinite(want)
    assert fine.mean() > 0.9 and (abs(got - want)[fine] <= 2 * 11 * 2.0 ** -24 * want[fine] * 2).all()

"""Row products of graphs whose entries are spread over all columns (sweep_rows_kernel, sweep_for in csrc/tf_rows.h): the sums are added in the row's
order whatever the limit lets through, so both products of a two-hop call have the oracle's bits."""
import ctypes as C

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
    assert fine.mean() > 0.9 and (abs(got[fine] - want[fine]) <= 2 * 11 * 2.0 ** -24 * want[fine] * 2).all()


def spread(rows, cols, mean, seed):
    """Rows of `mean` entries and a few more or less, anywhere; signs of both kinds."""
    rng = np.random.default_rng(seed)
    ptr = np.concatenate([[0], np.cumsum(rng.integers(mean - 3, mean + 4, rows))]).astype(np.int32)
    key = np.unique(np.repeat(np.arange(rows, dtype=np.int64), np.diff(ptr)) * cols + rng.integers(0, cols, ptr[-1]))
    ptr = np.searchsorted(key, np.arange(rows + 1, dtype=np.int64) * cols).astype(np.int32)
    return sp.csr_matrix((rng.uniform(-1, 1, len(key)).astype(np.float32), (key % cols).astype(np.int32), ptr), shape=(rows, cols))


def roundings(A, X, extra=0.0):
    """Within the roundings of a row's sum: 2^-24 of the magnitudes, once an entry and a product."""
    size = abs(A).astype(np.float64) @ abs(X.astype(np.float64)) + abs(extra)
    return size * (2.0 ** -24 * 2 * (int(np.diff(A.indptr).max()) + 2))


# rows and columns: as many, more of either; N: slices, whole rows at a line and anywhere
@pytest.mark.parametrize("rows,cols,N", [(60001, 60001, 64), (41000, 70003, 100), (90001, 40000, 128), (52000, 130001, 30)])
@pytest.mark.parametrize("relu", [False, True])
def test_spread_row_products(gpu, tf, rows, cols, N, relu):
    """One product of a schedule of its own, square and not, with a ReLU, onto what Y holds, and with values that change between calls."""
    say(f"spread row products {rows} x {cols}, N={N}, relu={relu}")
    A = spread(rows, cols, 9, 55)
    X = tf.workloads.uniform((cols, N), 56)
    Y0 = tf.workloads.uniform((rows, N), 57)
    Ah = tf.CsrMatrix.from_scipy(A)
    h = C.c_void_p()
    assert tf.lib().tf_inspect_spmm(rows, cols, Ah._pp, Ah._pi, N, 0, C.byref(h)) == 0
    S = tf.FusedSchedule(h, Ah)
    S.set_profiling(True)
    own = [tf.DenseMatrix.from_numpy(np.ascontiguousarray(x).view(np.float32).reshape(1, -1)) for x in (A.indptr, A.indices, A.data)]
    Aw = tf.CsrMatrix.wrap_device(Ah, *(x.device_ptr() for x in own))
    Xd = tf.DenseMatrix.from_numpy(X)
    for step, M in enumerate((Ah, Aw, Aw)):
        if step == 2:
            A.data = np.random.default_rng(58).uniform(-1, 1, A.nnz).astype(np.float32)
            own[2].copy_from(tf.DenseMatrix.from_numpy(A.data.reshape(1, -1)))
        want = A.astype(np.float64) @ X.astype(np.float64)
        for acc in (False, True):
            Y = tf.DenseMatrix(rows, N, Y0)
            assert tf.lib().tf_spmm_scheduled(M.to_device().h, Xd.h, Y.h, S.h, (4 if relu else 0) | (1 if acc else 0), None) == 0
            tf.device_synchronize()
            assert [n for n, _ in S.profile()] == ["sweep_rows_kernel"]
            ref = want + Y0 if acc else want
            if relu:
                ref = np.maximum(ref, 0)
            assert (abs(Y.to_numpy() - ref) <= roundings(A, X, Y0 if acc else 0.0)).all(), (step, acc)


@pytest.mark.parametrize("rows,cols,K,N", [(60001, 60001, 96, 64), (50000, 61007, 130, 100), (80003, 44000, 160, 128)])
def test_spread_gemm_spmm(gpu, tf, rows, cols, K, N):
    """A layer on such a graph: the dense product, then the rows out of it; square and not, with a ReLU, onto what D holds."""
    say(f"spread layer {rows} x {cols}, {K} -> {N}")
    A = spread(rows, cols, 10, 61)
    rng = np.random.default_rng(62)
    X, W = rng.uniform(0, 1, (cols, K)).astype(np.float32), rng.uniform(-1, 1, (K, N)).astype(np.float32)
    D0 = tf.workloads.uniform((rows, N), 63)
    Ah = tf.CsrMatrix.from_scipy(A)
    S = tf.inspector(Ah, 1, op=tf.OP_GEMM_SPMM, N=N, K=K)
    S.set_profiling(True)
    T = X.astype(np.float64) @ W.astype(np.float64)
    want = A.astype(np.float64) @ T
    # (the product's own roundings: K terms of magnitudes |X| |W|, each as good as an fp32 sum's)
    allowed = (abs(A).astype(np.float64) @ (X.astype(np.float64) @ abs(W.astype(np.float64))) + abs(D0)) * (2.0 ** -24 * 2 * (K + 24))
    for flags in (0, 4, 1, 5):
        D = tf.DenseMatrix(rows, N, D0)
        assert tf.lib().tf_gemm_spmm(Ah.to_device().h, tf.DenseMatrix.from_numpy(X).h, tf.DenseMatrix.from_numpy(W).h, D.h, S.h, flags, None) == 0
        tf.device_synchronize()
        assert [n for n, _ in S.profile()][-1] == "sweep_rows_kernel" and len(S.profile()) == 2, S.profile()
        ref = want + D0 if flags & 1 else want
        if flags & 4:
            ref = np.maximum(ref, 0)
        assert (abs(D.to_numpy() - ref) <= allowed).all(), flags

"""The dense products beside the executors (Y = X W in any shape and storage of W, the gradient of a layer's weights) and the
scheduled row product, at the sizes where their kernels change hands or have remainders, against float64."""
import ctypes as C

import numpy as np
import pytest
import scipy.sparse as sp

pytestmark = pytest.mark.gpu
RELU, C_TRANSPOSED = 4, 16


def say(*a):
    print(*a, flush=True)


def rel(got, want):
    return float(np.abs(got - want).max() / max(np.abs(want).max(), 1e-30))


@pytest.mark.parametrize("M,K,N", [(1, 1, 1), (15, 16, 3), (17, 33, 16), (64, 500, 32), (3000, 500, 32), (3000, 7, 41), (1000, 300, 64),
                                   (70000, 20, 7), (5000, 251, 130), (40000, 64, 300), (777, 1433, 64)])
@pytest.mark.parametrize("w_t", [False, True])
def test_gemm_of_any_shape(gpu, tf, M, K, N, w_t):
    say(f"gemm {M} x {K} x {N} w_t={w_t}")
    rng = np.random.default_rng(M + 7 * K + 13 * N)
    X, W, m = (rng.uniform(-1, 1, s).astype(np.float32) for s in ((M, K), (K, N), (M, N)))
    Xd, Wd = tf.DenseMatrix.from_numpy(X), tf.DenseMatrix.from_numpy(np.ascontiguousarray(W.T) if w_t else W)
    want = X.astype(np.float64) @ W.astype(np.float64)
    for mask in (None, m):
        Y = tf.DenseMatrix.from_numpy(np.full((M, N), np.nan, np.float32))
        md = tf.DenseMatrix.from_numpy(mask) if mask is not None else None
        assert tf.lib().tf_gemm_ex(Xd.h, Wd.h, Y.h, md.h if md else None, C_TRANSPOSED if w_t else 0, None) == 0
        tf.device_synchronize()
        ref = want if mask is None else np.where(mask > 0, want, 0.0)
        assert rel(Y.to_numpy(), ref) <= 1e-5, (mask is not None)


@pytest.mark.parametrize("M,K,N", [(13001, 4, 33), (12999, 17, 64), (20481, 18, 17), (13007, 19, 129), (13001, 66, 97), (262145, 131, 35), (40000, 100, 100),
                                   (13000, 5, 257), (262145, 8, 32), (262144, 16, 64), (262143, 15, 33), (66000, 17, 40), (20479, 16, 31), (20480, 4, 17)])
def test_gemm_panel_edges(gpu, tf, M, K, N):
    """W in LDS: steps of k that end after one to four values, a last lane whose columns overlap its neighbour's, rows and panels
    that end early; non-finite values beside the edges stay where they are."""
    say(f"gemm panel {M} x {K} x {N}")
    rng = np.random.default_rng(M + K + N)
    X, W = (rng.uniform(-1, 1, s).astype(np.float32) for s in ((M, K), (K, N)))
    X[M - 2, K - 1] = np.inf
    m = rng.uniform(-1, 1, (M, N)).astype(np.float32)
    Xd, md = tf.DenseMatrix.from_numpy(X), tf.DenseMatrix.from_numpy(m)
    with np.errstate(invalid="ignore"):
        want = X.astype(np.float64) @ W.astype(np.float64)
    ok = np.arange(M) != M - 2
    for w_t in (False, True):
        Wd = tf.DenseMatrix.from_numpy(np.ascontiguousarray(W.T) if w_t else W)
        for mask in (None, md):
            Y = tf.DenseMatrix.from_numpy(np.full((M, N), np.nan, np.float32))
            assert tf.lib().tf_gemm_ex(Xd.h, Wd.h, Y.h, mask.h if mask else None, C_TRANSPOSED if w_t else 0, None) == 0
            tf.device_synchronize()
            got, ref = Y.to_numpy(), want if mask is None else np.where(m > 0, want, 0.0)
            assert rel(got[ok], ref[ok]) <= 1e-5
            assert np.array_equal(np.isinf(got[~ok]), np.isinf(ref[~ok]))


@pytest.mark.parametrize("M,K,N", [(18432, 4, 65), (18431, 4, 65), (18433, 31, 66), (24001, 33, 65), (24000, 51, 96), (18447, 64, 97), (50000, 65, 128),
                                   (30001, 128, 128), (18437, 161, 72), (18439, 213, 128), (10241, 214, 129), (10239, 214, 129), (10240, 300, 100),
                                   (10243, 426, 65), (18434, 427, 65), (38400, 64, 33), (38399, 64, 33), (38409, 96, 48), (49999, 130, 64),
                                   (38403, 427, 40), (38401, 853, 36), (38402, 854, 36), (262145, 67, 35),
                                   (18434, 16, 70), (18435, 17, 70), (38405, 48, 33), (38405, 49, 33), (38401, 63, 64),
                                   (18433, 192, 128), (18433, 193, 128), (18435, 256, 96), (18435, 257, 96), (18434, 416, 68), (18434, 417, 68),
                                   (18434, 415, 126), (38403, 416, 33), (38403, 416, 64), (38401, 417, 36)])
@pytest.mark.parametrize("w_t", [False, True])
def test_gemm_on_bf16_cores(gpu, tf, M, K, N, w_t):
    """Products as sums of bf16 parts, either side of where they begin and of what LDS holds (192 values of k for a panel of 128 columns, 256 for 96, 416 for
    64): within the bound of fp32 sums around float64, for operands of one size and of many sizes; infinities, NaN and values that bf16
    rounds to infinity stay in their rows, and come out as fp32 arithmetic has them."""
    say(f"gemm on bf16 cores {M} x {K} x {N} w_t={w_t}")
    rng = np.random.default_rng(M + 3 * K + 5 * N)
    W = rng.uniform(-0.2, 0.2, (K, N)).astype(np.float32)
    Wd = tf.DenseMatrix.from_numpy(np.ascontiguousarray(W.T) if w_t else W)
    flags = C_TRANSPOSED if w_t else 0
    big = np.float32(3.4e38)  # rounds to infinity in bf16
    for spread in (0.0, 20.0):
        X = (rng.uniform(-1, 1, (M, K)) * np.exp2(rng.uniform(-spread, spread, (M, K)))).astype(np.float32)
        X[1, K - 1], X[M - 1, 0], X[M // 2, 0], X[M - 2, K // 2] = np.inf, np.nan, big, -np.inf
        odd = np.zeros(M, bool)
        odd[[1, M - 1, M // 2, M - 2]] = True
        Xd, Y = tf.DenseMatrix.from_numpy(X), tf.DenseMatrix.from_numpy(np.full((M, N), 7.0, np.float32))
        assert tf.lib().tf_gemm_ex(Xd.h, Wd.h, Y.h, None, flags, None) == 0
        tf.device_synchronize()
        got = Y.to_numpy()
        with np.errstate(invalid="ignore", over="ignore"):
            want = X.astype(np.float64) @ W.astype(np.float64)
            size = np.abs(X[~odd]).astype(np.float64) @ np.abs(W).astype(np.float64)
        # K roundings of partial sums, each below the sum of magnitudes
        assert np.all(np.abs(got[~odd] - want[~odd]) <= (K + 8) * 2.0 ** -24 * size)
        assert np.array_equal(np.isnan(got[odd]), np.isnan(want[odd]))
        assert np.array_equal(np.sign(got[[1, M - 2]]), np.sign(want[[1, M - 2]])) and np.all(np.isinf(got[[1, M - 2]]))
        assert np.all(np.abs(got[M // 2] - want[M // 2]) <= (K + 8) * 2.0 ** -24 * np.abs(want[M // 2]).max())


def few_values(rng, M, K, q):
    """Rows of q values at random places (all K where q is K), the rest zeros: what bag-of-words features are."""
    X = rng.uniform(-1, 1, (M, K)).astype(np.float32)
    if q < K:
        keep = np.zeros((M, K), bool)
        np.put_along_axis(keep, np.argsort(rng.random((M, K)), axis=1)[:, :q], True, 1)
        X[~keep] = 0
    return X


def fp32_sums(X, W):
    """X W as a chain of fp32 fmas, each rounded to nearest."""
    s = np.zeros((X.shape[0], W.shape[1]), np.float32)
    for k in range(X.shape[1]):
        s = (s + X[:, k:k + 1].astype(np.float64) * W[k].astype(np.float64)).astype(np.float32)
    return s


def no_further_than_fp32(got, X, W, q):
    """The error against float64 over the sum of magnitudes: its root mean square is at most that of fp32 sums; one product is rounded once, and sums of more
    lose less than 2^-23 of themselves with every further value and are rounded once at the end.  (2^-6 for what is left out and for second roundings.)"""
    def error(y, X):
        size = np.abs(X).astype(np.float64) @ np.abs(W).astype(np.float64)
        e = np.abs(y - X.astype(np.float64) @ W.astype(np.float64)) / np.maximum(size, 1e-300)
        return e[size > 0]
    e, part = error(got, X), slice(0, 6000)
    fp32 = error(fp32_sums(X[part], W), X[part])
    print(f"  {q} values: largest {e.max():.3g} ({fp32.max():.3g}), rms {np.sqrt((e ** 2).mean()):.4g} ({np.sqrt((fp32 ** 2).mean()):.4g})", flush=True)
    assert np.sqrt((e ** 2).mean()) <= 1.02 * np.sqrt((fp32 ** 2).mean())  # (two samples of some 400,000 values or more: 0.3 %)
    assert e.max() <= (2 * q - 1) * 2.0 ** -24 * (1 + 2.0 ** -6)


@pytest.mark.parametrize("M,K,N", [(18433, 128, 128), (40000, 64, 64), (30000, 301, 100)])
@pytest.mark.parametrize("q", [1, 2, 3, 4, 8, 64])
def test_gemm_of_few_features_a_row(gpu, tf, M, K, N, q):
    say(f"gemm of rows of few features {M} x {K} x {N}, {q} a row")
    rng = np.random.default_rng(M + K + q)
    X, W = few_values(rng, M, K, q), rng.uniform(-1, 1, (K, N)).astype(np.float32)
    Xd, Wd, Y = tf.DenseMatrix.from_numpy(X), tf.DenseMatrix.from_numpy(W), tf.DenseMatrix(M, N)
    assert tf.lib().tf_gemm_ex(Xd.h, Wd.h, Y.h, None, 0, None) == 0
    tf.device_synchronize()
    no_further_than_fp32(Y.to_numpy(), X, W, q)


@pytest.mark.parametrize("small", [-148, -140, -125, -110])
@pytest.mark.parametrize("what", ["gemm", "gemm weights", "streamed", "weight gradient"])
def test_small_operands_on_bf16_cores(gpu, tf, what, small):
    """Values of 2^small, denormal ones among them, times values whose products are normal floats: as precise as any others; and times values that leave
    the results denormal, to their last place."""
    say(f"small operands {what} 2^{small}")
    rng = np.random.default_rng(-small)
    M, K, N = 25000, 96, 72
    lib = tf.lib()
    for other in (35, -4):
        # sums and differences of the smallest floats: what counts is kept whole by the first rounding, to fp32
        tiny = lambda m, n: (rng.uniform(-1, 1, (m, n)) * 2.0 ** small).astype(np.float32)
        X = tiny(M, K) if what != "gemm weights" else rng.uniform(-1, 1, (M, K)).astype(np.float32) * np.float32(2.0 ** other)
        if what == "weight gradient":
            G, Y = (rng.uniform(-1, 1, (M, N)) * 2.0 ** other).astype(np.float32), tf.DenseMatrix(N, K)
            ws = tf.DenseMatrix(1, max(1, lib.tf_weight_grad_workspace(M, N, K) // 4))
            Gd, Xd = tf.DenseMatrix.from_numpy(G), tf.DenseMatrix.from_numpy(X)
            assert lib.tf_weight_grad(Gd.h, Xd.h, Y.h, C.c_void_p(ws.device_ptr()), None) == 0
            a, b, terms = G.T, X, 300
        else:
            W = tiny(K, N) if what == "gemm weights" else (rng.uniform(-1, 1, (K, N)) * 2.0 ** other).astype(np.float32)
            Xd, Wd, Y = tf.DenseMatrix.from_numpy(X), tf.DenseMatrix.from_numpy(W), tf.DenseMatrix(M, N)
            if what == "streamed":
                Ah = tf.CsrMatrix.from_scipy(sp.identity(M, dtype=np.float32, format="csr"))
                S = tf.inspector(Ah, op=tf.OP_GEMM_SPMM, N=N, K=K, lds_budget_bytes=163840)
                assert S.info()["streamed"] == 1
                tf.gemm_spmm(Ah.to_device(), Xd, Wd, Y, S)
            else:
                assert lib.tf_gemm_ex(Xd.h, Wd.h, Y.h, None, 0, None) == 0
            a, b, terms = X, W, K + 8
        tf.device_synchronize()
        a, b = a.astype(np.float64), b.astype(np.float64)
        # roundings of sums, each below the sum of magnitudes, or half a place of the smallest float where a group's sum is denormal
        bound = terms * 2.0 ** -24 * (np.abs(a) @ np.abs(b)) + 600 * 2.0 ** -150
        assert np.all(np.abs(Y.to_numpy() - a @ b) <= bound), (what, small, other)


@pytest.mark.parametrize("K,N", [(128, 128), (120, 96), (64, 64), (40, 32), (136, 32), (256, 64), (256, 128)])
def test_streamed_runs_on_bf16_cores(gpu, tf, K, N):
    """Banded rows whose intermediate never leaves LDS: within fp32's rounding of float64, values of many sizes, and what is not finite
    stays with the rows that read it."""
    say(f"streamed runs {K} x {N}")
    rng = np.random.default_rng(K + N)
    M, width, n = 26001, 24, 7
    cols = np.clip(np.arange(M)[:, None] + np.sort(np.argsort(rng.random((M, width)), axis=1)[:, :n], axis=1) - width // 2, 0, M - 1)
    A = sp.csr_matrix((rng.uniform(-1, 1, M * n).astype(np.float32), cols.ravel(), np.arange(M + 1) * n), shape=(M, M))
    A.sum_duplicates()
    A.sort_indices()
    B = (rng.uniform(-1, 1, (M, K)) * np.exp2(rng.uniform(-20, 20, (M, K)))).astype(np.float32)
    W = rng.uniform(-0.2, 0.2, (K, N)).astype(np.float32)
    B[0, K - 1], B[M - 1, 0], B[M // 2, 5] = np.inf, np.nan, 3.4e38
    read = np.zeros(M, bool)
    read[[0, M - 1, M // 2]] = True
    odd = (A != 0).astype(np.float32) @ read.astype(np.float32) > 0
    Ah = tf.CsrMatrix.from_scipy(A)
    S = tf.inspector(Ah, op=tf.OP_GEMM_SPMM, N=N, K=K, lds_budget_bytes=163840)  # (a given budget: tiles, never two products)
    assert S.info()["streamed"] == 1
    D, Bd, Wd = tf.DenseMatrix(M, N), tf.DenseMatrix.from_numpy(B), tf.DenseMatrix.from_numpy(W)
    tf.gemm_spmm(Ah.to_device(), Bd, Wd, D, S)
    tf.device_synchronize()
    got = D.to_numpy()
    with np.errstate(invalid="ignore", over="ignore"):
        want = A.astype(np.float64) @ (B.astype(np.float64) @ W.astype(np.float64))
    size = abs(A).astype(np.float64) @ (np.where(np.isfinite(B), np.abs(B), 0).astype(np.float64) @ np.abs(W).astype(np.float64))
    assert np.all(np.abs(got[~odd] - want[~odd]) <= (K + n + 8) * 2.0 ** -24 * size[~odd])
    assert np.array_equal(np.isnan(got[odd]), np.isnan(want[odd])) and not odd.all() and odd.sum() >= 3


@pytest.mark.parametrize("K,N", [(128, 128), (120, 96), (64, 64), (40, 32), (128, 64), (64, 96), (256, 64), (256, 128), (200, 32), (136, 96)])
@pytest.mark.parametrize("q", [1, 2, 4, 8, 64])
def test_streamed_runs_of_few_features_a_row(gpu, tf, K, N, q):
    """The rows of the intermediate themselves (A is the identity)."""
    q = min(q, K)
    say(f"streamed runs of few features a row {K} x {N}, {q} a row")
    M = 25000
    rng = np.random.default_rng(K + N + q)
    X, W = few_values(rng, M, K, q), rng.uniform(-1, 1, (K, N)).astype(np.float32)
    Ah = tf.CsrMatrix.from_scipy(sp.identity(M, dtype=np.float32, format="csr"))
    S = tf.inspector(Ah, op=tf.OP_GEMM_SPMM, N=N, K=K, lds_budget_bytes=163840)
    assert S.info()["streamed"] == 1
    D, Xd, Wd = tf.DenseMatrix(M, N), tf.DenseMatrix.from_numpy(X), tf.DenseMatrix.from_numpy(W)
    tf.gemm_spmm(Ah.to_device(), Xd, Wd, D, S)
    tf.device_synchronize()
    no_further_than_fp32(D.to_numpy(), X, W, q)


@pytest.mark.parametrize("K,N", [(129, 33), (64, 100), (18, 128)])
def test_gemm_of_listed_rows(gpu, tf, K, N):
    """The rows an R-MAT graph reads, gathered by the product itself and stored in the order of their reads."""
    say(f"listed rows {K} x {N}")
    A = tf.workloads.rmat(15, 8 << 15, seed=5)
    M = A.shape[0]
    rng = np.random.default_rng(K)
    X, W = (rng.uniform(-1, 1, s).astype(np.float32) for s in ((M, K), (K, N)))
    Ah = tf.CsrMatrix.from_scipy(A)
    S = tf.inspector(Ah, op=tf.OP_GEMM_SPMM, N=N, K=K)
    D = tf.DenseMatrix(M, N)
    Xd, Wd = tf.DenseMatrix.from_numpy(X), tf.DenseMatrix.from_numpy(W)
    assert tf.lib().tf_gemm_spmm(Ah.to_device().h, Xd.h, Wd.h, D.h, S.h, 0, None) == 0
    tf.device_synchronize()
    assert rel(D.to_numpy(), A.astype(np.float64) @ (X.astype(np.float64) @ W.astype(np.float64))) <= 1e-5


@pytest.mark.parametrize("K,N", [(131, 101), (257, 70), (80, 97)])
def test_gemm_of_listed_rows_on_bf16_cores(gpu, tf, K, N):
    """The same with rows enough for the bf16 cores: every read row of a larger graph, K and N no multiples of four, one row that is not finite."""
    say(f"gemm of many listed rows {K} x {N}")
    rng = np.random.default_rng(K * N)
    A = tf.workloads.rmat(16, 8 << 16, seed=5)
    M = A.shape[0]
    read = np.flatnonzero(np.bincount(A.indices, minlength=M))
    assert 72 * 256 <= read.size < M  # (rows that nothing reads: the product takes a list)
    B, W = rng.uniform(-1, 1, (M, K)).astype(np.float32), rng.uniform(-1, 1, (K, N)).astype(np.float32)
    row = read[read.size // 2]
    Ah = tf.CsrMatrix.from_scipy(A)
    S = tf.inspector(Ah, op=tf.OP_GEMM_SPMM, N=N, K=K)
    Bf = B.astype(np.float64)
    for bad in (None, np.inf):
        if bad is not None:
            B[row, K - 1] = bad
        D, Bd, Wd = tf.DenseMatrix(M, N), tf.DenseMatrix.from_numpy(B), tf.DenseMatrix.from_numpy(W)
        tf.gemm_spmm(Ah.to_device(), Bd, Wd, D, S)
        tf.device_synchronize()
        got, want = D.to_numpy(), A.astype(np.float64) @ (Bf @ W.astype(np.float64))
        hit = np.asarray((A[:, [row]] != 0).todense()).ravel() if bad is not None else np.zeros(M, bool)
        assert rel(got[~hit], want[~hit]) <= 1e-6  # (K products and a row's entries, each rounded once)
        assert not np.isfinite(got[hit]).any() and (bad is None or hit.any())


@pytest.mark.parametrize("M,N,K", [(1, 1, 1), (31, 7, 5), (33, 32, 128), (3000, 7, 32), (3000, 32, 500), (10000, 64, 300), (5001, 33, 161),
                                   (100000, 64, 128), (20011, 130, 31), (64, 300, 97), (4096, 65, 33), (4097, 31, 30)])
def test_weight_gradient(gpu, tf, M, N, K):
    say(f"weight gradient {M} rows, {N} x {K}")
    rng = np.random.default_rng(M + N + K)
    G, X = rng.uniform(-1, 1, (M, N)).astype(np.float32), rng.uniform(0, 1, (M, K)).astype(np.float32)
    Gd, Xd, Y = tf.DenseMatrix.from_numpy(G), tf.DenseMatrix.from_numpy(X), tf.DenseMatrix.from_numpy(np.full((N, K), np.nan, np.float32))
    lib = tf.lib()
    ws = tf.DenseMatrix(1, max(1, lib.tf_weight_grad_workspace(M, N, K) // 4))
    for _ in range(2):
        assert lib.tf_weight_grad(Gd.h, Xd.h, Y.h, C.c_void_p(ws.device_ptr()), None) == 0
    tf.device_synchronize()
    assert rel(Y.to_numpy(), G.astype(np.float64).T @ X.astype(np.float64)) <= 1e-5


@pytest.mark.parametrize("M,N,K", [(4097, 1, 1), (4100, 3, 2), (4128, 17, 48), (4129, 33, 49), (5000, 49, 65), (9999, 64, 64), (33000, 100, 20), (150001, 7, 129)])
def test_weight_gradient_on_bf16_cores(gpu, tf, M, N, K):
    """Every width of tile, last blocks of any number of rows: within fp32's rounding of float64 for values of many sizes; what is not
    finite stays in its row and column of the result."""
    say(f"weight gradient on bf16 cores {M} rows, {N} x {K}")
    rng = np.random.default_rng(M + N + K)
    G, X = ((rng.uniform(-1, 1, (M, w)) * np.exp2(rng.uniform(-8, 8, (M, w)))).astype(np.float32) for w in (N, K))
    lib = tf.lib()
    ws = tf.DenseMatrix(1, max(1, lib.tf_weight_grad_workspace(M, N, K) // 4))
    for odd in (False, True):
        if odd:
            G[M - 1, N - 1], X[M // 2, K - 1] = np.inf, np.nan
        Gd, Xd, Y = tf.DenseMatrix.from_numpy(G), tf.DenseMatrix.from_numpy(X), tf.DenseMatrix.from_numpy(np.full((N, K), np.nan, np.float32))
        assert lib.tf_weight_grad(Gd.h, Xd.h, Y.h, C.c_void_p(ws.device_ptr()), None) == 0
        tf.device_synchronize()
        got = Y.to_numpy()
        with np.errstate(invalid="ignore"):
            want = G.astype(np.float64).T @ X.astype(np.float64)
        ok = np.isfinite(want)
        size = np.abs(np.where(np.isfinite(G), G, 0)).astype(np.float64).T @ np.abs(np.where(np.isfinite(X), X, 0)).astype(np.float64)
        # fewer than 300 roundings of sums on the way of any term, each below the sum of magnitudes
        assert np.all(np.abs(got[ok] - want[ok]) <= 300 * 2.0 ** -24 * size[ok])
        assert np.array_equal(np.isnan(got), np.isnan(want)) and np.array_equal(np.isinf(got), np.isinf(want)) and ok.all() == (not odd)


# workgroups of eight wavefronts from 2,048 blocks of 32 rows on (256 compute units), of four below
@pytest.mark.parametrize("M,N,K", [(65504, 17, 130), (65505, 17, 130), (65537, 64, 48), (70001, 130, 257), (131071, 2, 3)])
def test_weight_gradient_of_many_rows(gpu, tf, M, N, K):
    test_weight_gradient_on_bf16_cores(gpu, tf, M, N, K)


@pytest.mark.parametrize("M,N,K", [(5000, 64, 100), (40000, 40, 128)])
@pytest.mark.parametrize("q", [1, 2, 4, 8, 64])
def test_weight_gradient_of_rare_features(gpu, tf, M, N, K, q):
    """Columns of X of q values in all: no further from float64 than rounded fp32 products added up in fp32."""
    say(f"weight gradient of rare features {M} rows, {N} x {K}, {q} a column")
    rng = np.random.default_rng(M + q)
    G, X = rng.uniform(-1, 1, (M, N)).astype(np.float32), np.ascontiguousarray(few_values(rng, K, M, q).T)
    lib = tf.lib()
    ws = tf.DenseMatrix(1, max(1, lib.tf_weight_grad_workspace(M, N, K) // 4))
    Gd, Xd, Y = tf.DenseMatrix.from_numpy(G), tf.DenseMatrix.from_numpy(X), tf.DenseMatrix(N, K)
    assert lib.tf_weight_grad(Gd.h, Xd.h, Y.h, C.c_void_p(ws.device_ptr()), None) == 0
    tf.device_synchronize()
    rows = np.stack([np.flatnonzero(X[:, k]) for k in range(K)])                             # K x q
    products = G[rows].astype(np.float64) * X[rows, np.arange(K)[:, None]][:, :, None]       # K x q x N
    want, size = products.sum(1).T, np.abs(products).sum(1).T
    fp32 = np.zeros((K, N), np.float32)
    for p in np.moveaxis(products.astype(np.float32), 1, 0):
        fp32 += p
    e, ref = np.abs(Y.to_numpy() - want) / size, np.abs(fp32.T - want) / size
    say(f"  largest {e.max():.3g} ({ref.max():.3g}), rms {np.sqrt((e ** 2).mean()):.4g} ({np.sqrt((ref ** 2).mean()):.4g})")
    assert e.max() <= q * 2.0 ** -24 * (1 + 2.0 ** -6)  # every product and every sum rounded once
    assert np.sqrt((e ** 2).mean()) <= 1.05 * np.sqrt((ref ** 2).mean())  # (of some 6,000 values each: 1.3 %)


@pytest.mark.parametrize("what,M,K,N", [("gemm", 18437, 300, 65), ("gemm", 18437, 300, 67), ("gemm", 18437, 257, 130), ("gemm", 18437, 300, 68), ("gradient", 9000, 193, 40),
                                        ("gradient", 9000, 40, 195), ("gradient", 9000, 194, 129), ("gradient", 4097, 70, 65)])
@pytest.mark.parametrize("bad", [np.inf, np.nan, 1e38])
def test_columns_of_other_panels_keep_their_bits(gpu, tf, what, M, K, N, bad):
    """A value in the last column that takes its panel (chunk) to the fp32 cores changes nothing in the panels before it, also where
    the last one is narrower than what a lane works on."""
    say(f"panels {what} {M} x {K} x {N} {bad}")
    rng = np.random.default_rng(M + K + N)
    lib = tf.lib()
    X, W, G = (rng.uniform(-1, 1, s).astype(np.float32) for s in ((M, K), (K, N), (M, N)))
    got = []
    for value in (0.5, bad, bad):
        W[0, N - 1] = G[M // 2, N - 1] = value
        Xd, Wd, Gd = (tf.DenseMatrix.from_numpy(a) for a in (X, W, G))
        if what == "gemm":
            Y = tf.DenseMatrix(M, N)
            assert lib.tf_gemm_ex(Xd.h, Wd.h, Y.h, None, 0, None) == 0
        else:
            Y, ws = tf.DenseMatrix(N, K), tf.DenseMatrix(1, lib.tf_weight_grad_workspace(M, N, K) // 4)
            assert lib.tf_weight_grad(Gd.h, Xd.h, Y.h, C.c_void_p(ws.device_ptr()), None) == 0
        tf.device_synchronize()
        got.append(Y.to_numpy() if what == "gemm" else Y.to_numpy().T)
    panel = 64 if what == "gemm" else 16 * -(-(-(-N // -(-N // 64))) // 16)  # (gradients: chunks of up to 64 columns, evenly)
    before = (N - 1) // panel * panel
    assert before > 0 or N <= 64
    assert np.array_equal(got[0][:, :before], got[1][:, :before])
    assert np.array_equal(got[1], got[2], equal_nan=True)


@pytest.mark.parametrize("M1,M2", [(100, 100), (3072, 3072), (3073, 3073), (4096, 4096), (4097, 4097), (20001, 20001), (3000, 5000), (5000, 3000), (4096, 4097)])
def test_two_weight_gradients_in_one_call(gpu, tf, M1, M2):
    """Sharing their launches changes no bit of either, of few rows and of many (and of one and the other)."""
    say(f"two weight gradients {M1} {M2}")
    rng = np.random.default_rng(M1 + M2)
    lib = tf.lib()
    alone, pair = [], []
    for M, N, K in ((M1, 32, 69), (M2, 7, 130)):
        Gd, Xd = (tf.DenseMatrix.from_numpy(rng.uniform(-1, 1, (M, w)).astype(np.float32)) for w in (N, K))
        ws = tf.DenseMatrix(1, max(1, lib.tf_weight_grad_workspace(M, N, K) // 4))
        Y = [tf.DenseMatrix.from_numpy(np.full((N, K), np.nan, np.float32)) for _ in range(2)]
        assert lib.tf_weight_grad(Gd.h, Xd.h, Y[0].h, C.c_void_p(ws.device_ptr()), None) == 0
        alone.append((Y[0], Gd, Xd, ws))
        pair.append((Gd, Xd, Y[1], ws))
    args = [a for g, x, y, ws in pair for a in (g.h, x.h, y.h, C.c_void_p(ws.device_ptr()))]
    tf.device_synchronize()
    assert lib.tf_weight_grad_pair(*args, None) == 0
    tf.device_synchronize()
    for (want, G, X, _), (_, _, got, _) in zip(alone, pair):
        assert np.array_equal(got.to_numpy(), want.to_numpy())
        assert rel(got.to_numpy(), G.to_numpy().astype(np.float64).T @ X.to_numpy().astype(np.float64)) <= 1e-5
    for bad in range(8):  # every operand is checked before either product runs
        if bad % 4 != 3:
            assert lib.tf_weight_grad_pair(*[None if i == bad else a for i, a in enumerate(args)], None) != 0


@pytest.mark.parametrize("M1,M2", [(65505, 65505), (65504, 65505), (66000, 4096)])
def test_two_weight_gradients_of_many_rows_in_one_call(gpu, tf, M1, M2):
    test_two_weight_gradients_in_one_call(gpu, tf, M1, M2)



@pytest.mark.parametrize("N", [1, 3, 4, 7, 16, 40, 64, 100, 128, 257])
@pytest.mark.parametrize("relu", [False, True])
def test_scheduled_row_product(gpu, tf, N, relu):
    """Hub rows of one and of several chunks, rows without entries, rows of up to 32 entries."""
    say(f"scheduled spmm N={N} relu={relu}")
    rng = np.random.default_rng(N)
    M = 4000
    A = sp.random(M, M, density=3.0 / M, random_state=5, format="lil", dtype=np.float32)
    for r, n in ((0, 33), (1, 900), (2000, 1024), (2001, 1025), (3999, 3500)):
        A[r, :] = 0
        A[r, rng.choice(M, n, replace=False)] = rng.uniform(-1, 1, n)
    A = sp.csr_matrix(A, dtype=np.float32)
    A.sort_indices()
    X = rng.uniform(-1, 1, (M, N)).astype(np.float32)
    Ah = tf.CsrMatrix.from_scipy(A).to_device()
    lib = tf.lib()
    s = C.c_void_p()
    assert lib.tf_inspect_spmm(M, M, Ah._pp, Ah._pi, N, 0, C.byref(s)) == 0
    try:
        Xd, Y = tf.DenseMatrix.from_numpy(X), tf.DenseMatrix.from_numpy(np.full((M, N), np.nan, np.float32))
        want = A.astype(np.float64) @ X.astype(np.float64)
        for flags in (RELU if relu else 0, 1 | (RELU if relu else 0)):  # then D += A X
            assert lib.tf_spmm_scheduled(Ah.h, Xd.h, Y.h, s, flags, None) == 0
            tf.device_synchronize()
            ref = want if not flags & 1 else (np.maximum(want, 0) if relu else want) + want
            assert rel(Y.to_numpy(), np.maximum(ref, 0) if relu else ref) <= 1e-5, flags
    finally:
        lib.tf_schedule_free(s)


@pytest.mark.parametrize("N", [1, 3, 30, 64, 128, 260])
@pytest.mark.parametrize("empty", [0.3, 0.9])
def test_rows_without_entries(gpu, tf, N, empty):
    """Fewer and more rows without entries than with, cleared by the row product's own launch; with accumulation untouched but for
    a ReLU."""
    say(f"empty rows N={N} {empty}")
    rng = np.random.default_rng(N)
    M = 17000
    A = sp.csr_matrix(sp.diags((rng.random(M) >= empty).astype(np.float32)) @ tf.workloads.erdos_renyi_gcn(M, 9.0, seed=1), dtype=np.float32)
    A.eliminate_zeros()
    X, D0 = (rng.uniform(-1, 1, (M, N)).astype(np.float32) for _ in range(2))
    Ah = tf.CsrMatrix.from_scipy(A).to_device()
    lib = tf.lib()
    s = C.c_void_p()
    assert lib.tf_inspect_spmm(M, M, Ah._pp, Ah._pi, N, 0, C.byref(s)) == 0
    try:
        Xd = tf.DenseMatrix.from_numpy(X)
        want = A.astype(np.float64) @ X.astype(np.float64)
        for flags in (0, RELU, 1, 1 | RELU):
            Y = tf.DenseMatrix.from_numpy(D0 if flags & 1 else np.full((M, N), np.nan, np.float32))
            assert lib.tf_spmm_scheduled(Ah.h, Xd.h, Y.h, s, flags, None) == 0
            tf.device_synchronize()
            ref = want + D0 if flags & 1 else want
            assert rel(Y.to_numpy(), np.maximum(ref, 0) if flags & RELU else ref) <= 1e-5, flags
    finally:
        lib.tf_schedule_free(s)


@pytest.mark.parametrize("K,N", [(30, 7), (500, 32), (251, 47), (64, 300), (300, 128), (32, 1)])
def test_layer_that_fuses_nothing_in_any_width(gpu, tf, K, N):
    """GeMM-SpMM on a graph: K and N as they come, either storage of the weights, accumulation, a ReLU of the result."""
    say(f"unfused layer K={K} N={N}")
    A = tf.workloads.rmat(12, 4096 * 8, seed=3)
    M = A.shape[0]
    rng = np.random.default_rng(K + N)
    X, W, D0 = (rng.uniform(-1, 1, s).astype(np.float32) for s in ((M, K), (K, N), (M, N)))
    Ah = tf.CsrMatrix.from_scipy(A)
    S = tf.inspector(Ah, op=tf.OP_GEMM_SPMM, N=N, K=K)
    Xd = tf.DenseMatrix.from_numpy(X)
    want = A.astype(np.float64) @ (X.astype(np.float64) @ W.astype(np.float64))
    for flags in (0, 1, RELU, C_TRANSPOSED, 1 | RELU | C_TRANSPOSED):
        Wd = tf.DenseMatrix.from_numpy(np.ascontiguousarray(W.T) if flags & C_TRANSPOSED else W)
        D = tf.DenseMatrix.from_numpy(D0)
        assert tf.lib().tf_gemm_spmm(Ah.to_device().h, Xd.h, Wd.h, D.h, S.h, flags, None) == 0
        tf.device_synchronize()
        ref = want + D0 if flags & 1 else want
        assert rel(D.to_numpy(), np.maximum(ref, 0) if flags & RELU else ref) <= 1e-5, flags


@pytest.mark.parametrize("K,N", [(64, 64), (30, 40)])
def test_fused_layer_with_transposed_weights(gpu, tf, K, N):
    """The same flags where rows fuse (a band), through the padded copies and the transposing one."""
    say(f"fused layer K={K} N={N}")
    A = tf.workloads.banded_random(3000, 32, 16, seed=9)
    M = A.shape[0]
    rng = np.random.default_rng(K)
    X, W = (rng.uniform(-1, 1, s).astype(np.float32) for s in ((M, K), (K, N)))
    Ah = tf.CsrMatrix.from_scipy(A)
    S = tf.inspector(Ah, op=tf.OP_GEMM_SPMM, N=N, K=K)
    want = A.astype(np.float64) @ (X.astype(np.float64) @ W.astype(np.float64))
    for flags in (0, C_TRANSPOSED, C_TRANSPOSED | RELU):
        Wd = tf.DenseMatrix.from_numpy(np.ascontiguousarray(W.T) if flags & C_TRANSPOSED else W)
        D = tf.DenseMatrix(M, N)
        assert tf.lib().tf_gemm_spmm(Ah.to_device().h, tf.DenseMatrix.from_numpy(X).h, Wd.h, D.h, S.h, flags, None) == 0
        tf.device_synchronize()
        assert rel(D.to_numpy(), np.maximum(want, 0) if flags & RELU else want) <= 1e-5, flags


@pytest.mark.parametrize("M,K,N", [(17, 4, 1), (500, 30, 30), (4096, 64, 64), (4096, 5, 130), (3000, 128, 7), (2000, 100, 129), (23999, 33, 17), (24001, 30, 30),
                                   (24500, 64, 96), (30000, 7, 16), (25000, 61, 64)])
@pytest.mark.parametrize("listed", [False, True])
def test_layer_in_one_launch(gpu, tf, M, K, N, listed):
    """(A B) C in one kernel: rows in order and in lists (two length classes, rows without entries), either storage of the weights,
    accumulation and a ReLU of the result."""
    say(f"one launch M={M} {K}x{N} listed={listed}")
    rng = np.random.default_rng(M + K + N)
    if listed:
        A = tf.workloads.erdos_renyi_gcn(M, 8.0, seed=3)
        if M > 100:
            keep = np.ones(M)
            keep[rng.integers(0, M, M // 3)] = 0.0
            A = sp.csr_matrix(sp.diags(keep) @ A)
            A.eliminate_zeros()
        A = sp.csr_matrix(A, dtype=np.float32)
    else:
        A = sp.csr_matrix(sp.diags([1.0, -2.0, 3.0], [-1, 0, 2], shape=(M, M)), dtype=np.float32)
    A.sort_indices()
    X, W, D0 = (rng.uniform(-1, 1, s).astype(np.float32) for s in ((M, K), (K, N), (M, N)))
    Ah = tf.CsrMatrix.from_scipy(A)
    S = tf.inspector(Ah, op=tf.OP_GEMM_SPMM, N=N, K=K)
    S.validate()
    want = A.astype(np.float64) @ (X.astype(np.float64) @ W.astype(np.float64))
    Xd = tf.DenseMatrix.from_numpy(X)
    S.set_profiling(True)
    for flags in (0, C_TRANSPOSED, 1, RELU, 1 | RELU | C_TRANSPOSED):
        Wd = tf.DenseMatrix.from_numpy(np.ascontiguousarray(W.T) if flags & C_TRANSPOSED else W)
        D = tf.DenseMatrix.from_numpy(D0)
        assert tf.lib().tf_gemm_spmm(Ah.to_device().h, Xd.h, Wd.h, D.h, S.h, flags, None) == 0
        tf.device_synchronize()
        if flags == 0:
            assert "spmm_gemm_kernel" in [n for n, _ in S.profile()]
        ref = want + D0 if flags & 1 else want
        assert rel(D.to_numpy(), np.maximum(ref, 0) if flags & RELU else ref) <= 1e-5, flags


@pytest.mark.parametrize("M,K,N,one", [(19999, 32, 97, True), (20000, 32, 97, False), (20000, 31, 97, True), (20001, 128, 128, False), (23999, 64, 96, True),
                                       (29999, 64, 96, True), (30000, 64, 96, False), (30000, 65, 97, False), (30001, 44, 65, True), (30003, 32, 65, False)])
def test_layer_beyond_64_columns(gpu, tf, M, K, N, one):
    """One launch or two, on either side of the row counts and widths between them: the same sums, a value that is not finite included."""
    say(f"beyond 64 columns M={M} {K}x{N}")
    rng = np.random.default_rng(M + K + N)
    A = sp.csr_matrix(tf.workloads.erdos_renyi_gcn(M, 4.0, seed=5), dtype=np.float32)
    X, W, D0 = (rng.uniform(-1, 1, s).astype(np.float32) for s in ((M, K), (K, N), (M, N)))
    Ah = tf.CsrMatrix.from_scipy(A)
    S = tf.inspector(Ah, op=tf.OP_GEMM_SPMM, N=N, K=K)
    S.set_profiling(True)
    for bad in (None, np.inf, np.nan):
        if bad is not None:
            X[M // 2, K - 1] = bad
        with np.errstate(invalid="ignore"):
            want = A.astype(np.float64) @ (X.astype(np.float64) @ W.astype(np.float64))
        for flags in (0, C_TRANSPOSED, 1, RELU):
            Wd = tf.DenseMatrix.from_numpy(np.ascontiguousarray(W.T) if flags & C_TRANSPOSED else W)
            D = tf.DenseMatrix.from_numpy(D0)
            Xd = tf.DenseMatrix.from_numpy(X)
            assert tf.lib().tf_gemm_spmm(Ah.to_device().h, Xd.h, Wd.h, D.h, S.h, flags, None) == 0
            tf.device_synchronize()
            assert ("spmm_gemm_kernel" in [n for n, _ in S.profile()]) == one
            ref = want + D0 if flags & 1 else want
            got, fine = D.to_numpy(), np.isfinite(ref).all(axis=1)  # a row that reads the value is not finite anywhere
            if bad is not None and not flags & RELU:
                assert not fine.all() and not np.isfinite(got[~fine]).any()
            # K products and the row's entries, each rounded once, in single precision
            assert rel(got[fine], np.maximum(ref, 0)[fine] if flags & RELU else ref[fine]) <= 1e-6, flags


@pytest.mark.parametrize("M,K,N", [(500, 2544, 1273), (500, 2545, 1273), (500, 3000, 2000), (60, 6001, 3001)])
def test_layer_of_few_rows_and_wide_features(gpu, tf, M, K, N):
    """Up to the K whose rows fill LDS in one launch, and beyond it."""
    say(f"few rows M={M} {K}x{N}")
    rng = np.random.default_rng(K)
    A = sp.csr_matrix(sp.diags([1.0, -2.0, 3.0], [-1, 0, 2], shape=(M, M)), dtype=np.float32)
    X, W, D0 = (rng.uniform(-1, 1, s).astype(np.float32) for s in ((M, K), (K, N), (M, N)))
    Ah = tf.CsrMatrix.from_scipy(A)
    S = tf.inspector(Ah, op=tf.OP_GEMM_SPMM, N=N, K=K)
    S.set_profiling(True)
    want = A.astype(np.float64) @ (X.astype(np.float64) @ W.astype(np.float64))
    for flags in (0, 1 | RELU | C_TRANSPOSED):
        Wd = tf.DenseMatrix.from_numpy(np.ascontiguousarray(W.T) if flags & C_TRANSPOSED else W)
        D = tf.DenseMatrix.from_numpy(D0)
        assert tf.lib().tf_gemm_spmm(Ah.to_device().h, tf.DenseMatrix.from_numpy(X).h, Wd.h, D.h, S.h, flags, None) == 0
        tf.device_synchronize()
        ref = np.maximum(want + D0, 0) if flags else want
        assert rel(D.to_numpy(), ref) <= 1e-5, flags
        assert ("spmm_gemm_kernel" in [n for n, _ in S.profile()]) == (K <= 2544)


@pytest.mark.parametrize("K,N", [(64, 80), (30, 40), (128, 140), (128, 96)])
def test_layer_on_a_band_with_hub_rows(gpu, tf, K, N):
    """Rows of 1,500 entries (two chunks, whose sums are added up) among rows of 17, more columns behind the products than before them
    and fewer."""
    say(f"band with hubs {K}x{N}")
    M = 3000
    rng = np.random.default_rng(K + N)
    A = sp.diags([1.0] * 17, list(range(-8, 9)), shape=(M, M), format="lil", dtype=np.float32)
    for r in (500, 1500, 2500):
        A[r, ::2] = 1.0
    A = sp.csr_matrix(A, dtype=np.float32)
    A.data = rng.uniform(-1, 1, A.nnz).astype(np.float32)
    X, W = (rng.uniform(-1, 1, s).astype(np.float32) for s in ((M, K), (K, N)))
    Ah = tf.CsrMatrix.from_scipy(A)
    S = tf.inspector(Ah, op=tf.OP_GEMM_SPMM, N=N, K=K)
    D = tf.DenseMatrix.from_numpy(np.full((M, N), np.nan, np.float32))
    tf.gemm_spmm(Ah, tf.DenseMatrix.from_numpy(X), tf.DenseMatrix.from_numpy(W), D, S)
    tf.device_synchronize()
    assert rel(D.to_numpy(), A.astype(np.float64) @ (X.astype(np.float64) @ W.astype(np.float64))) <= 1e-5

"""SpMM-SpMM of any width: windowed tiles with a ragged last strip (aligned and unaligned rows, a last strip of fewer than four
columns, accumulation), and the patterns that run as two row products instead of in tiles or marching runs, bit for bit against the oracle."""
import numpy as np
import pytest

from test_gpu_parity import oracle_spmm_spmm, say

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N", [4, 5, 7, 20, 29, 31, 33, 60, 63, 65, 66, 68, 77, 127, 129, 140, 257])
@pytest.mark.parametrize("rows", [700, 20000])
def test_windowed_tiles_of_any_width(gpu, tf, orc, N, rows):
    say(f"window N={N} rows={rows}")
    A = tf.workloads.banded_random(rows, 32, 11, seed=N)
    C = tf.workloads.uniform((rows, N), 2)
    Ah = tf.CsrMatrix.from_scipy(A)
    S = tf.inspector(Ah, op=tf.OP_SPMM_SPMM, N=N, inner=Ah)
    S.validate()
    assert S.info()["windowed"] and S.info()["wide_strips"] == 1
    want = oracle_spmm_spmm(orc, A, A, C)
    Cd, D = tf.DenseMatrix.from_numpy(C), tf.DenseMatrix.from_numpy(np.full((rows, N), np.nan, np.float32))
    tf.spmm_spmm(Ah, Ah, Cd, D, S)
    tf.device_synchronize()
    assert np.array_equal(D.to_numpy(), want)
    tf.spmm_spmm(Ah, Ah, Cd, D, S, accumulate=True)
    tf.device_synchronize()
    assert np.abs(D.to_numpy() - 2 * want).max() <= 1e-5 * np.abs(want).max()


@pytest.mark.parametrize("pattern,N", [("grid2d", 24), ("grid2d", 64), ("grid3d", 64), ("grid3d", 77), ("box3d", 64), ("box3d", 3), ("hub", 40)])
@pytest.mark.parametrize("other_inner", [False, True])
def test_two_row_products(gpu, tf, orc, pattern, N, other_inner):
    say(f"two products {pattern} N={N} other_inner={other_inner}")
    w = tf.workloads
    if pattern == "hub":
        A = w.rmat(11, 2048 * 8, seed=4)
    else:
        A = {"grid2d": lambda: w.laplacian_2d(70, 45), "grid3d": lambda: w.laplacian_3d(17), "box3d": lambda: w.box_stencil_3d(15)}[pattern]()
    B = A.copy()
    if other_inner:
        B.data = np.random.default_rng(1).uniform(-1, 1, B.nnz).astype(np.float32)
    C = w.uniform((A.shape[0], N), 5)
    Ah = tf.CsrMatrix.from_scipy(A)
    Bh = tf.CsrMatrix.from_scipy(B) if other_inner else Ah
    S = tf.inspector(Ah, op=tf.OP_SPMM_SPMM, N=N, inner=Bh)
    D = tf.DenseMatrix(A.shape[0], N)
    S.set_profiling(True)
    tf.spmm_spmm(Ah, Bh, tf.DenseMatrix.from_numpy(C), D, S)
    tf.device_synchronize()
    assert [n.split("_kernel")[0] for n, _ in S.profile() if n.startswith(("spmm_rows", "fused"))] == ["spmm_rows"] * 2
    want = oracle_spmm_spmm(orc, A, B, C)
    if pattern == "hub":
        assert np.abs(D.to_numpy() - want).max() <= 1e-5 * np.abs(want).max()
    else:
        assert np.array_equal(D.to_numpy(), want)


@pytest.mark.parametrize("N", [97, 100, 128, 52, 64])
def test_column_slices(gpu, tf, orc, N):
    """Graphs of the sizes at which the row kernel deals column slices to the XCDs (row counts that are no multiple of its blocks)."""
    say(f"column slices N={N}")
    n = 30011
    A = tf.workloads.erdos_renyi_gcn(n, 3.0, seed=N)
    C = tf.workloads.uniform((n, N), 7)
    Ah = tf.CsrMatrix.from_scipy(A)
    S = tf.inspector(Ah, op=tf.OP_SPMM_SPMM, N=N, inner=Ah)
    D = tf.DenseMatrix(n, N)
    tf.spmm_spmm(Ah, Ah, tf.DenseMatrix.from_numpy(C), D, S)
    tf.device_synchronize()
    assert np.array_equal(D.to_numpy(), oracle_spmm_spmm(orc, A, A, C))


@pytest.mark.parametrize("N", [97, 98, 99, 100, 128, 49, 64])
@pytest.mark.parametrize("op", ["spmm", "gemm"])
def test_column_slices_accumulate(gpu, tf, N, op):
    """D += A (B C) at those sizes: every column of D is added to once, whichever workgroups store it.  Whole numbers, so that the
    sums are exact in fp32 in any order: entries and operands of 1 to 4, below 2^24 altogether."""
    say(f"column slices accumulate N={N} {op}")
    n, K = 30011, 2 * N
    rng = np.random.default_rng(N)
    A = tf.workloads.erdos_renyi_gcn(n, 3.0, seed=N)
    A.data = rng.integers(1, 3, A.nnz).astype(np.float32)
    D0 = rng.integers(-4, 5, (n, N)).astype(np.float32)
    Ah = tf.CsrMatrix.from_scipy(A)
    D = tf.DenseMatrix.from_numpy(D0)
    A64 = A.astype(np.float64)
    if op == "spmm":
        C = rng.integers(-4, 5, (n, N)).astype(np.float32)
        S = tf.inspector(Ah, op=tf.OP_SPMM_SPMM, N=N, inner=Ah)
        step = A64 @ (A64 @ C.astype(np.float64))
        operands = (Ah, tf.DenseMatrix.from_numpy(C))
    else:
        B, C = (rng.integers(-2, 3, s).astype(np.float32) for s in ((n, K), (K, N)))
        S = tf.inspector(Ah, op=tf.OP_GEMM_SPMM, N=N, K=K)
        step = A64 @ (B.astype(np.float64) @ C.astype(np.float64))
        operands = (tf.DenseMatrix.from_numpy(B), tf.DenseMatrix.from_numpy(C))
    assert np.abs(D0).max() + 2 * np.abs(step).max() < 2 ** 24
    for k in (1, 2):
        (tf.spmm_spmm if op == "spmm" else tf.gemm_spmm)(Ah, *operands, D, S, accumulate=True)
        tf.device_synchronize()
        assert np.array_equal(D.to_numpy(), D0 + k * step), k

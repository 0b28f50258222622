"""Runs over a grid whose 27-point stencil both matrices are (csrc/tf_box.hip): the oracle's bits at the edges of its
tiles, strips and planes, and where C holds infinities and NaN; patterns that are nearly the stencil stay with the general runs."""
import numpy as np
import pytest
import scipy.sparse as sp

from test_gpu_march import box_stencil, march, stencil_3d
from test_gpu_parity import oracle_spmm_spmm, say


# (x, y, z): one and two points more than a column, two planes, one column, fewer lines than a run takes; columns of C: a strip's edges, ragged
@pytest.mark.gpu
@pytest.mark.parametrize("dims,N", [((9, 31, 12), 64), ((25, 13, 9), 64), ((13, 26, 12), 128), ((30, 40, 2), 64), ((2, 200, 20), 64), ((200, 2, 23), 192),
                                    ((24, 12, 13), 64), ((48, 47, 50), 37), ((47, 48, 50), 65), ((48, 50, 47), 49)])
def test_box_bit_exact(gpu, tf, orc, dims, N):
    say(f"box {dims} N={N}")
    A = box_stencil(*dims, True, seed=31)
    B = A.copy()
    B.data = np.random.default_rng(32).uniform(-1, 1, B.nnz).astype(np.float32)
    Cd = tf.workloads.uniform((A.shape[0], N), 33)
    D0 = tf.workloads.uniform((A.shape[0], N), 34)
    want = oracle_spmm_spmm(orc, A, B, Cd)
    Ah, Bh = tf.CsrMatrix.from_scipy(A), tf.CsrMatrix.from_scipy(B)
    for kw in (dict(), dict(compute_units=7)):
        S = tf.inspector(Ah, 1, op=tf.OP_SPMM_SPMM, N=N, inner=Ah, march=1 if N % 64 == 0 else 0, **kw)
        S.validate()
        info = S.info()
        if N % 64 and kw:
            assert info["marched"] == 0  # (few compute units: more turns of the runs than two products take)
            continue
        assert info["marched"] == 1 and info["march_tile_x"] in (8, 12) and info["march_tile_y"] <= 6, info
        for acc in (False, True):
            D = tf.DenseMatrix(A.shape[0], N, D0) if acc else tf.DenseMatrix(A.shape[0], N)
            if not acc:
                D.fill(float("nan"))
            tf.spmm_spmm(Ah, Bh, tf.DenseMatrix.from_numpy(Cd), D, S, accumulate=acc)
            tf.device_synchronize()
            assert np.array_equal(D.to_numpy(), D0 + want if acc else want), (dims, N, kw, acc)


@pytest.mark.gpu
def test_box_keeps_infinities_where_they_are(gpu, tf, orc):
    """A row of C that is not finite reaches the rows of D within two points of it and no others, at corners and across tiles too."""
    say("box with infinities and NaN")
    nx, ny, nz = 20, 13, 14
    A = box_stencil(nx, ny, nz, True, seed=35)
    Cd = tf.workloads.uniform((A.shape[0], 64), 36)
    hit = [0, nx - 1, nx * ny * (nz - 1), (5 * ny + 6) * nx + 12, (7 * ny + 12) * nx + 7]
    Cd[hit] = np.array([np.inf, -np.inf, np.nan, np.inf, np.nan], np.float32)[:, None]
    with np.errstate(invalid="ignore"):
        want = oracle_spmm_spmm(orc, A, A, Cd)
    got, _ = march(tf, A, A, Cd)
    assert np.array_equal(got, want, equal_nan=True)
    reach = np.zeros(A.shape[0], bool)
    for h in hit:
        p, q = np.arange(A.shape[0]), h
        reach |= (abs(p % nx - q % nx) <= 2) & (abs(p // nx % ny - q // nx % ny) <= 2) & (abs(p // nx // ny - q // nx // ny) <= 2)
    assert np.isfinite(got[~reach]).all()


def test_box_only_where_the_pattern_is_the_stencil(tf):
    """An entry moved, missing or out of order, two patterns of different grids, a wrong grid hint: not this kernel's runs (its columns are 8 or 12
    by at most 6 points, the general runs' of 27 points 8 by 5 or 4 unless told otherwise) or refused by the validator."""
    A = box_stencil(24, 20, 18, True, seed=39)
    Ah = tf.CsrMatrix.from_scipy(A)
    S = tf.inspector(Ah, 1, op=tf.OP_SPMM_SPMM, N=64, inner=Ah, march=1)
    S.validate()
    slots = S.info()["march_slots"]
    for kind in ("moved", "swapped", "missing", "other"):
        B = A.copy()
        mid = B.indptr[(9 * 20 + 10) * 24 + 12]
        if kind == "moved":
            B.indices[mid] -= 1
        elif kind == "swapped":
            B.indices[mid], B.indices[mid + 1] = B.indices[mid + 1], B.indices[mid]
        elif kind == "missing":
            B.data[mid + 3] = 0
            B.eliminate_zeros()
        else:
            B = box_stencil(20, 24, 18, True, seed=39)
        Bh = tf.CsrMatrix.from_scipy(sp.csr_matrix((B.data, B.indices, B.indptr), shape=B.shape))
        for outer, inner in ((Bh, Bh), (Ah, Bh), (Bh, Ah)):
            if kind == "other" and outer is inner:
                continue
            try:
                T = tf.inspector(outer, 1, op=tf.OP_SPMM_SPMM, N=64, inner=inner, march=1)
                T.validate()
                assert T.info()["march_slots"] != slots, kind
            except tf.TileFusionError as e:
                assert e.status == -5, (kind, str(e))
        S._inner = Bh
        with pytest.raises(tf.TileFusionError):
            S.validate(Bh)
    S._inner = Ah
    assert tf.inspector(Ah, 1, op=tf.OP_SPMM_SPMM, N=64, inner=Ah, grid=(20, 24, 18)).info()["march_slots"] != slots
    with pytest.raises(tf.TileFusionError):   # (whole strips, as ever, for who insists on marching runs)
        tf.inspector(Ah, 1, op=tf.OP_SPMM_SPMM, N=48, inner=Ah, march=1)
    assert tf.inspector(Ah, 1, op=tf.OP_SPMM_SPMM, N=64, inner=Ah, march=-1).info()["marched"] == 0


@pytest.mark.parametrize("dims,N,points", [((16, 16, 16), 37, 27), ((12, 13, 14), 20, 27), ((16, 16, 16), 36, 7), ((300, 1, 30), 36, 5), ((2, 9, 11), 50, 27)])
def test_two_products_are_nothing_else(tf, dims, N, points):
    """A grid's stencil in a width that whole strips do not divide, on so few points that two products are faster: no runs are reported, and A's
    pattern alone validates the schedule."""
    A = box_stencil(*dims, True, seed=71) if points == 27 else stencil_3d(*dims, seed=71)
    Ah = tf.CsrMatrix.from_scipy(A)
    S = tf.inspector(Ah, 1, op=tf.OP_SPMM_SPMM, N=N, inner=Ah, strip_cols=64, compute_units=256)
    info = S.info()
    assert info["marched"] == 0 and info["march_tile_x"] == 0, info
    if not info["windowed"]:
        assert info["march_declined"] == 2
    S.validate()
    S._inner = None
    if not info["windowed"]:
        S.validate()


def beside_two_products(tf, points, N):
    """A grid's whole stencil and the schedule of its runs in a width that only they take."""
    A = box_stencil(40, 41, 39, True, seed=72) if points == 27 else stencil_3d(48, 47, 50, seed=72) if points == 7 else stencil_3d(300, 1, 310, seed=72)
    Ah = tf.CsrMatrix.from_scipy(A)
    S = tf.inspector(Ah, 1, op=tf.OP_SPMM_SPMM, N=N, inner=Ah, compute_units=256)
    assert S.info()["marched"] == 1
    return A, Ah, S


def one_entry_moved(tf, A):
    i = A.shape[0] // 2
    B = sp.csr_matrix((A.data, A.indices.copy(), A.indptr), shape=A.shape)
    B.indices[B.indptr[i]] -= 1
    return B, tf.CsrMatrix(B.shape[0], B.shape[1], B.indptr, B.indices, B.data)


@pytest.mark.parametrize("points,N", [(27, 61), (27, 100), (7, 100), (5, 60)])
def test_the_outer_pattern_alone_validates(tf, points, N):
    """Runs that stand in for two products are validated against A's pattern, as two products are; another pattern is not A's."""
    A, Ah, S = beside_two_products(tf, points, N)
    assert tf.lib().tf_schedule_validate(S.h, Ah.M, Ah.N, Ah._pp, Ah._pi) == 0
    _, Bh = one_entry_moved(tf, A)
    assert tf.lib().tf_schedule_validate(S.h, Bh.M, Bh.N, Bh._pp, Bh._pi) == -4


def other_inners(tf, A):
    """Inner matrices of A's shape and entry count, with an entry more, and with other columns."""
    M = A.shape[0]
    moved = one_entry_moved(tf, A)[0]
    more = sp.csr_matrix(A + sp.csr_matrix((np.ones(1, np.float32), ([3], [M - 1])), shape=A.shape))
    wide = sp.random(M, 500, density=6 / 500, format="csr", random_state=73, dtype=np.float32)
    for B in (moved, more, wide):
        B.indices = B.indices.astype(np.int32)
        B.indptr = B.indptr.astype(np.int32)
    return moved, more, wide


@pytest.mark.parametrize("points,N", [(27, 61), (7, 100), (5, 60)])
def test_other_inner_patterns_validate(tf, points, N):
    A, Ah, S = beside_two_products(tf, points, N)
    for B in other_inners(tf, A):
        S._inner = tf.CsrMatrix(B.shape[0], B.shape[1], B.indptr, B.indices, B.data)
        S.validate()
    S._inner = None
    S.validate()


@pytest.mark.gpu
@pytest.mark.parametrize("points,N", [(27, 61), (27, 100), (7, 100), (5, 60)])
def test_other_inner_matrices(gpu, tf, orc, points, N):
    """A schedule whose runs stand in for two products takes any inner matrix, and with the one it was made for it runs them, before and after."""
    say(f"other inner matrices on {points} points N={N}")
    A, Ah, S = beside_two_products(tf, points, N)
    S.set_profiling(True)
    runs = "fused_box_kernel" if points == 27 else "fused_star_kernel"
    for B in (A, *other_inners(tf, A), A):
        Bh = Ah if B is A else tf.CsrMatrix(B.shape[0], B.shape[1], B.indptr, B.indices, B.data)
        Cd = tf.workloads.uniform((B.shape[1], N), 74)
        D0 = tf.workloads.uniform((A.shape[0], N), 75)
        want = oracle_spmm_spmm(orc, A, B, Cd)
        for acc in (False, True):
            D = tf.DenseMatrix(A.shape[0], N, D0)
            tf.spmm_spmm(Ah, Bh, tf.DenseMatrix.from_numpy(Cd), D, S, accumulate=acc)
            tf.device_synchronize()
            names = [n for n, _ in S.profile()]
            assert (names == [runs]) == (B is A) and len(names) == (1 if B is A else 2), names
            if not acc:
                assert np.array_equal(D.to_numpy(), want)
            else:  # (the runs add a whole sum to D; the rows' sums start at D: 27 roundings more of the magnitudes there are)
                size = abs(A.astype(np.float64)) @ abs(B.astype(np.float64) @ Cd) + abs(D0)
                assert (abs(D.to_numpy() - (want + D0.astype(np.float64))) <= 2 * 28 * 2.0 ** -24 * size).all()


@pytest.mark.gpu
@pytest.mark.parametrize("points,N", [(27, 61), (27, 64), (7, 100), (7, 64), (5, 60), (5, 64)])
def test_wrapped_inner_matrices_of_unknown_pattern(gpu, tf, orc, points, N):
    """A wrapped inner matrix without a hash may have any pattern with A's count of entries: the runs, which go by their own pattern, are not for it.
    With the hash of the inner pattern, or on A's own row pointers and columns, they are."""
    say(f"wrapped inner matrices on {points} points N={N}")
    A, Ah, S = beside_two_products(tf, points, N)
    S.set_profiling(True)
    other = one_entry_moved(tf, A)[0]
    Cd = tf.workloads.uniform((A.shape[0], N), 76)
    Ch = tf.DenseMatrix.from_numpy(Cd)
    D = tf.DenseMatrix(A.shape[0], N)

    def wrap(B, hash=0, like=None):
        own = [tf.DenseMatrix.from_numpy(np.ascontiguousarray(x).view(np.float32).reshape(1, -1)) for x in (B.indptr, B.indices, B.data)]
        own[:2] = like or own[:2]
        return tf.CsrMatrix.wrap_device(tf.CsrMatrix.from_scipy(B), *(x.device_ptr() for x in own), hash), own

    Aw, A_dev = wrap(A)
    values = A.copy()
    values.data = np.random.default_rng(77).uniform(-1, 1, A.nnz).astype(np.float32)
    for outer, (inner, _keep), B, by_runs in ((Ah, wrap(other), other, False), (Ah, wrap(values), values, False), (Ah, wrap(values, tf.pattern_hash(A)), values, True),
                                              (Aw, (Aw, None), A, True), (Aw, wrap(values, like=A_dev[:2]), values, True)):
        D.fill(float("nan"))
        tf.spmm_spmm(outer, inner, Ch, D, S)
        tf.device_synchronize()
        assert np.array_equal(D.to_numpy(), oracle_spmm_spmm(orc, A, B, Cd))
        assert (len(S.profile()) == 1) == by_runs, S.profile()


# (whole strips on grids that were two products before there were runs for them, and larger ones, which make their intermediate then)
@pytest.mark.gpu
@pytest.mark.parametrize("points,dims,N", [(27, (40, 41, 39), 61), (27, (40, 41, 39), 64), (7, (48, 47, 50), 100), (7, (48, 47, 50), 64), (5, (300, 1, 310), 60), (7, (60, 55, 60), 64)])
def test_in_place(gpu, tf, orc, points, dims, N):
    """D in C's memory, all of it or a part: what C holds before the call is multiplied."""
    say(f"in place on {points} points {dims} N={N}")
    A = box_stencil(*dims, True, seed=78) if points == 27 else stencil_3d(*dims, seed=78)
    M = A.shape[0]
    Ah = tf.CsrMatrix.from_scipy(A)
    S = tf.inspector(Ah, 1, op=tf.OP_SPMM_SPMM, N=N, inner=Ah, compute_units=256)
    S.set_profiling(True)
    Cd = tf.workloads.uniform((M, N), 79)
    want = oracle_spmm_spmm(orc, A, A, Cd)
    both = tf.DenseMatrix(M + 8, N)  # C from row 0 or 8 on, D from row 8 on (rows of 240 bytes and more, in whole 16 bytes after four of them)
    for first in (0, 8):
        C = tf.DenseMatrix.wrap_device(M, N, both.device_ptr() + first * N * 4)
        D = tf.DenseMatrix.wrap_device(M, N, both.device_ptr() + 8 * N * 4)
        C.copy_from(tf.DenseMatrix.from_numpy(Cd))
        tf.spmm_spmm(Ah, Ah, C, D, S)
        tf.device_synchronize()
        assert np.array_equal(D.to_numpy(), want), (first, S.profile())
        assert len(S.profile()) == 2
    D = tf.DenseMatrix(M, N)
    tf.spmm_spmm(Ah, Ah, tf.DenseMatrix.from_numpy(Cd), D, S)
    tf.device_synchronize()
    assert np.array_equal(D.to_numpy(), want) and len(S.profile()) == 1


@pytest.mark.parametrize("points,N", [(27, 61), (27, 100), (7, 100), (5, 60)])
def test_options_that_shape_tiles_get_tiles(tf, points, N):
    """Runs that stand in for two products do so where nothing is asked of the tiles; a budget of LDS, a tile's rows or halo and what becomes of long rows
    shape the schedule as before."""
    A, Ah, _ = beside_two_products(tf, points, N)
    for kw in (dict(lds_budget_bytes=65536), dict(tile_rows=700), dict(max_redundancy=1.0), dict(long_row_nnz=8), dict(long_row_partition=-1)):
        S = tf.inspector(Ah, 1, op=tf.OP_SPMM_SPMM, N=N, inner=Ah, compute_units=256, **kw)
        info = S.info()
        assert info["marched"] == 0 and info["lds_bytes"] <= kw.get("lds_budget_bytes", 81920), (kw, info)
        assert info["n_producer_rows"] == A.shape[0] or "max_redundancy" not in kw, info
        S.validate()


# (N: one strip of part of its columns, a whole and half of one, one and a bit; the grid's edges off the columns' both ways)
@pytest.mark.gpu
@pytest.mark.parametrize("dims,N", [((61, 59, 47), 36), ((61, 59, 47), 60), ((48, 47, 50), 96), ((47, 48, 50), 100), ((60, 62, 49), 44), ((61, 59, 47), 132)])
def test_box_sixteen_byte_loads_of_part_of_a_strip(gpu, tf, orc, dims, N):
    """Widths of whole sixteen bytes that are no whole strips: the form that loads four columns at once, some of its lanes with nothing to load."""
    say(f"box {dims} N={N}")
    A = box_stencil(*dims, True, seed=41)
    B = A.copy()
    B.data = np.random.default_rng(42).uniform(-1, 1, B.nnz).astype(np.float32)
    Cd = tf.workloads.uniform((A.shape[0], N), 43)
    D0 = tf.workloads.uniform((A.shape[0], N), 44)
    want = oracle_spmm_spmm(orc, A, B, Cd)
    Ah, Bh = tf.CsrMatrix.from_scipy(A), tf.CsrMatrix.from_scipy(B)
    S = tf.inspector(Ah, 1, op=tf.OP_SPMM_SPMM, N=N, inner=Ah, compute_units=256)
    S.set_profiling(True)
    for acc in (False, True):
        D = tf.DenseMatrix(A.shape[0], N, D0) if acc else tf.DenseMatrix(A.shape[0], N)
        if not acc:
            D.fill(float("nan"))
        tf.spmm_spmm(Ah, Bh, tf.DenseMatrix.from_numpy(Cd), D, S, accumulate=acc)
        tf.device_synchronize()
        assert np.array_equal(D.to_numpy(), D0 + want if acc else want), (dims, N, acc)
        assert [n for n, _ in S.profile()] == ["fused_box_kernel"]

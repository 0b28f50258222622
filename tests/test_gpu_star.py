"""Runs over a grid whose 7-point (in two dimensions 5-point) stencil both matrices are (csrc/tf_star.hip): the oracle's bits at the edges of its columns, strips and
planes, and where C and the values hold infinities and NaN; patterns that are nearly the stencil stay with the general runs."""
import numpy as np
import pytest

from test_gpu_march import march, stencil_3d
from test_gpu_parity import oracle_spmm_spmm, say


# (x, y, z): a column and one or two points more, two planes, three, two points wide, lines that do not divide; columns of C: a strip, its edges, four
# columns behind it; y = 1: lines of one column, one point more, two and three of them, two lines,
# and a D of more than 320 MB whose rows are no whole lines.  (Small grids of widths that are no strips of 64 go to two products: the larger ones are those that do not.)
@pytest.mark.gpu
@pytest.mark.parametrize("dims,N", [((16, 8, 9), 64), ((17, 9, 12), 64), ((18, 10, 2), 64), ((33, 17, 3), 128), ((2, 150, 6), 64), ((150, 2, 6), 64),
                                    ((290, 2, 5), 192), ((31, 23, 40), 64), ((90, 80, 70), 60), ((63, 61, 67), 100), ((110, 100, 60), 32), ((96, 40, 70), 96),
                                    ((94, 1, 20), 64), ((95, 1, 41), 64), ((93, 1, 50), 128), ((189, 1, 33), 192), ((2500, 1, 2), 64), ((700, 1, 300), 36), ((501, 1, 400), 100), ((1003, 1, 850), 100)])
def test_star_bit_exact(gpu, tf, orc, dims, N):
    say(f"star {dims} N={N}")
    A = stencil_3d(*dims, seed=61)
    B = A.copy()
    B.data = np.random.default_rng(62).uniform(-1, 1, B.nnz).astype(np.float32)
    Cd = tf.workloads.uniform((A.shape[0], N), 63)
    D0 = tf.workloads.uniform((A.shape[0], N), 64)
    wants = oracle_spmm_spmm(orc, A, B, Cd), oracle_spmm_spmm(orc, A, A, Cd)
    Ah, Bh = tf.CsrMatrix.from_scipy(A), tf.CsrMatrix.from_scipy(B)
    for kw in (dict(), dict(compute_units=7)):
        S = tf.inspector(Ah, 1, op=tf.OP_SPMM_SPMM, N=N, inner=Ah, **(dict(march=1, march_tile=(94, 1) if dims[1] == 1 else (16, 8)) if N % 64 == 0 else {}), **kw)
        S.validate()
        info = S.info()
        if N % 64 and not info["marched"]:
            assert kw  # (few compute units: more turns of the runs than two products take)
            continue
        columns = range(48, 95) if dims[1] == 1 else [16]
        assert info["marched"] == 1 and info["march_tile_x"] in columns and info["march_tile_y"] <= 8, info
        # two matrices, and one that is both (its values are read once)
        for inner, want, acc in ((Bh, wants[0], False), (Bh, wants[0], True), (Ah, wants[1], False), (Ah, wants[1], True)):
            D = tf.DenseMatrix(A.shape[0], N, D0) if acc else tf.DenseMatrix(A.shape[0], N)
            if not acc:
                D.fill(float("nan"))
            tf.spmm_spmm(Ah, inner, tf.DenseMatrix.from_numpy(Cd), D, S, accumulate=acc)
            tf.device_synchronize()
            assert np.array_equal(D.to_numpy(), D0 + want if acc else want), (dims, N, kw, acc)


@pytest.mark.gpu
@pytest.mark.parametrize("nx,ny,nz", [(35, 13, 14), (130, 1, 49)])
def test_star_keeps_infinities_where_they_are(gpu, tf, orc, nx, ny, nz):
    """A row of C or a value that is not finite reaches the rows of D within two steps along the axes and no others, at corners and across columns too."""
    say(f"star with infinities and NaN {nx} {ny} {nz}")
    A = stencil_3d(nx, ny, nz, seed=65)
    Cd = tf.workloads.uniform((A.shape[0], 64), 66)
    hit = [0, nx - 1, nx * ny * (nz - 1), (5 * ny + ny // 2) * nx + 15, (7 * ny + ny - 1) * nx + 16, (9 * ny + ny // 2) * nx + nx // 2]
    Cd[hit] = np.array([np.inf, -np.inf, np.nan, np.inf, np.nan, -np.inf], np.float32)[:, None]
    B = A.copy()
    B.data[B.indptr[4000]] = np.inf
    with np.errstate(invalid="ignore"):
        want = oracle_spmm_spmm(orc, A, B, Cd)
    got, info = march(tf, A, B, Cd, march_tile=(94, 1) if ny == 1 else (16, 8))
    assert info["march_tile_x"] == (66 if ny == 1 else 16)
    assert np.array_equal(got, want, equal_nan=True)
    p = np.arange(A.shape[0])
    reach = np.zeros(A.shape[0], bool)
    for q in hit + [4000]:
        reach |= abs(p % nx - q % nx) + abs(p // nx % ny - q // nx % ny) + abs(p // nx // ny - q // nx // ny) <= 2
    assert np.isfinite(got[~reach]).all()


def test_star_only_where_the_pattern_is_the_stencil(tf):
    """An entry moved, two out of order, two patterns of different grids, a grid hint that is another: not this kernel's runs (16 points wide), or refused."""
    A = stencil_3d(24, 20, 18, seed=69)
    Ah = tf.CsrMatrix.from_scipy(A)
    S = tf.inspector(Ah, 1, op=tf.OP_SPMM_SPMM, N=64, inner=Ah, march=1, march_tile=(16, 8))
    S.validate()
    assert S.info()["march_tile_x"] == 16
    slots = S.info()["march_slots"]
    mid = A.indptr[(9 * 20 + 10) * 24 + 12]
    for kind in ("moved", "swapped", "other"):
        B = A.copy()
        if kind == "moved":
            B.indices[mid] -= 1
        elif kind == "swapped":
            B.indices[mid], B.indices[mid + 1] = B.indices[mid + 1], B.indices[mid]
        else:
            B = stencil_3d(20, 24, 18, seed=69)
        Bh = tf.CsrMatrix(B.shape[0], B.shape[1], B.indptr, B.indices, B.data)
        for outer, inner in ((Bh, Bh), (Ah, Bh), (Bh, Ah)):
            if kind == "other" and outer is inner:
                continue
            try:
                T = tf.inspector(outer, 1, op=tf.OP_SPMM_SPMM, N=64, inner=inner, march=1, march_tile=(16, 8))
                assert T.info()["march_slots"] != slots, kind
            except tf.TileFusionError as e:
                assert e.status == -5, (kind, str(e))
        S._inner = Bh
        with pytest.raises(tf.TileFusionError):
            S.validate(Bh)
    S._inner = Ah
    assert tf.inspector(Ah, 1, op=tf.OP_SPMM_SPMM, N=64, inner=Ah, grid=(20, 24, 18)).info()["march_tile_x"] != 16
    assert tf.inspector(Ah, 1, op=tf.OP_SPMM_SPMM, N=64, inner=Ah, march=1).info()["march_tile_x"] != 16
    assert tf.inspector(Ah, 1, op=tf.OP_SPMM_SPMM, N=36, inner=Ah).info()["march_declined"] == 2
    assert tf.inspector(Ah, 1, op=tf.OP_SPMM_SPMM, N=64, inner=Ah, march_tile=(8, 8)).info()["march_tile_x"] == 8


def test_star_of_two_dimensions_only_where_the_pattern_is_the_stencil(tf):
    A = stencil_3d(188, 1, 40, seed=70)
    Ah = tf.CsrMatrix.from_scipy(A)
    S = tf.inspector(Ah, 1, op=tf.OP_SPMM_SPMM, N=64, inner=Ah, march=1, march_tile=(94, 1))
    S.validate()
    slots = S.info()["march_slots"]
    assert S.info()["march_tile_x"] == 94
    for at, to in ((A.indptr[20 * 188 + 7], -1), (A.indptr[20 * 188 + 187] + 3, -2), (A.indptr[39 * 188] + 1, 1)):
        B = A.copy()
        B.indices[at] += to
        Bh = tf.CsrMatrix(B.shape[0], B.shape[1], B.indptr, B.indices, B.data)
        try:
            assert tf.inspector(Bh, 1, op=tf.OP_SPMM_SPMM, N=64, inner=Bh, march=1, march_tile=(94, 1)).info()["march_slots"] != slots
        except tf.TileFusionError as e:
            assert e.status == -5, str(e)
        S._inner = Bh
        with pytest.raises(tf.TileFusionError):
            S.validate(Bh)
    S._inner = Ah
    # general runs for who insists on marching runs and names no column of these
    assert tf.inspector(Ah, 1, op=tf.OP_SPMM_SPMM, N=64, inner=Ah, march=1).info()["march_slots"] != slots

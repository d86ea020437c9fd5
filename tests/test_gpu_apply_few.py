"""The vector-unit apply at the right-hand-side counts, segment heights and
column counts where its chunks, lane map and split change: single dense
blocks against numpy, and butterflies against the one-column apply."""
import ctypes as C

import numpy as np
import pytest

from conftest import box_problem, curve_problem
from test_block_algebra import Dense, L, rand

pytestmark = pytest.mark.gpu


def rel(a, b):
    return np.linalg.norm(a - b) / np.linalg.norm(b)


def apply(bf, F, X, prec):
    dt = np.complex128 if prec == "fp64" else np.complex64
    n, nrhs = X.shape
    dx = bf.DeviceArray.from_numpy(X.astype(dt))
    dy = bf.DeviceArray.from_numpy(np.full((F.shape[0], nrhs), np.nan, dt))
    bf.mul_device(F, dx, dy, nrhs, prec)
    return dy.to_numpy(dt, (F.shape[0], nrhs)).astype(complex)


# m, n: one dense block (one segment of m rows and n columns): below, at and
# above one row, the 64 rows of a split segment's pass, the 128 of an unsplit
# one, and the columns at which segments split over 2 to 16 waves
@pytest.mark.parametrize("m,n", [(1, 1), (1, 700), (2, 3), (3, 31), (17, 31), (31, 33), (63, 64), (64, 65), (65, 130),
                                 (127, 17), (128, 100), (129, 33), (300, 5), (40, 400), (9, 1700)])
def test_one_dense_block(gpu_lib, m, n):
    lib = L()
    rng = np.random.default_rng(m * 1000 + n)
    A = rand(rng, m, n)
    dense, d = Dense(A), lib.bfMatBlockDiagNew()
    lib.bfMatBlockDiagInit(d, 1, 1)
    lib.bfMatBlockDiagSetBlock(d, 0, dense.ptr)
    P = gpu_lib.Mat(lib.bfhipMatPack(d))
    for nrhs in (1, 2, 3, 5, 8, 9, 13, 15):
        X = rand(rng, n, nrhs)
        # each of n complex products and sums is off by at most a few 2^-53 of |A| |X|
        bound = 4 * n * 2.0 ** -52 * (np.abs(A) @ np.abs(X))
        assert (np.abs(P @ X - A @ X) <= bound).all(), nrhs
    lib.bfMatDelete(C.byref(C.c_void_p(d)))


@pytest.mark.parametrize("geometry,n,leaf", [("curve", 5003, 32), ("box", 3001, 1)])
def test_few_columns_equal_one_column(gpu_lib, geometry, n, leaf):
    bf = gpu_lib
    src, tgt, k = curve_problem(n) if geometry == "curve" else box_problem(n)
    ts, tt = bf.Quadtree(src, leaf), bf.Quadtree(tgt, leaf)
    opts = bf.options(tol=1e-8, rank_const=1.25, pass_through=True, pinv_rcond=1e-11) if geometry == "curve" else None
    F = bf.FacHelm2.make_multilevel(bf.Helm2(k), ts, tt, opts)
    rng = np.random.default_rng(3)
    X = rng.standard_normal((n, 15)) + 1j * rng.standard_normal((n, 15))
    one = np.concatenate([apply(bf, F, X[:, c:c + 1], "fp64") for c in range(15)], 1)
    for nrhs in range(2, 16):
        # the same sums, split over waves in another order at most
        assert rel(apply(bf, F, X[:, :nrhs], "fp64"), one[:, :nrhs]) < 1e-13, nrhs
    # FP32 factors: one-row segments too, whose pair loads read a row twice
    F.orthogonalize()
    F.prepare_mixed("fp32")
    for nrhs in (1, 3, 8, 11):
        assert rel(apply(bf, F, X[:, :nrhs], "fp32"), one[:, :nrhs]) < 1e-6, nrhs

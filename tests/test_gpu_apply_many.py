"""The matrix-core apply where its row passes and columns are split over
waves: single dense blocks against numpy, and butterflies against the
one-column apply."""
import ctypes as C

import numpy as np
import pytest

from conftest import box_problem, curve_problem
from test_block_algebra import Dense, L, rand
from test_gpu_apply_few import apply, rel

pytestmark = pytest.mark.gpu


# one segment of m rows and n columns: below, at and above a row tile and a
# pass of two, and the columns at which 2, 4 and 8 waves share a pass, with
# remainders of the 4-column step
@pytest.mark.parametrize("m,n", [(1, 1), (1, 700), (15, 63), (16, 64), (17, 65), (31, 127), (32, 128), (33, 130),
                                 (64, 255), (65, 257), (130, 515), (300, 5), (9, 1701)])
def test_one_dense_block(gpu_lib, m, n):
    lib = L()
    rng = np.random.default_rng(m * 1000 + n)
    A = rand(rng, m, n)
    dense, d = Dense(A), lib.bfMatBlockDiagNew()
    lib.bfMatBlockDiagInit(d, 1, 1)
    lib.bfMatBlockDiagSetBlock(d, 0, dense.ptr)
    P = gpu_lib.Mat(lib.bfhipMatPack(d))
    for nrhs in (5, 8, 15, 16, 17, 32, 33, 64, 130):
        X = rand(rng, n, nrhs)
        # each of n complex products and sums is off by at most a few 2^-53 of |A| |X|
        bound = 4 * n * 2.0 ** -52 * (np.abs(A) @ np.abs(X))
        assert (np.abs(P @ X - A @ X) <= bound).all(), nrhs
    lib.bfMatDelete(C.byref(C.c_void_p(d)))


# many short segments beside a tall one: the waves that the tall one's passes
# get are bounded by the passes of all (one wave per pass in every segment
# would be 4e9 threads and more at the second size)
@pytest.mark.parametrize("short,m,nrhs", [(300, 20000, 40), (16000, 300000, 16), (3000, 33, 16)])
def test_one_tall_block_among_short_ones(gpu_lib, short, m, nrhs):
    lib = L()
    rng = np.random.default_rng(m)
    blocks = [rand(rng, 1 + i % 3, 2) for i in range(short)]
    blocks.insert(short // 2, rand(rng, m, 3))
    dense, d = [Dense(A) for A in blocks], lib.bfMatBlockDiagNew()
    lib.bfMatBlockDiagInit(d, len(dense), len(dense))
    for i, D in enumerate(dense):
        lib.bfMatBlockDiagSetBlock(d, i, D.ptr)
    P = gpu_lib.Mat(lib.bfhipMatPack(d))
    X = rand(rng, 2 * short + 3, nrhs)
    cols = np.cumsum([0] + [A.shape[1] for A in blocks])
    want = np.concatenate([A @ X[c:c + A.shape[1]] for A, c in zip(blocks, cols)])
    bound = np.concatenate([np.abs(A) @ np.abs(X[c:c + A.shape[1]]) for A, c in zip(blocks, cols)])
    # at most three products and their sum, each off by a few 2^-53
    assert (np.abs(P @ X - want) <= 12 * 2.0 ** -52 * bound).all()
    lib.bfMatDelete(C.byref(C.c_void_p(d)))


@pytest.mark.parametrize("geometry,n,leaf", [("curve", 4099, 64), ("box", 3001, 1)])
def test_many_columns_equal_one_column(gpu_lib, geometry, n, leaf):
    bf = gpu_lib
    src, tgt, k = curve_problem(n) if geometry == "curve" else box_problem(n)
    ts, tt = bf.Quadtree(src, leaf), bf.Quadtree(tgt, leaf)
    opts = bf.options(tol=1e-8, rank_const=1.25, pass_through=True, pinv_rcond=1e-11) if geometry == "curve" else None
    F = bf.FacHelm2.make_multilevel(bf.Helm2(k), ts, tt, opts)
    F.orthogonalize()
    rng = np.random.default_rng(5)
    X = rng.standard_normal((n, 70)) + 1j * rng.standard_normal((n, 70))
    one = np.concatenate([apply(bf, F, X[:, c:c + 1], "fp64") for c in range(70)], 1)
    many = (5, 6, 7, 8, 11, 15, 16, 19, 33, 70)
    for nrhs in many:
        # the same products in another order: the sums of a stage have up to
        # 2000 terms, of 10 stages
        assert rel(apply(bf, F, X[:, :nrhs], "fp64"), one[:, :nrhs]) < 1e-12, nrhs
    for prec in ("fp32x2", "fp32"):
        F.prepare_mixed(prec)
        for comp in (2, 1, 0) if prec == "fp32" else (2,):
            bf.lib().bfhipSetApplyCompensation(comp)
            try:
                for nrhs in many:
                    # FP32 vectors between ten stages: 6e-8 each, and with
                    # plain FP32 sums their length's root on top
                    assert rel(apply(bf, F, X[:, :nrhs], prec), one[:, :nrhs]) < (1e-6 if comp else 5e-6), (prec, comp)
            finally:
                bf.lib().bfhipSetApplyCompensation(2)


@pytest.mark.parametrize("comp", [3, 5, 9])
def test_split_stages_with_coarser_folds(gpu_lib, comp):
    """FP32 tiles folded into the FP64 sums every 2, 4 or 8 steps, in stages
    whose columns are split over waves: the last of a curve (about 130
    segments of 2000 columns, no multiple of 8 steps times the waves) and a
    small box's.  A tile that a wave left unfolded would cost a share of the
    columns, 1e-2 and more."""
    bf = gpu_lib
    for (src, tgt, k), leaf in ((curve_problem(4099), 64), (box_problem(1500), 32)):
        n = len(src)
        ts, tt = bf.Quadtree(src, leaf), bf.Quadtree(tgt, leaf)
        F = bf.FacHelm2.make_multilevel(bf.Helm2(k), ts, tt,
                                        bf.options(tol=1e-8, rank_const=1.25, pass_through=True, pinv_rcond=1e-11))
        F.orthogonalize()
        rng = np.random.default_rng(6)
        X = rng.standard_normal((n, 37)) + 1j * rng.standard_normal((n, 37))
        one = np.concatenate([apply(bf, F, X[:, c:c + 1], "fp64") for c in range(37)], 1)
        F.prepare_mixed("fp32")
        bf.lib().bfhipSetApplyCompensation(comp)
        try:
            for nrhs in (5, 16, 19, 37):
                # FP32 vectors between ten stages, sums of 32 columns in FP32:
                # 6e-8 each, times the root of 10 x (1 + 32 / 4)
                assert rel(apply(bf, F, X[:, :nrhs], "fp32"), one[:, :nrhs]) < 1e-6, nrhs
        finally:
            bf.lib().bfhipSetApplyCompensation(2)

"""Orthogonalization of column blocks with fewer rows than columns: their Q
and R, and the single entries of the FP32 apply, which such columns decide
where they are left as they are."""
import numpy as np
import pytest

from conftest import curve_problem
from test_gpu_apply_few import apply
from test_gpu_parity import _columns_of

pytestmark = pytest.mark.gpu


def factor(bf, n, tol):
    src, tgt, k = curve_problem(n)
    ts, tt = bf.Quadtree(src, 64), bf.Quadtree(tgt, 64)
    opts = bf.options(tol=tol, rank_const=1.25, pass_through=True, pinv_rcond=1e-11)
    return bf.FacHelm2.make_multilevel(bf.Helm2(k), ts, tt, opts), ts, tt


def test_wide_columns_are_rotated(gpu_lib):
    """Q = [orthonormal | 0] in every column block that proxy rows feed, wide
    or not, and the operator is unchanged."""
    F, _, _ = factor(gpu_lib, 4096, 1e-6)
    rng = np.random.default_rng(2)
    x = rng.standard_normal((4096, 3)) + 1j * rng.standard_normal((4096, 3))
    y = F @ x
    F.orthogonalize()
    assert np.linalg.norm(F @ x - y) < 1e-11 * np.linalg.norm(y)
    lt, ft, bt = F.plan()
    cols, rowkinds = _columns_of(lt, ft, bt)
    fed = [k for k in cols if k[1] >= 1 and rowkinds.get((k[0], k[1] - 1, k[2])) == {0}]
    height = {k: sum(bt[b][2] for b in cols[k]) for k in fed}
    wide = [k for k in fed if height[k] < bt[cols[k][0]][3]]
    tall = [k for k in fed if height[k] >= bt[cols[k][0]][3]]
    assert len(wide) > 100
    for key in wide + tall[::20]:
        Q = np.vstack([F.block(b, bt[b][2], bt[b][3]) for b in cols[key]])
        m, n = Q.shape
        eye = np.diag((np.arange(n) < m).astype(float))
        # up to 64 reflections, each off by a few 2^-53
        assert np.abs(Q.conj().T @ Q - eye).max() < 1e-13, (key, Q.shape)


@pytest.mark.parametrize("nrhs", [1, 3, 16])
def test_single_entries_of_the_fp32_apply(gpu_lib, nrhs):
    """Through orthonormal columns every rounding of a stage (10 of them; an
    intermediate and a factor each, 2^-24 at most, 2^-24 / sqrt(3) in the
    mean) reaches an output row with its share of the norm: sqrt(20) 2^-24 /
    sqrt(3) = 1.5e-7 in the mean, and the largest of 2 x 30000 x 16 entries is
    about 5.5 of these, 8.5e-7.  Three times that for rows with more than the
    mean share.  With the wide columns left alone: 4e-5 to 1.3e-4."""
    bf, n = gpu_lib, 30000
    F, _, _ = factor(bf, n, 1e-6)
    rng = np.random.default_rng(4)
    X = (rng.standard_normal((n, nrhs)) + 1j * rng.standard_normal((n, nrhs))).astype(np.complex64)
    y = apply(bf, F, X, "fp64").view(float)
    F.orthogonalize()
    F.prepare_mixed("fp32")
    off = np.abs(apply(bf, F, X, "fp32").view(float) - y) / np.maximum(np.abs(y), np.sqrt(np.mean(y ** 2)))
    assert off.max() < 3 * 8.5e-7

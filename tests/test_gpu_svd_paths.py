"""The batched SVD at the shapes where its path changes: QR in registers (up to
256 rows and 32 or 64 columns) and in global memory, Jacobi of the triangle by
a whole workgroup (up to 70 columns) and by blocks of 8 rows (71 to 256), of
the columns over the whole chip (from 257), and by one workgroup (more than
256 rows, less than 2^15 entries), each as is and transposed, several shapes
in one batch; and at the inputs where one of them could go wrong."""
import os
import subprocess
import sys

import numpy as np
import pytest

from conftest import ROOT

pytestmark = pytest.mark.gpu


def graded(rng, m, n):
    """sigma_0 = 1, exponents spread over 14 decades but none within a factor
    of 10 of the cut 1e-7, where rounding would decide the rank"""
    p = min(m, n)
    u = np.linalg.qr(rng.standard_normal((m, p)) + 1j * rng.standard_normal((m, p)))[0]
    v = np.linalg.qr(rng.standard_normal((n, p)) + 1j * rng.standard_normal((n, p)))[0]
    e = 12 * rng.random(p)
    e = np.where(e > 6, e + 2, e)
    e[0] = 0
    return (u * 10.0 ** -np.sort(e)) @ v.conj().T


@pytest.mark.parametrize("m,n", [(1, 1), (2, 1), (16, 16), (17, 17), (33, 8), (70, 70), (71, 71), (72, 71), (255, 64),
                                 (256, 64), (257, 64), (256, 65), (256, 70), (256, 71), (200, 150), (256, 256),
                                 (512, 32), (512, 33), (513, 32), (700, 80), (256, 32), (256, 33), (481, 68),
                                 (482, 68), (469, 70), (462, 71), (300, 256), (257, 257), (300, 257)])
def test_svd_at_the_edges_of_its_paths(gpu_lib, m, n):
    rng = np.random.default_rng(1000 * m + n)
    # the shape twice, transposed, rank 3 with a zero column, and a small one
    mats = [graded(rng, m, n), graded(rng, m, n), graded(rng, n, m), graded(rng, 9, 5)]
    r = min(3, m, n)
    low = (rng.standard_normal((m, r)) + 1j * rng.standard_normal((m, r))) @ rng.standard_normal((r, n))
    if n > 1:
        low[:, n // 2] = 0
    mats.append(low)
    tol = 1e-7
    for A, (U, W, k) in zip(mats, gpu_lib.svd_batched(mats, tol)):
        s = np.linalg.svd(A, compute_uv=False)
        assert k == int(np.sum(s >= tol * s[0]))
        # each of ~10 sweeps of n rotations is off by a few 2^-53
        eps = 2.0 ** -52 * max(m, n) * 40
        assert np.abs(U.conj().T @ U - np.eye(k)).max() < eps
        assert np.abs(np.linalg.norm(W, axis=1) - s[:k]).max() <= eps * s[0]
        rest = s[k] if k < len(s) else 0
        assert np.linalg.norm(U @ W - A, 2) <= rest * 1.0001 + eps * s[0]


FIRST = """
import numpy as np
import butterfly_amd as bf
rng = np.random.default_rng(7)
shapes = {shapes}
mats = [rng.standard_normal(s) + 1j * rng.standard_normal(s) for s in shapes]
first, second = bf.svd_batched(mats, 1e-7), bf.svd_batched(mats, 1e-7)
for A, (U, W, k), (U2, W2, k2) in zip(mats, first, second):
    assert k == k2 == min(A.shape) and np.array_equal(U, U2) and np.array_equal(W, W2), A.shape
    eps = 2.0 ** -52 * max(A.shape) * 40
    assert np.abs(U.conj().T @ U - np.eye(k)).max() < eps, A.shape
    assert np.linalg.norm(U @ W - A, 2) < eps * np.linalg.norm(A, 2), A.shape
print("same")
"""


@pytest.mark.parametrize("shapes", [[(40, 2), (2, 9), (5, 1)], [(60, 30), (200, 90), (3, 2), (12, 12)]])
def test_svd_as_the_first_call_of_a_process(gpu_lib, shapes):
    """A process whose first device call is a batched SVD takes the same path
    as one that has used the device before, also where no matrix has more
    than two columns."""
    out = subprocess.run([sys.executable, "-c", FIRST.format(shapes=shapes)], cwd=ROOT, capture_output=True, text=True,
                         timeout=100, env=dict(os.environ, PYTHONPATH=ROOT))
    assert out.returncode == 0 and "same" in out.stdout, out.stdout + out.stderr


@pytest.mark.parametrize("scale", [1.0, 1e-50, 1e-60])
@pytest.mark.parametrize("m,copies", [(60, 24), (300, 24), (120, 40)])
def test_svd_of_many_copies_of_two_columns(gpu_lib, scale, m, copies):
    """What the elimination leaves of a column's copies shrinks by 2^-52 with
    each step, down to numbers whose squares have no reciprocal."""
    mats = []
    for seed in range(30):
        rng = np.random.default_rng(seed)
        mats.append(scale * np.repeat(rng.standard_normal((m, 2)) + 1j * rng.standard_normal((m, 2)), copies, axis=1))
    eps = 2.0 ** -52 * max(m, 2 * copies) * 40
    for A, (U, W, k) in zip(mats, gpu_lib.svd_batched(mats, 1e-7)):
        assert k == 2
        assert np.abs(U.conj().T @ U - np.eye(2)).max() < eps
        assert np.linalg.norm(U @ W - A, 2) <= eps * np.linalg.norm(A, 2)
        if scale < 1e-55:  # what rounding leaves is out of the column Jacobi's range (300 rows)
            continue
        U0, W0, k0 = gpu_lib.svd_batched([A.T], 0.0)[0]
        assert k0 == min(A.shape)
        assert np.abs(U0.conj().T @ U0 - np.eye(k0)).max() < eps
        assert np.linalg.norm(U0 @ W0 - A.T, 2) <= eps * np.linalg.norm(A, 2)


@pytest.mark.parametrize("m,n", [(6, 9), (21, 48), (48, 300), (60, 64), (90, 120), (96, 400)])
def test_svd_of_repeated_rows_and_columns(gpu_lib, m, n):
    """Exact copies leave exactly zero rows in the triangle: with no cut, the
    vectors that belong to them are orthonormal to the others (U of a wide
    matrix; a tall one's U has zero columns there)."""
    rng = np.random.default_rng(m + n)
    A = np.repeat(rng.standard_normal((m // 3, n)) + 1j * rng.standard_normal((m // 3, n)), 3, axis=0)
    Z = np.zeros((m, n), complex)
    Z[: m // 2] = rng.standard_normal((m // 2, n))
    eps = 2.0 ** -52 * max(m, n) * 40
    for B in (A, Z, np.zeros((m, n), complex)):
        (U, W, k), (Ut, Wt, kt) = gpu_lib.svd_batched([B, B.T], 0.0)
        assert k == kt == m
        assert np.abs(U.conj().T @ U - np.eye(m)).max() < eps
        assert np.linalg.norm(U @ W - B, 2) <= eps * np.linalg.norm(B, 2)
        assert np.linalg.norm(Ut @ Wt - B.T, 2) <= eps * np.linalg.norm(B, 2)


@pytest.mark.parametrize("scale", [1e-70, 1e70])
@pytest.mark.parametrize("m,n", [(40, 12), (60, 60), (90, 200), (256, 250)])
def test_svd_far_from_one(gpu_lib, scale, m, n):
    """Entries whose fourth powers are out of range."""
    A = scale * graded(np.random.default_rng(m), m, n)
    U, W, k = gpu_lib.svd_batched([A], 1e-7)[0]
    s = np.linalg.svd(A, compute_uv=False)
    eps = 2.0 ** -52 * max(m, n) * 40
    assert k == int(np.sum(s >= 1e-7 * s[0]))
    assert np.abs(U.conj().T @ U - np.eye(k)).max() < eps
    assert np.linalg.norm(U @ W - A, 2) <= (s[k] if k < len(s) else 0) * 1.0001 + eps * s[0]


@pytest.mark.parametrize("m,n", [(40, 12), (60, 60), (90, 200), (256, 250), (300, 50), (300, 260)])
@pytest.mark.parametrize("bad", [np.nan, np.inf])
def test_svd_of_what_is_not_finite(gpu_lib, bad, m, n):
    """It shows in the factors; its neighbours in the batch are not touched."""
    rng = np.random.default_rng(n)
    A = rng.standard_normal((m, n)) + 1j * rng.standard_normal((m, n))
    B = A.copy()
    B[3, 5] = bad
    alone = gpu_lib.svd_batched([A], 1e-7)[0]
    (U, W, k), beside = gpu_lib.svd_batched([B, A], 1e-7)
    assert k > 0 and not np.isfinite(U @ W).all()
    assert beside[2] == alone[2] and np.array_equal(beside[0], alone[0]) and np.array_equal(beside[1], alone[1])

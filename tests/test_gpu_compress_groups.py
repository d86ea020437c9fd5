"""Re-expansion blocks of one row share one solve: groups of one to four
blocks, ragged and clipped at the LDS capacity, each block against a host
solve of its own least-squares problem."""
import numpy as np
import pytest

import oracle as orc
from test_gpu_layers import LAYERS, starfish

pytestmark = pytest.mark.gpu


def problem(geometry):
    rng = np.random.default_rng(9)
    if geometry == "curve":
        pts, nrm, tgt, _, k = starfish(6000)
        return pts, nrm, tgt, k, 16
    # boxes of a quadtree six levels deep that keep one to four children each;
    # the high wavenumber gives groups of more than the LDS size
    cells = [(0.0, 0.0)]
    for lev in range(1, 7):
        cells = [(x + (q & 1) / 2 ** lev, y + (q >> 1) / 2 ** lev) for x, y in cells
                 for q in (rng.permutation(4)[:rng.integers(1, 5)] if lev > 1 else range(4))]
    cells = np.array(cells)[rng.permutation(len(cells))[:200]]
    pts = (cells[:, None] + rng.uniform(0, 1 / 64, (len(cells), 30, 2))).reshape(-1, 2)
    ang = rng.uniform(0, 2 * np.pi, len(pts))
    return pts, np.stack([np.cos(ang), np.sin(ang)], 1), rng.uniform(0, 1, (len(pts), 2)) + [2, 0], 150.0, 1


@pytest.mark.parametrize("geometry,layer", [("box", "single"), ("box", "combined"), ("curve", "double")])
def test_grouped_blocks_solve_their_own_problems(gpu_lib, geometry, layer):
    bf = gpu_lib
    pts, nrm, tgt, k, leaf = problem(geometry)
    alpha, beta = 1.0, -0.5j
    helm = bf.Helm2(k) if layer == "single" else bf.Helm2(k, getattr(bf, LAYERS[layer]), alpha, beta)
    ts = bf.Quadtree(pts, leaf, normals=None if layer == "single" else nrm)
    tt = bf.Quadtree(tgt, leaf)
    F = bf.FacHelm2.make_multilevel(helm, ts, tt, bf.options(tol=1e-10, rank_const=1.25, pinv_rcond=1e-11))
    _, _, bt = F.plan()
    idx = np.nonzero(bt[:, 4] == 0)[0]
    geo = {i: F.block_geometry(i) for i in idx}
    runs = []
    for i in idx:
        g, prev = geo[i], runs[-1][-1] if runs else None
        if prev == i - 1 and (geo[prev][:6] == g[:6]).all() and geo[prev][10] == g[10]:
            runs[-1].append(i)
        else:
            runs.append([i])
    by = {}
    for r in runs:
        by.setdefault(len(r), []).append(r)
    assert set(by) >= ({1, 2, 3, 4} if geometry == "box" else {1, 2}), {s: len(v) for s, v in by.items()}
    lds = [geo[r[0]][10] * (geo[r[0]][10] + sum(geo[i][11] for i in r)) * 16 for r in runs]
    assert geometry != "box" or max(lds) > 160 * 1024, max(lds)
    p_sorted = np.argsort([geo[r[0]][10] for r in runs])
    pick = [runs[q] for q in p_sorted[-6:]] + [r for v in by.values() for r in v[:: max(1, len(v) // 8)]]

    def ker(t, s, ns):
        if layer == "single":
            return orc.kernel_matrix(k, t, s)
        return orc.kernel_matrix_layer(k, t, s, ns, layer, alpha, beta)

    sp, sn = pts[ts.perm], nrm[ts.perm]
    for i in (i for r in pick for i in r):
        ecx, ecy, er, tcx, tcy, tr, ocx, ocy, orr, off, p, n = geo[i]
        p, n, off = int(p), int(n), int(off)
        e, t = orc.circle_points(ecx, ecy, er, p), orc.circle_points(tcx, tcy, tr, p)
        o, no = (sp[off:off + n], sn[off:off + n]) if off >= 0 else (orc.circle_points(ocx, ocy, orr, n), None)
        if no is None:
            no = (o - [ocx, ocy]) / orr
        Ze, Zo = ker(t, e, (e - [ecx, ecy]) / er), ker(t, o, no)
        X = F.block(i, bt[i, 2], bt[i, 3])
        u, s, vh = np.linalg.svd(Ze)
        keep = s >= max(p * 2.2e-16 * s[0] + 2.2e-16, 1e-11 * s[0])
        Xn = vh[keep].conj().T @ ((u[:, keep].conj().T @ Zo) / s[keep, None])
        r_dev, r_np = (np.linalg.norm(Ze @ Y - Zo) / np.linalg.norm(Zo) for Y in (X, Xn))
        # as the blocks one by one: within rounding, grown by the condition
        # that the cut allows, of the host's truncated solution
        assert r_dev < 1000 * r_np + 1e-11, (i, p, n, r_dev, r_np)

"""The work that users of the butterfly library have it do, as timed cases.

A case is one call (or the short fixed sequence of calls that a program
makes together) on a problem of stated geometry and size:

  apply   Y = A X with a factorization in hand (the matvec of a solver, a
          field evaluation, a block of right-hand sides), on device buffers
  factor  trees, factorization, and one apply of it: what a program with a
          new geometry or wavenumber pays
  batch   Y = A X of independent problems factored as one operator
  solve   GMRES on the second-kind boundary equation of a closed curve
  stream  the streaming factorization fed with the columns of a matrix, and
          one apply of the finished product

Geometries: "curve" (n sources on r = 1 + 0.3 cos 5t, n targets on the
circle of radius 3, ppw points per wavelength along the curve) and "box" (n
sources in [0,1]^2, n targets in [2,3]x[0,1], ppw points per wavelength
across the box).  All use the pass-through planner with rank constant 1.25
and pseudo-inverse cut 1e-11, as bench.py does.

Vectors are in the order of the device-built quadtrees (the points sorted
stably by their quadrant path).
"""
import numpy as np
import torch

CURVE_L = 9.017203500515143  # length of r = 1 + 0.3 cos(5 theta)
# Kapur-Rokhlin correction weights of order 6 (SIAM J. Numer. Anal. 34, 1997)
KR6 = (4.967362978287758, -16.20501504859126, 25.85153761832639,
       -22.22599466791883, 9.930104998037539, -1.817995878141594)
RANK_CONST = 1.25
RCOND = 1e-11
SOLVE_TOL = 1e-10
SOLVE_ITERATIONS = 50
COMBINED = (1.0, -0.5j)  # alpha S + beta D


def listed():
    return [
        # the smallest call: one matvec of a 4096-point scatterer inside an
        # iterative method, bound by launches and latency
        {"name": "apply_curve_4k", "kind": "apply", "geometry": "curve", "layer": "single", "n": 4096, "ppw": 10.0,
         "leaf": 64, "tol": 1e-8, "prec": "fp64", "nrhs": 1, "graphs": False},
        # the volume-to-volume box problem of the plain method at its own
        # size, replayed as a graph the way a solver's inner loop would
        {"name": "apply_box_16k", "kind": "apply", "geometry": "box", "layer": "single", "n": 16384, "ppw": 8.0,
         "leaf": 64, "tol": 1e-8, "prec": "fp64", "nrhs": 1, "graphs": True},
        # the headline: one right-hand side at 2^20 points, bound by HBM
        {"name": "apply_curve_1m", "kind": "apply", "geometry": "curve", "layer": "single", "n": 1 << 20, "ppw": 10.0,
         "leaf": 64, "tol": 1e-8, "prec": "fp64", "nrhs": 1, "graphs": False},
        # a handful of incident directions on a ragged size
        {"name": "apply_few_100k", "kind": "apply", "geometry": "curve", "layer": "single", "n": 100003, "ppw": 10.0,
         "leaf": 64, "tol": 1e-8, "prec": "fp64", "nrhs": 6, "graphs": False},
        # many right-hand sides (a far-field matrix, a block of directions)
        {"name": "apply_256_fp64", "kind": "apply", "geometry": "curve", "layer": "single", "n": 180000, "ppw": 10.0,
         "leaf": 64, "tol": 1e-8, "prec": "fp64", "nrhs": 256, "graphs": False},
        # the same in the mixed form: orthogonalized FP32 factors, FP32
        # vectors, compensated sums
        {"name": "apply_256_fp32", "kind": "apply", "geometry": "curve", "layer": "single", "n": 180000, "ppw": 10.0,
         "leaf": 64, "tol": 1e-8, "prec": "fp32", "nrhs": 256, "graphs": False},
        # the mixed form's single matvec (the inner apply of a refinement)
        {"name": "apply_curve_fp32", "kind": "apply", "geometry": "curve", "layer": "single", "n": 1 << 19,
         "ppw": 10.0, "leaf": 64, "tol": 1e-8, "prec": "fp32", "nrhs": 1, "graphs": False},
        # a new small problem from its points on: trees, factorization in the
        # mixed form, first apply
        {"name": "factor_box_16k", "kind": "factor", "geometry": "box", "layer": "single", "n": 16384, "ppw": 8.0,
         "leaf": 64, "tol": 1e-8, "prec": "fp32", "nrhs": 1, "graphs": False},
        # a new large one, FP64
        {"name": "factor_curve_256k", "kind": "factor", "geometry": "curve", "layer": "single", "n": 1 << 18,
         "ppw": 10.0, "leaf": 64, "tol": 1e-8, "prec": "fp64", "nrhs": 1, "graphs": False},
        # independent problems of mixed sizes and leaf sizes as one operator,
        # 16 right-hand sides each, FP32
        {"name": "batch_16rhs_fp32", "kind": "batch", "problems": 16, "mix": 3, "low": 4096, "high": 65536,
         "ppw": 8.0, "tol": 1e-7, "prec": "fp32", "nrhs": 16, "graphs": False},
        # the boundary equation I/2 + (S + C)W solved for a plane wave
        {"name": "solve_64k", "kind": "solve", "n": 1 << 16, "ppw": 10.0, "leaf": 64, "tol": 1e-8, "graphs": False},
        # the streaming factorization of a matrix given by its columns
        {"name": "stream_2k", "kind": "stream", "n": 2048, "ppw": 10.0, "leaf": 64, "tol": 1e-7, "graphs": False},
    ]


def _log(rng, low, high):
    return int(round(low * (high / low) ** rng.random()))


def draw(rng):
    """One more case of the listed ranges: sizes and right-hand sides over
    their logarithm, any point count, every precision, layer and leaf size."""
    kind = rng.choice(["apply"] * 11 + ["factor"] * 3 + ["batch"] * 2 + ["solve"] * 2 + ["stream"] * 2)
    tol = 10.0 ** -rng.uniform(6, 9)
    leaf = rng.choice([32, 64, 128])
    graphs = rng.random() < 0.3
    if kind == "solve":
        return {"kind": kind, "n": _log(rng, 4096, 65536), "ppw": round(rng.uniform(8, 12), 2), "leaf": leaf,
                "tol": 10.0 ** -rng.uniform(7, 9), "graphs": graphs}
    if kind == "stream":
        return {"kind": kind, "n": _log(rng, 512, 2048), "ppw": round(rng.uniform(8, 12), 2), "leaf": 64, "tol": tol,
                "graphs": False}
    prec = rng.choice(["fp64", "fp64", "fp32", "fp32", "fp32x2"])
    if kind == "batch":
        return {"kind": kind, "problems": rng.randint(2, 16), "mix": rng.randint(0, 10 ** 6), "low": 4096,
                "high": 65536, "ppw": 8.0, "tol": tol, "prec": prec, "nrhs": _log(rng, 1, 64), "graphs": graphs}
    geometry = rng.choice(["curve", "curve", "box"])
    layer = rng.choice(["single", "single", "single", "double", "combined"]) if geometry == "curve" else "single"
    c = {"kind": kind, "geometry": geometry, "layer": layer, "n": _log(rng, 4096, 1 << 18),
         "ppw": round(rng.uniform(8, 12), 2), "leaf": leaf, "tol": tol, "prec": prec, "nrhs": 1, "graphs": graphs}
    if kind == "apply":
        # one, a few (2-15) and many (16-256) right-hand sides alike
        c["nrhs"] = rng.choice([1, _log(rng, 2, 15), _log(rng, 16, 256)])
    else:
        c["n"] = _log(rng, 4096, 1 << 17)
    return c


# ------------------------------------------------------------- the inputs


def _curve(n, ppw, turn):
    """Points, outward unit normals and trapezoid weights of the curve, the
    targets on the circle, and the wavenumber; `turn` shifts the parameter."""
    th = 2 * np.pi * (np.arange(n) + turn) / n
    c, s = np.cos(th), np.sin(th)
    r, dr = 1 + 0.3 * np.cos(5 * th), -1.5 * np.sin(5 * th)
    tx, ty = dr * c - r * s, dr * s + r * c
    speed = np.hypot(tx, ty)
    return (np.stack([r * c, r * s], 1), np.stack([ty, -tx], 1) / speed[:, None], speed * (2 * np.pi / n),
            np.stack([3 * c, 3 * s], 1), 2 * np.pi * n / (ppw * CURVE_L))


def _box(n, ppw, rng):
    src, tgt = rng.uniform(0, 1, (n, 2)), rng.uniform(0, 1, (n, 2))
    tgt[:, 0] += 2
    return src, tgt, 2 * np.pi * np.sqrt(n) / ppw


def _problems(case, seed):
    """[(sources, normals or None, targets, k, leaf)] of a case."""
    rng = np.random.RandomState(seed % (1 << 31))
    if case["kind"] == "batch":
        out, mix = [], np.random.RandomState(case["mix"])
        for i in range(case["problems"]):
            # sizes log-uniform over the range, the largest always among them
            at = 1.0 if i == 0 else mix.uniform()
            n = int(round(case["low"] * (case["high"] / case["low"]) ** at))
            leaf = int(mix.choice([32, 64, 128]))
            src, tgt, k = _box(n, case["ppw"], rng)
            out.append((src, None, tgt, k, leaf))
        return out
    if case.get("geometry") == "box":
        src, tgt, k = _box(case["n"], case["ppw"], rng)
        return [(src, None, tgt, k, case["leaf"])]
    src, nrm, _, tgt, k = _curve(case["n"], case["ppw"], rng.uniform())
    return [(src, nrm, tgt, k, case["leaf"])]


def _vectors(rows, cols, seed, prec="fp64"):
    """Standard complex Gaussian right-hand sides, row-major on the GPU."""
    g = torch.Generator(device="cuda").manual_seed(seed)
    x = torch.randn(rows, cols, 2, dtype=torch.float64, device="cuda", generator=g)
    return torch.view_as_complex(x if prec == "fp64" else x.float())


class _Buffer:
    """A torch tensor as the device buffer that the library's calls take."""

    def __init__(self, tensor):
        self.tensor, self.ptr = tensor, tensor.data_ptr()


def _helm(bf, k, layer="single"):
    if layer == "double":
        return bf.Helm2(k, bf.BF_LAYER_POTENTIAL_PV_DOUBLE)
    if layer == "combined":
        return bf.Helm2(k, bf.BF_LAYER_POTENTIAL_COMBINED_FIELD, *COMBINED)
    return bf.Helm2(k)


def _options(bf, tol):
    return bf.options(tol=tol, rank_const=RANK_CONST, pass_through=True, pinv_rcond=RCOND)


def _factor(bf, problem, case):
    """One problem's factorization in the case's precision, from its points."""
    src, nrm, tgt, k, leaf = problem
    layer = case.get("layer", "single")
    ts = bf.Quadtree(src, leaf, normals=nrm if layer != "single" else None, device=True)
    tt = bf.Quadtree(tgt, leaf, device=True)
    return _mixed(bf.FacHelm2.make_multilevel(_helm(bf, k, layer), ts, tt, _options(bf, case["tol"])), case["prec"])


def _mixed(fac, prec):
    if prec != "fp64":
        fac.orthogonalize()
        fac.prepare_mixed(prec, release_fp64=True)
    return fac


def _apply_state(fac, rows, cols, case, seed):
    x = _vectors(cols, case["nrhs"], seed, case["prec"])
    y = torch.empty(rows, case["nrhs"], dtype=x.dtype, device="cuda")
    return {"fac": fac, "x": _Buffer(x), "y": _Buffer(y)}


def prepare(case, seed):
    import butterfly_amd as bf

    kind = case["kind"]
    state = {"case": case, "bf": bf}
    problems = _problems(case, seed)
    if kind == "apply":
        n = case["n"]
        state.update(_apply_state(_factor(bf, problems[0], case), n, n, case, seed))
    elif kind == "factor":
        n = case["n"]
        state["problem"] = problems[0]
        state.update(_apply_state(None, n, n, case, seed))
    elif kind == "batch":
        trees = [(bf.Quadtree(s, leaf, device=True), bf.Quadtree(t, leaf, device=True))
                 for s, _, t, _, leaf in problems]
        fac = bf.FacHelm2.make_batched([bf.Helm2(p[3]) for p in problems], [t[0] for t in trees],
                                       [t[1] for t in trees], [_options(bf, case["tol"]) for _ in problems])
        n = sum(len(p[0]) for p in problems)
        state.update(_apply_state(_mixed(fac, case["prec"]), n, n, case, seed))
    elif kind == "solve":
        pts, _, w, _, k = _curve(case["n"], case["ppw"], np.random.RandomState(seed % (1 << 31)).uniform())
        tree = bf.Quadtree(pts, case["leaf"], device=True)
        fac = bf.FacHelm2.make_multilevel(bf.Helm2(k), tree, tree, _options(bf, case["tol"]))
        state["op"] = bf.BoundaryOperator(fac, bf.Helm2(k), tree, w, kr_order=6, alpha=0.5)
        state["b"] = _wave(pts, k, seed)[tree.perm]
    else:
        src, _, tgt, k, leaf = problems[0]
        ts, tt = bf.Quadtree(src, leaf, device=True), bf.Quadtree(tgt, leaf, device=True)
        sp, tp = src[ts.perm], tgt[tt.perm]
        # the column blocks in the order in which the streamer asks for them
        spans = sorted((a, b) for a, b in _leaf_spans(ts))
        state["trees"] = (tt, ts)
        state["blocks"] = [bf.Helm2(k).get_kernel_matrix(sp[a:b], tp) for a, b in spans]
        state["x"] = _vectors(case["n"], 1, seed)[:, 0].cpu().numpy()
    torch.cuda.synchronize()
    return state


def _leaf_spans(tree):
    for i in range(tree.num_nodes):
        node = tree.node(i)
        if all(c < 0 for c in node.child):
            yield int(node.offset[0]), int(node.offset[4])


def _wave(points, k, seed):
    """A plane wave; its direction comes from the seed."""
    angle = 2 * np.pi * np.random.RandomState((seed + 1) % (1 << 31)).uniform()
    return np.exp(1j * k * (points @ np.array([np.cos(angle), np.sin(angle)])))


def run(state):
    bf, case = state["bf"], state["case"]
    kind = case["kind"]
    bf.set_apply_graphs(case["graphs"])
    if kind == "solve":
        return state["op"].solve(state["b"], SOLVE_TOL, SOLVE_ITERATIONS)[0]
    if kind == "stream":
        rows, cols = state["trees"]
        streamer = bf.FacStreamer(rows, cols, case["tol"], init_depth=2, min_rows=20, min_cols=20)
        for block in state["blocks"]:
            streamer.feed(block)
        return streamer.fac().mat() @ state["x"]
    fac = state["fac"] if kind != "factor" else _factor(bf, state["problem"], case)
    bf.mul_device(fac, state["x"], state["y"], case["nrhs"], case["prec"])
    return state["y"].tensor


# ----------------------------------------------------------- what it costs

ELEM = {"fp64": 16, "fp32": 8, "fp32x2": 8}       # bytes of a vector entry
FACTOR = {"fp64": 16, "fp32": 8, "fp32x2": 16}    # bytes of a stored factor entry
_plans = {}


def _plan(case):
    """(stored entries, flops of the re-expansion solves) of the case's plan,
    for the inputs of seed 0: 84 p^3 + 16 p^2 n per truncated least-squares
    block of p x p against n columns."""
    key = repr(sorted((k, v) for k, v in case.items() if k != "name"))
    if key not in _plans:
        import butterfly_amd as bf

        entries = flops = 0.0
        problems = _problems(case, 0)
        if case["kind"] == "solve":
            src, _, _, _, k = _curve(case["n"], case["ppw"], 0.0)
            problems = [(src, None, src, k, case["leaf"])]
        for src, _, tgt, k, leaf in problems:
            ts = bf.Quadtree(src, leaf)
            tt = ts if tgt is src else bf.Quadtree(tgt, leaf)
            fac = bf.FacHelm2.plan_only(bf.Helm2(k), ts, tt, _options(bf, case["tol"]))
            entries += fac.stats()["entries"]
            if case["kind"] == "factor":
                blocks = fac.plan()[2]
                solved = blocks[blocks[:, 4] == 0].astype(np.float64)
                p, n = solved[:, 2], solved[:, 3]
                flops += float((84 * p ** 3 + 16 * p ** 2 * n).sum())
        _plans[key] = (entries, flops)
    return _plans[key]


def work(case):
    kind = case["kind"]
    if kind == "stream":
        # every entry is read once and meets an orthonormal basis of at least
        # a leaf's width once
        n = float(case["n"])
        return {"bytes": 16 * n * n, "flops": 8 * n * n * case["leaf"]}
    entries, flops = _plan(case)
    if kind == "solve":
        # four Krylov steps, each reading the factors once
        return {"bytes": 4 * 16.0 * (entries + 4 * case["n"]), "flops": 4 * 8.0 * entries}
    n = sum(len(p[0]) for p in _problems(case, 0)) if kind == "batch" else case["n"]
    vectors = 2.0 * n * case["nrhs"] * ELEM[case["prec"]]
    if kind == "factor":
        # the FP64 blocks are written once; the apply reads the stored form
        return {"bytes": 16.0 * entries + FACTOR[case["prec"]] * entries + vectors, "flops": flops + 8.0 * entries}
    return {"bytes": FACTOR[case["prec"]] * entries + vectors, "flops": 8.0 * entries * case["nrhs"]}


def tolerance(case):
    """About four times the largest distance from exact() seen over the
    ranges: on the curve 6 times the factorization's tolerance, in the box
    (whose rank estimate is far on the safe side) 0.01 times it, plus what
    FP32 vectors (3e-7 with split factors, 8e-7 with FP32 ones) cost; the
    solution of a boundary equation is off by 3.5e-10 when GMRES stops at
    1e-10, the streamed product by 0.5 times its tolerance."""
    kind, tol = case["kind"], case["tol"]
    if kind == "solve":
        return {"rel": 1.5e-9}
    if kind == "stream":
        return {"rel": 2 * tol}
    box = kind == "batch" or case["geometry"] == "box"
    rel = {"fp64": 0.0, "fp32": 3.2e-6, "fp32x2": 1.2e-6}[case["prec"]]
    return {"rel": rel + (0.05 if box else 25) * tol}


# ------------------------------------------------------ the same in 64 bits


def _order(points):
    """Positions of the points along their quadrant paths: the root square,
    halved at each level, quadrant 2 (x > sx) + (y > sy), stable."""
    lo, hi = points.min(0), points.max(0)
    w = hi - lo
    a = int(w[0] > w[1])  # the axis that is stretched
    c = (lo[a] + hi[a]) / 2
    lo[a], hi[a] = w[1 - a] * (lo[a] - c) / w[a] + c, w[1 - a] * (hi[a] - c) / w[a] + c
    low, high = np.tile(lo, (len(points), 1)), np.tile(hi, (len(points), 1))
    key = np.zeros(len(points), np.uint64)
    for _ in range(31):
        split = (low + high) / 2
        up = points > split
        key = (key << np.uint64(2)) | (2 * up[:, 0] + up[:, 1]).astype(np.uint64)
        low, high = np.where(up, split, low), np.where(up, high, split)
    return np.argsort(key, kind="stable")


def _kernel(k, tgt, src, nrm, layer):
    """(real, imaginary) parts of the layer's kernel, targets x sources."""
    dx, dy = tgt[:, None, 0] - src[None, :, 0], tgt[:, None, 1] - src[None, :, 1]
    r = torch.hypot(dx, dy)
    zero = r < 1e-15
    z = torch.where(zero, 1.0, k * r)
    re = im = torch.zeros((), dtype=torch.float64, device=r.device)
    if layer != "double":  # (i/4) H0(kr)
        re, im = -0.25 * torch.special.bessel_y0(z), 0.25 * torch.special.bessel_j0(z)
    if layer != "single":  # (i/4) k H1(kr) n.(t - s)/r
        f = 0.25 * k * (nrm[None, :, 0] * dx + nrm[None, :, 1] * dy) / torch.where(zero, 1.0, r)
        dre, dim = -f * torch.special.bessel_y1(z), f * torch.special.bessel_j1(z)
        if layer == "combined":
            a, b = complex(COMBINED[0]), complex(COMBINED[1])
            re, im = (a.real * re - a.imag * im + b.real * dre - b.imag * dim,
                      a.real * im + a.imag * re + b.real * dim + b.imag * dre)
        else:
            re, im = dre, dim
    return re.masked_fill(zero, 0.0), im.masked_fill(zero, 0.0)


def _dense(k, tgt, src, nrm, layer, x):
    """The dense kernel matrix times x, in row chunks."""
    dev = x.device
    tgt, src = torch.from_numpy(tgt).to(dev), torch.from_numpy(src).to(dev)
    nrm = torch.from_numpy(nrm).to(dev) if nrm is not None else None
    parts = torch.cat([x.real, x.imag], 1).contiguous()
    cols, y = x.shape[1], []
    step = max(1, (1 << 27) // len(src))
    for i in range(0, len(tgt), step):
        re, im = _kernel(k, tgt[i:i + step], src, nrm, layer)
        a, b = re @ parts, im @ parts
        y.append(torch.complex(a[:, :cols] - b[:, cols:], a[:, cols:] + b[:, :cols]))
    return torch.cat(y)


def _dense_boundary(k, pts, w, x):
    """alpha x + (S + C) W x of the boundary equation, points in any order
    with `w` and the neighbours of boundary order given by _order."""
    u = w * x
    y = 0.5 * x + _dense(k, pts, pts, None, "single", u[:, None])[:, 0]
    p = torch.from_numpy(pts).to(x.device)
    for q, g in enumerate(KR6):
        for shift in (q + 1, -q - 1):
            nb = torch.roll(p, -shift, 0)
            z = k * torch.hypot(p[:, 0] - nb[:, 0], p[:, 1] - nb[:, 1])
            e = torch.complex(-0.25 * torch.special.bessel_y0(z), 0.25 * torch.special.bessel_j0(z))
            y += g * e * torch.roll(u, -shift, 0)
    return y


def _gmres(op, b, tol, most):
    """Plain GMRES with modified Gram-Schmidt from a zero guess."""
    beta = torch.linalg.norm(b)
    basis, h = [b / beta], np.zeros((most + 1, most), complex)
    for j in range(most):
        v = op(basis[j])
        for i, q in enumerate(basis):
            c = torch.vdot(q, v)
            h[i, j] = complex(c)
            v = v - c * q
        h[j + 1, j] = float(torch.linalg.norm(v))
        rhs = np.zeros(j + 2, complex)
        rhs[0] = float(beta)
        y = np.linalg.lstsq(h[:j + 2, :j + 1], rhs, rcond=None)[0]
        if np.linalg.norm(h[:j + 2, :j + 1] @ y - rhs) <= tol * float(beta):
            break
        basis.append(v / h[j + 1, j].real)
    return sum(complex(c) * q for c, q in zip(y, basis))


def exact(case, seed):
    """The dense matrix in the place of its factorization.  None where its
    n^2 kernel values would take too long (about 2e9 a second)."""
    kind = case["kind"]
    if case.get("n", 0) > 181000:
        return None
    if kind == "solve":
        pts, _, w, _, k = _curve(case["n"], case["ppw"], np.random.RandomState(seed % (1 << 31)).uniform())
        b = torch.from_numpy(_wave(pts, k, seed)).cuda()
        w = torch.from_numpy(w).cuda()
        x = _gmres(lambda v: _dense_boundary(k, pts, w, v), b, 1e-13, SOLVE_ITERATIONS)
        return x.cpu().numpy()[_order(pts)]
    problems = _problems(case, seed)
    rows = sum(len(p[0]) for p in problems)
    x = _vectors(rows, case.get("nrhs", 1), seed, case.get("prec", "fp64")).to(torch.complex128)
    y, at = [], 0
    for src, nrm, tgt, k, _ in problems:
        so, to = _order(src), _order(tgt)
        layer = case.get("layer", "single")
        y.append(_dense(k, tgt[to], src[so], nrm[so] if layer != "single" else None, layer, x[at:at + len(src)]))
        at += len(src)
    y = torch.cat(y)
    return y[:, 0].cpu().numpy() if kind == "stream" else y

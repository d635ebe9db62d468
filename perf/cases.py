"""The work a user of this solver has it do, as measurable cases.

Every case is one pass through the public entry points of the Python binding,
from the smallest call (the pressure at one exterior point) to the largest
solve (40962 nodes, 32 point sources).  The surfaces are geodesic spheres of
frequency n (10 n^2 + 2 nodes, 20 n^2 triangles; n = 8, 16, 32, 64 have the
sizes of icosphere subdivisions 3 to 6), mapped to the sphere r = 0.1 m or to
the ellipsoid 0.075 / 0.09 / 0.11 m with up to 5 % of seeded bumps of degree 2
to 6.  Solutions of the FP32 paths are taken as complex64, the precision of the
assembled system; those of the FP64 path as complex128.
"""
import math

import numpy as np
import torch

import bem_gpu_clean_cpp_amd as bem

SPEED = 343.21  # m/s, the library's default medium (kg/m^3 below)
DENSITY = 1.2041

# boundary condition ca p + cb v = cc by name
BC = {
    "rigid": (0.0, 1.0, 0.0),
    "pulsating": (0.0, 1.0, -1.0),
    "impedance": (0.5 + 0.25j, 1.0 - 0.5j, 0.3 + 0.1j),
}
METHODS = {"qr": bem.SOLVE_QR, "gmres": bem.SOLVE_GMRES, "cgls": bem.SOLVE_CGLS, "block": bem.SOLVE_BLOCK_CG}
KINDS = {"plane": bem.RHS_PLANE, "point": bem.RHS_POINT}


def listed():
    return [
        # the end of the reference's driver: the exterior pressure at one point
        # of a small body, called point by point (latency)
        dict(name="point", path="point", n=8, shape="sphere", bc="pulsating", freq=171.5),
        # the small workload: 642 nodes, 8 CHIEF points, QR, and the field at
        # 64 points on r = 1 m
        dict(name="plain", path="plain", n=8, shape="sphere", bc="rigid", freq=171.0, chief=8, points=64),
        # the reference's driver on host buffers: the system, then the QR least
        # squares; an odd size (1692 nodes, 1 CHIEF point)
        dict(name="driver_qr", path="driver_qr", n=13, shape="ellipsoid", bc="pulsating", freq=500.0, chief=1),
        # the reference's other solver on host buffers: the square system, then
        # unrestarted GMRES (2562 nodes)
        dict(name="driver_gmres", path="driver_gmres", n=16, shape="sphere", bc="pulsating", freq=1000.0),
        # one plane wave on 10242 nodes at 2 kHz, 16 CHIEF points: GMRES on the
        # normal equations with FP64 refinement
        dict(name="single", path="solve", n=32, shape="sphere", bc="rigid", freq=2000.0, chief=16, rhs=1, kind="plane",
             method="gmres", precision=32),
        # a frequency sweep: 16 frequencies 100 Hz - 8 kHz x 16 plane waves on
        # one 2562-node mesh, 4 resident workers, lockstep GMRES
        dict(name="sweep", path="sweep", n=16, shape="ellipsoid", bc="rigid", flo=100.0, fhi=8000.0, nfreq=16, rhs=16),
        # the headline size: 40962 nodes, 12 kHz, 32 CHIEF points, 32 point
        # sources, block conjugate gradients
        dict(name="large", path="solve", n=64, shape="ellipsoid", bc="rigid", freq=12000.0, chief=32, rhs=32,
             kind="point", method="block", precision=32),
        # the all-FP64 option (complex128 matrix) on 5762 nodes
        dict(name="fp64", path="solve", n=24, shape="ellipsoid", bc="rigid", freq=2000.0, chief=16, rhs=4, kind="plane",
             method="gmres", precision=64),
        # an absorbing body (impedance terms) with a few point sources, each
        # right-hand side on its own, and the field at 100 points; 4412 nodes
        dict(name="impedance", path="solve_field", n=21, shape="ellipsoid", bc="impedance", freq=3000.0, chief=12,
             rhs=5, kind="point", method="cgls", points=100),
        # a field map: the radiation operator of 6001 points applied to 16
        # solutions at hand
        dict(name="field_map", path="field_map", n=16, shape="ellipsoid", bc="rigid", freq=2500.0, chief=16, rhs=16,
             points=6001),
        # the request server: 8 requests of uneven size at once on 4 slots
        dict(name="serve", path="serve", requests=8, nlo=8, nhi=32, rhslo=1, rhshi=32),
    ]


def _log(rng, lo, hi):
    return math.exp(rng.uniform(math.log(lo), math.log(hi)))


def _size(rng, lo, hi):
    return int(round(_log(rng, lo, hi)))


def _freq(rng, n, lo=0.2, hi=0.9):
    """A frequency with at least about 6 elements per wavelength (ka <= 0.9 n)
    and ka <= 20 on a body of radius 0.1 m."""
    return round(_log(rng, lo, min(20.0, hi * n)) * SPEED / (2 * math.pi * 0.1), 1)


def draw(rng):
    path = rng.choice(["point", "plain", "driver_qr", "driver_gmres", "solve", "solve", "sweep", "large", "fp64",
                       "solve_field", "field_map", "serve"])
    shape = rng.choice(["sphere", "ellipsoid"])
    kind = rng.choice(["plane", "point"])
    if path == "point":
        n = _size(rng, 4, 32)
        return dict(path=path, n=n, shape=shape, bc=rng.choice(["pulsating", "impedance"]), freq=_freq(rng, n))
    if path == "plain":
        n = _size(rng, 4, 12)
        return dict(path=path, n=n, shape=shape, bc="rigid", freq=_freq(rng, n), chief=rng.randint(8, 16),
                    points=_size(rng, 10, 1000))
    if path == "driver_qr":
        n = _size(rng, 5, 14)
        return dict(path=path, n=n, shape=shape, bc="pulsating", freq=_freq(rng, n, 0.2, 0.3),
                    chief=rng.randint(1, 8))
    if path == "driver_gmres":  # below the first interior resonance: the square system has no CHIEF points
        n = _size(rng, 6, 18)
        return dict(path=path, n=n, shape=shape, bc="pulsating", freq=_freq(rng, n, 0.2, 2.0 / n))
    if path == "solve":
        n = _size(rng, 12, 40)
        return dict(path=path, n=n, shape=shape, bc="rigid", freq=_freq(rng, n), chief=rng.randint(16, 32),
                    rhs=_size(rng, 1, 16), kind=kind, method=rng.choice(["gmres", "cgls", "block"]), precision=32)
    if path == "sweep":
        n = _size(rng, 8, 17)
        return dict(path=path, n=n, shape=shape, bc="rigid", flo=100.0, fhi=round(_freq(rng, n, 2.0, 0.6), 1),
                    nfreq=rng.randint(5, 16), rhs=rng.randint(2, 16))
    if path == "large":
        n = rng.randint(40, 63)
        return dict(path="solve", n=n, shape="ellipsoid", bc="rigid", freq=_freq(rng, n, 4.0, 0.3),
                    chief=rng.randint(24, 40), rhs=rng.randint(17, 32), kind=kind, method="block", precision=32)
    if path == "fp64":
        n = _size(rng, 6, 24)
        return dict(path="solve", n=n, shape=shape, bc="rigid", freq=_freq(rng, n, 0.2, 0.5),
                    chief=rng.randint(8, 16), rhs=rng.randint(1, 4), kind=kind, method="gmres", precision=64)
    if path == "solve_field":
        n = _size(rng, 8, 26)
        return dict(path=path, n=n, shape=shape, bc="impedance", freq=_freq(rng, n, 0.5, 0.6),
                    chief=rng.randint(8, 16), rhs=rng.randint(1, 8), kind=kind, method="cgls",
                    points=_size(rng, 1, 1000))
    if path == "field_map":
        n = _size(rng, 8, 18)
        return dict(path=path, n=n, shape=shape, bc="rigid", freq=_freq(rng, n, 0.2, 0.5), chief=16,
                    rhs=rng.randint(1, 32), points=_size(rng, 200, 6000))
    lo = rng.randint(6, 14)
    return dict(path=path, requests=rng.randint(3, 8), nlo=lo, nhi=rng.randint(lo + 4, 30), rhslo=1,
                rhshi=rng.randint(4, 32))


# ------------------------------------------------------------- geometry ---
def _geodesic(n):
    """Unit geodesic sphere of frequency n: (10 n^2 + 2, 3) nodes and
    (20 n^2, 3) triangles, counter-clockwise from inside, as the solver's
    meshes are wound (normals into the body)."""
    g = (1 + math.sqrt(5)) / 2
    v = np.array([(0, s, t * g) for s in (-1, 1) for t in (-1, 1)])
    v = np.concatenate([np.roll(v, r, axis=1) for r in range(3)])
    d = np.linalg.norm(v[:, None] - v[None], axis=2)
    faces = [(a, b, c) for a in range(12) for b in range(a + 1, 12) for c in range(b + 1, 12)
             if max(d[a, b], d[b, c], d[a, c]) < 2.001]
    ii = np.array([(i, j) for i in range(n + 1) for j in range(n + 1 - i)])
    at = {(i, j): q for q, (i, j) in enumerate(ii)}
    tri = []
    for i in range(n):
        for j in range(n - i):
            tri.append((at[i, j], at[i + 1, j], at[i, j + 1]))
            if i + j < n - 1:
                tri.append((at[i + 1, j], at[i + 1, j + 1], at[i, j + 1]))
    tri = np.array(tri)
    pts, els = [], []
    for q, f in enumerate(faces):
        A, B, C = v[list(f)]
        if np.dot(np.cross(B - A, C - A), A) > 0:  # outward: wind it the other way
            B, C = C, B
        pts.append((A * (n - ii.sum(1))[:, None] + B * ii[:, :1] + C * ii[:, 1:]) / n)
        els.append(tri + q * len(ii))
    pts, els = np.concatenate(pts), np.concatenate(els)
    key = np.round(pts * (1 << 18)).astype(np.int64)
    key = (key[:, 0] << 42) + (key[:, 1] << 21) + key[:, 2]
    _, first, back = np.unique(key, return_index=True, return_inverse=True)
    order = np.argsort(first)  # nodes in the order in which the faces bring them
    rank = np.empty(len(order), np.int64)
    rank[order] = np.arange(len(order))
    pts = pts[first[order]]
    return pts / np.linalg.norm(pts, axis=1, keepdims=True), rank[back.ravel()][els].astype(np.int32)


def _directions(rng, count):
    v = rng.standard_normal((count, 3))
    return v / np.linalg.norm(v, axis=1, keepdims=True)


def _surface(n, shape, rng):
    """Nodes (float32) and triangles of a seeded body."""
    u, els = _geodesic(n)
    axes = np.full(3, 0.1) if shape == "sphere" else np.array([0.075, 0.09, 0.11])
    degree = rng.integers(2, 7, 8)
    amp = rng.uniform(-1, 1, 8) * (0.01 if shape == "sphere" else 0.05) / 8
    f = np.ones(len(u))
    for l, a, d in zip(degree, amp, _directions(rng, 8)):
        f += a * np.polynomial.legendre.legval(u @ d, [0] * l + [1])
    return (u * axes * f[:, None]).astype(np.float32), els


def _ball(rng, count, radius):
    return (_directions(rng, count) * radius * rng.random((count, 1)) ** (1 / 3)).astype(np.float32)


def _sources(rng, kind, count, pts):
    """Plane-wave directions, or point sources 1 cm outside the surface."""
    if kind == "plane":
        return _directions(rng, count).astype(np.float32)
    p = pts[rng.choice(len(pts), count, replace=False)].astype(np.float64)
    return (p * (1 + 0.01 / np.linalg.norm(p, axis=1, keepdims=True))).astype(np.float32)


def _wavenumber(freq):
    return float(np.float32(2 * np.pi * freq / SPEED))


def _problems(case, seed):
    """What the case computes on, from the seed alone: a list of requests, each
    with its mesh arrays and right-hand sides."""
    rng = np.random.default_rng(seed)
    if case["path"] == "serve":
        out = []
        for i in range(case["requests"]):
            # sizes, frequencies and counts belong to the case, not to the seed
            c = np.random.default_rng(1000 * case["nlo"] + 10 * case["nhi"] + i)
            n = int(round(math.exp(c.uniform(math.log(case["nlo"]), math.log(case["nhi"])))))
            one = dict(n=n, shape=("sphere", "ellipsoid")[i % 2], chief=16, rhs=int(c.integers(case["rhslo"],
                       case["rhshi"] + 1)), kind=("plane", "point")[int(c.integers(2))], bc="rigid",
                       freq=float(c.uniform(0.5, min(20.0, 0.9 * n))) * SPEED / (2 * math.pi * 0.1))
            out.append(_problem(one, rng))
        return out
    return [_problem(case, rng)]


def _problem(case, rng):
    pts, els = _surface(case["n"], case["shape"], rng)
    p = dict(pts=pts, els=els, bc=BC[case["bc"]], chief=_ball(rng, case.get("chief", 0), 0.05))
    if case["shape"] == "ellipsoid":
        p["chief"] = (p["chief"] * 0.8).astype(np.float32)
    kind = case.get("kind", "plane")
    p["kind"] = kind
    if "freq" in case:
        p["k"] = _wavenumber(case["freq"])
        p["params"] = _sources(rng, kind, case.get("rhs", 1), pts)
    else:
        p["ks"] = np.array([_wavenumber(f) for f in np.geomspace(case["flo"], case["fhi"], case["nfreq"])], np.float32)
        p["params"] = np.stack([_sources(rng, kind, case["rhs"], pts) for _ in p["ks"]])
    if "points" in case or case.get("path") == "point":
        p["xs"] = (_directions(rng, case.get("points", 1)) * rng.uniform(0.3, 1.0)).astype(np.float32)
    if case.get("path") == "point":  # a smooth surface pressure
        q = pts.astype(np.float64) @ (_directions(rng, 1)[0] * p["k"])
        p["surf"] = ((1 + 0.3 * rng.standard_normal()) * np.exp(-1j * q)).astype(np.complex64)
    return p


def _mesh(p):
    m = bem.Mesh().set(p["pts"], p["els"], p["bc"])
    if len(p["chief"]):
        m.set_chief(p["chief"])
    return m


_REFINED = dict(restart=30, tol=1e-6, maxit=6000, refine_tol=1e-10, max_refine=50)
_FULL = dict(restart=30, tol=1e-6, maxit=6000, refine_tol=1e-12, max_refine=50)


def prepare(case, seed):
    """The meshes, and the solver, batch or server handle that a user's program
    keeps between its calls."""
    ps = _problems(case, seed)
    meshes = [_mesh(p) for p in ps]
    p, m, path = ps[0], meshes[0], case["path"]
    s = dict(case=case, ps=ps, meshes=meshes)
    if path in ("plain", "solve", "solve_field", "field_map"):
        s["solver"] = bem.Solver(m)
    elif path == "sweep":
        s["batch"] = bem.Batch(m, 4)
    elif path == "serve":
        s["server"] = bem.Server(slots=4)
    elif path == "point":  # the mesh is resident before the points are asked for
        bem.ext_pressure(p["k"], m, (0, 0, 0), p["xs"][0], p["surf"])
    if path == "field_map":  # solutions at hand
        sv = s["solver"]
        sv.assemble(p["k"], bem.PREC_FP32)
        sv.set_rhs(KINDS[p["kind"]], p["params"], 1.0)
        sv.solve(METHODS["block"], **_REFINED)
    return s


def run(state):
    case, p, m = state["case"], state["ps"][0], state["meshes"][0]
    path = case["path"]
    if path == "point":
        return np.array([bem.ext_pressure(p["k"], m, (1e6, 1e6, 1e6), p["xs"][0], p["surf"])], np.complex64)
    if path == "driver_qr":
        A, B = bem.bem_system(m, p["k"], [[1e6, 1e6, 1e6]])
        return {"A": A, "B": B, "x": bem.qr_solve(A, B)}
    if path == "driver_gmres":
        A, B = bem.bem_system(m, p["k"], [[1e6, 1e6, 1e6]])
        return {"x": bem.gmres(A, B[:, 0], 200, 1e-6)}
    if path == "sweep":
        X, _ = state["batch"].run(p["ks"], KINDS[p["kind"]], p["params"], 1.0, bem.PREC_FP32, method=METHODS["gmres"],
                                  restart=100, tol=1e-6, maxit=6000, refine_tol=1e-8, max_refine=50)
        return X.astype(np.complex64)
    if path == "serve":
        sv = state["server"]
        ids = [sv.submit(mm, q["k"], KINDS[q["kind"]], q["params"], 1.0, bem.PREC_FP32, method=METHODS["block"],
                         **_REFINED) for q, mm in zip(state["ps"], state["meshes"])]
        return [sv.wait(i)[0].astype(np.complex64) for i in ids]
    sv = state["solver"]
    if path == "field_map":
        return sv.field_matrix(p["xs"]).field_apply()
    double = case.get("precision") == 64
    sv.assemble(p["k"], bem.PREC_FP64 if double else bem.PREC_FP32)
    sv.set_rhs(KINDS[p["kind"]], p["params"], 1.0)
    if path == "plain":
        sv.solve(METHODS["qr"], refine_tol=1e-10, max_refine=10)
        x = sv.solution(fp64=False)
        return {"x": x, "field": sv.field_matrix(p["xs"]).field_apply()}
    sv.solve(METHODS[case["method"]], **(_FULL if double else _REFINED))
    x = sv.solution(fp64=double)
    return {"x": x, "field": sv.field(p["xs"])} if path == "solve_field" else {"x": x}


# ----------------------------------------------------------------- work ---
FLOP_PER_POINT = 80.0  # one kernel evaluation of the 6 x 6 rule (G, dG/dn, shape functions)


def work(case):
    """Bytes: the mesh and the results, and a matrix that is formed once and
    read once (a solver cannot do with less), at its element size.  Flops: the
    6 x 6 rule for every pair of row and element, and the least an answer
    takes from the matrix: the QR factorisation where that is the method, else
    one product with each right-hand side."""
    sizes = []
    if case["path"] == "serve":
        for i in range(case["requests"]):
            c = np.random.default_rng(1000 * case["nlo"] + 10 * case["nhi"] + i)
            n = int(round(math.exp(c.uniform(math.log(case["nlo"]), math.log(case["nhi"])))))
            sizes.append((n, 16, int(c.integers(case["rhslo"], case["rhshi"] + 1))))
    else:
        sizes = [(case["n"], case.get("chief", 0), case.get("rhs", 1))] * case.get("nfreq", 1)
    size = 16.0 if case.get("precision") == 64 else 8.0
    total = {"bytes": 0.0, "flops": 0.0}
    for n, chief, R in sizes:
        N, E = 10.0 * n * n + 2, 20.0 * n * n
        M = N + chief
        P = float(case.get("points", 1 if case["path"] == "point" else 0))
        total["bytes"] += 12 * M + 40 * E + size * N * R
        if case["path"] in ("point", "field_map"):
            total["bytes"] += 20 * P * R + (2 * size * P * N if case["path"] == "field_map" else 0)
            total["flops"] += 36 * FLOP_PER_POINT * P * E + 8 * P * N * R
            continue
        total["bytes"] += 2 * size * M * N + 8 * P * R
        total["flops"] += 36 * FLOP_PER_POINT * (M + P) * E
        qr = case["path"] in ("plain", "driver_qr")
        total["flops"] += 8 * M * N * N - 8 * N ** 3 / 3 if qr else 8 * M * N * R
    return total


# ------------------------------------------------- the same in 64 bits ---
def _rule(shape):
    """Points and weights of the 6 x 6 collapsed Gauss-Legendre rule on the
    triangle: `shape` None for the regular rule, else the vertex that the
    square collapses to."""
    x, w = np.polynomial.legendre.leggauss(6)
    th, rh = np.meshgrid(0.5 + 0.5 * x, 0.5 + 0.5 * x, indexing="ij")
    W = 0.25 * np.outer(w, w) * rh
    one = {None: (rh * (1 - th), rh * th), 0: (1 - rh, rh * (1 - th)), 1: (rh * th, 1 - rh),
           2: (rh * (1 - th), rh * th)}[shape]
    return np.stack([one[0].ravel(), one[1].ravel(), 1 - one[0].ravel() - one[1].ravel()], 1), W.ravel()


def _kernels(x, tri, k, shape):
    """h (.., 3), g (.., 3) and c of the elements `tri` (E, 3, 3) seen from the
    points x (broadcast against E)."""
    e1, e2 = tri[:, 0] - tri[:, 2], tri[:, 1] - tri[:, 2]
    nrm = torch.linalg.cross(e1, e2)
    J = torch.linalg.norm(nrm, dim=1)
    nrm = nrm / J[:, None]
    h, g, c = [0, 0, 0], [0, 0, 0], 0
    for N, w in zip(*_rule(shape)):
        y = float(N[0]) * tri[:, 0] + float(N[1]) * tri[:, 1] + float(N[2]) * tri[:, 2]
        d = [y[:, a] - x[..., a] for a in range(3)]
        r = torch.sqrt(d[0] * d[0] + d[1] * d[1] + d[2] * d[2])
        drdn = (d[0] * nrm[:, 0] + d[1] * nrm[:, 1] + d[2] * nrm[:, 2]) / r
        wJ = float(w) * J / (4 * math.pi)
        G = torch.polar(wJ / r, -k * r)
        H = G * torch.complex(-drdn / r, -k * drdn)
        c = c - wJ * drdn / (r * r)
        for j in range(3):
            h[j] = h[j] + float(N[j]) * H
            g[j] = g[j] + float(N[j]) * G
    return h, g, c


def _system64(p, k, xs=None):
    """The collocation system (A, boundary term) for the nodes and CHIEF
    points, or the radiation operator of the points xs."""
    dev = "cuda" if torch.cuda.is_available() else "cpu"
    t = lambda a: torch.from_numpy(np.asarray(a)).to(dev, torch.float64)  # noqa: E731
    pts, N = t(p["pts"]), len(p["pts"])
    els = torch.from_numpy(p["els"].astype(np.int64)).to(dev)
    tri = pts[els]
    E = len(els)
    X = torch.cat([pts, t(p["chief"])]) if xs is None else t(xs)
    ca, cb, cc = (complex(np.complex64(z)) for z in p["bc"])
    beta, gamma = ca / cb, cc / cb
    irw = 1j * float(np.float32(DENSITY)) * k * float(np.float32(SPEED))
    own = [_kernels(tri[:, v], tri, k, v) for v in range(3)] if xs is None else None
    A = torch.zeros(len(X), N, dtype=torch.complex128, device=dev)
    b = torch.zeros(len(X), dtype=torch.complex128, device=dev)
    step = max(1, int(2e7) // E)
    for r0 in range(0, len(X), step):
        r1 = min(len(X), r0 + step)
        h, g, c = _kernels(X[r0:r1, None, :], tri, k, None)
        if own is not None:
            for v in range(3):  # elements that hold the row's node: the rule collapsed to it
                e = torch.nonzero((els[:, v] >= r0) & (els[:, v] < min(r1, N)))[:, 0]
                row = els[e, v] - r0
                for j in range(3):
                    h[j][row, e] = own[v][0][j][e]
                    g[j][row, e] = own[v][1][j][e]
                c[row, e] = own[v][2][e]
        view = torch.view_as_real(A[r0:r1])
        for j in range(3):
            view.index_add_(1, els[:, j], torch.view_as_real(h[j] - beta * irw * g[j]))
        b[r0:r1] = (gamma * irw) * (g[0] + g[1] + g[2]).sum(1)
        if own is not None:
            i = torch.arange(r0, min(r1, N), device=dev)
            A[i, i] += 1 - c.sum(1)[: len(i)]
    return A, b


def _incident64(p, k, x, params, amp):
    dev = x.device
    q = torch.from_numpy(np.asarray(params, np.float64)).to(dev)
    if p["kind"] == "plane":
        return torch.polar(torch.full((len(x), len(q)), amp, dtype=torch.float64, device=dev), -k * (x @ q.T))
    r = torch.linalg.norm(x[:, None, :] - q[None], dim=2)
    return torch.polar(amp / (4 * math.pi * r), -k * r)


def _least_squares64(A, B):
    """min |A X - B| by the normal equations, refined twice."""
    if A.shape[0] == A.shape[1]:
        return torch.linalg.solve(A, B)
    Ah = A.conj().T.resolve_conj().contiguous()
    lu = torch.linalg.lu_factor(Ah @ A)
    x = torch.linalg.lu_solve(*lu, Ah @ B)
    for _ in range(2):
        x = x + torch.linalg.lu_solve(*lu, Ah @ (B - A @ x))
    return x


def _solve64(p, k, params, amp):
    A, b = _system64(p, k)
    X = torch.from_numpy(np.concatenate([p["pts"], p["chief"]]).astype(np.float64)).to(A.device)
    inc = _incident64(p, k, X, params, amp) if amp else 0
    B = inc - b[:, None]
    return A, B, _least_squares64(A, B)


def _field64(p, k, x, params, amp):
    F, b = _system64(p, k, p["xs"])
    X = torch.from_numpy(p["xs"].astype(np.float64)).to(F.device)
    inc = _incident64(p, k, X, params, amp) if amp else 0
    return inc - b[:, None] - F @ x


def exact(case, seed):
    """run()'s outputs in 64 bits; None for the largest bodies, whose dense
    factorisation takes too long."""
    path = case["path"]
    if case.get("n", case.get("nhi", 0)) > 36:
        return None
    ps = _problems(case, seed)
    p = ps[0]
    if path == "point":
        x = torch.from_numpy(p["surf"].astype(np.complex128)[:, None])
        return _field64(p, p["k"], x.to("cuda" if torch.cuda.is_available() else "cpu"), None, 0)[:, 0]
    if path == "sweep":
        return torch.stack([_solve64(p, float(k), q, 1.0)[2] for k, q in zip(p["ks"], p["params"])], 2)
    if path == "serve":
        return [_solve64(q, q["k"], q["params"], 1.0)[2] for q in ps]
    host = path.startswith("driver")  # the source strength is 0 by default
    A, B, x = _solve64(p, p["k"], np.zeros((1, 3)) if host else p["params"], 0.0 if host else 1.0)
    if path == "driver_qr":
        return {"A": A, "B": B, "x": x}
    if path == "driver_gmres":
        return {"x": x[:, 0]}
    if path == "solve":
        return {"x": x}
    f = _field64(p, p["k"], x, p["params"], 1.0)
    return f if path == "field_map" else {"x": x, "field": f}

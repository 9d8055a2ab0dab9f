"""The workloads this library is timed on: what a solver, a wave-propagation loop or an inversion
asks of it through its public entry points, from the smallest mesh (launch-bound) to the benchmark
mesh (24^3 Kuhn cubes, P4), with the FP64 value of every output from plain torch.

A case is a dict of plain values:
  what      "apply" (the MatShell's y = A x), "assembled" (the same through the assembled block rows),
            "jacobi" (element-block Jacobi application), "gradient" (adjoint lambda / mu gradient),
            "wave" (M^-1 (A x - b)), "solve" (p-multigrid solve to 1e-10)
  kind      "elasticity" or "poisson";  dim, degree, n0, n1, n2 (cells of the box, n2 = 0 in 2D)
  dtype     "f64" or "f32" vectors;  cols: columns handled by one call
  free      natural boundary on the last axis' upper side (a free surface), Dirichlet elsewhere
  mixed     vertex ids permuted, as a mesh generator numbers them (every pair of local faces meets)
"""
import itertools
import math
import os

import numpy as np
import torch

import tandem_amd as T

RULES = os.path.join(os.path.dirname(os.path.abspath(T.__file__)), "data", "simplex_rules.txt")
LEVELS = {2: (2, 1), 3: (3, 1), 4: (4, 2, 1), 6: (6, 3, 1)}  # p-multigrid hierarchies by fine degree


def _case(name, what, kind, dim, degree, n, dtype="f64", cols=1, free=False, mixed=False):
    n = tuple(n) + (0,) * (3 - len(n))
    return {"name": name, "what": what, "kind": kind, "dim": dim, "degree": degree, "n0": n[0], "n1": n[1], "n2": n[2],
            "dtype": dtype, "cols": cols, "free": free, "mixed": mixed}


def listed():
    return [
        # the benchmark's smallest problem: antiplane P2 on 2,048 triangles, one launch of a few us
        _case("poisson_p2_2d_small", "apply", "poisson", 2, 2, (32, 32)),
        # a 2D antiplane earthquake-cycle mesh: Poisson P4, 51,200 triangles with mesh-generator numbering
        _case("poisson_p4_2d", "apply", "poisson", 2, 4, (160, 160), free=True, mixed=True),
        # a rank's share or a test mesh: 384 P4 tetrahedra, where the launches count
        _case("apply_p4_small", "apply", "elasticity", 3, 4, (4, 4, 4)),
        # the headline: the FP64 MatShell mult on 82,944 P4 tetrahedra (8.7 million unknowns)
        _case("apply_p4_box24", "apply", "elasticity", 3, 4, (24, 24, 24)),
        # the mult of the FP32 inner solve and of the FP32 V-cycle
        _case("apply_p4_f32", "apply", "elasticity", 3, 4, (20, 20, 20), dtype="f32"),
        # an odd-sized P2 mesh (a p-multigrid middle level) under a free surface, arbitrary numbering
        _case("apply_p2_ragged", "apply", "elasticity", 3, 2, (13, 17, 11), free=True, mixed=True),
        # a block of 64 Green's-function columns: plane strain P6 in FP32 (the fine level of its V-cycle)
        _case("apply_p6_2d_64cols", "apply", "elasticity", 2, 6, (96, 96), dtype="f32", cols=64, free=True, mixed=True),
        # the coarse level of that solve: assembled P1 block rows times 64 columns
        _case("assembled_p1_2d_64cols", "assembled", "elasticity", 2, 1, (200, 200), dtype="f32", cols=64, free=True,
              mixed=True),
        # one gradient of the inversion for lambda and mu
        _case("gradient_p4_f32", "gradient", "elasticity", 3, 4, (16, 16, 16), dtype="f32", free=True),
        # the preconditioner of the FP64 CG
        _case("jacobi_p4", "jacobi", "elasticity", 3, 4, (12, 12, 12)),
        # the right-hand side of an explicit elastic-wave step with moving Dirichlet boundaries
        _case("wave_p3", "wave", "elasticity", 3, 3, (15, 14, 16), free=True, mixed=True),
        # a whole linear solve to 1e-10 (p-multigrid preconditioned flexible CG)
        _case("solve_p4", "solve", "elasticity", 3, 4, (8, 8, 8)),
    ]


def draw(rng):
    what = rng.choice(["apply"] * 5 + ["assembled", "jacobi", "gradient", "wave", "solve"])
    kind = "poisson" if what == "apply" and rng.random() < 0.25 else "elasticity"
    dim = rng.choice([2, 3, 3])
    degrees = {"apply": (1, 2, 3, 4, 5, 6), "assembled": (1, 2), "jacobi": (1, 2, 3, 4, 6), "gradient": (2, 3, 4, 6),
               "wave": (2, 3, 4, 5, 6), "solve": (2, 3, 4, 6)}[what]
    degree = rng.choice([p for p in degrees if p <= (6 if dim == 2 else 1 if what == "assembled" else 4)])
    cols, dtype = 1, "f64"
    if what in ("apply", "assembled"):
        dtype = rng.choice(["f64", "f32"])
        cols = rng.choice([1, 1, 1, 2, 8, 17, 64]) if what == "apply" else rng.choice([1, 8, 37, 64])
    if what == "gradient":
        dtype = rng.choice(["f64", "f32"])
    # unknowns (all columns) over their logarithm; the set-up of the largest stays a few seconds
    hi = {"apply": 3e6 * min(cols, 16), "assembled": 2.5e5 * cols, "jacobi": 1e6, "gradient": 2.5e6, "wave": 1e6,
          "solve": 2e5}[what]
    total = math.exp(rng.uniform(math.log(4e3 * cols), math.log(hi)))
    comps = dim if kind == "elasticity" else 1
    per_cell = (2 if dim == 2 else 6) * math.comb(degree + dim, dim) * comps
    n = max(2.0, (total / cols / per_cell) ** (1.0 / dim))
    sides = [max(2, round(n * math.exp(rng.uniform(-0.25, 0.25)))) for _ in range(dim)]
    c = _case("", what, kind, dim, degree, sides, dtype, cols, rng.random() < 0.5, rng.random() < 0.7)
    del c["name"]
    return c


# ------------------------------------------------------------------------------ inputs (no library code)
def _cells(case):
    return [case["n%d" % d] for d in range(case["dim"])]


def _mesh(case):
    """Vertices, elements (ascending vertex ids), boundary facets and their conditions of the unit box."""
    D, n = case["dim"], _cells(case)
    grid = np.stack(np.meshgrid(*[np.arange(k + 1) for k in n], indexing="ij"), -1).reshape(-1, D)
    stride = np.array([int(np.prod([k + 1 for k in n[d + 1:]])) for d in range(D)])
    cell = np.stack(np.meshgrid(*[np.arange(k) for k in n], indexing="ij"), -1).reshape(-1, D) @ stride
    paths = [[0] + list(np.cumsum([stride[a] for a in p])) for p in itertools.permutations(range(D))]
    el = (cell[:, None, None] + np.array(paths)[None]).reshape(-1, D + 1)
    v = grid / np.array(n, dtype=np.float64)
    if case["mixed"]:
        p = np.random.default_rng(11).permutation(len(v))
        w = np.empty_like(v)
        w[p] = v
        v, el = w, p[el]
    el = np.sort(el, axis=1)
    faces, key = _faces(el, len(v))
    _, first, count = np.unique(key, return_index=True, return_counts=True)
    bnd = faces.reshape(-1, D)[first[count == 1]]
    up = v[bnd].mean(axis=1)[:, D - 1] > 1.0 - 1e-9
    return v, el.astype(np.int64), bnd, np.where(up & case["free"], T.BC_NATURAL, T.BC_DIRICHLET).astype(np.int32)


def _faces(el, nv):
    """Vertices of every element face (face f leaves out vertex D - f) and one integer per vertex set."""
    D = el.shape[1] - 1
    faces = np.stack([np.delete(el, D - f, axis=1) for f in range(D + 1)], axis=1)
    key = np.zeros(faces.shape[:2], dtype=np.int64)
    for d in range(D):
        key = key * nv + faces[:, :, d]
    return faces, key.ravel()


def _field(dim, mean, length, rng, device):
    """A log-normal coefficient of standard deviation 0.3 as a function of points (..., dim)."""
    w = torch.tensor(rng.normal(scale=1.0 / length, size=(dim, 64)), device=device)
    b = torch.tensor(rng.uniform(0.0, 2.0 * np.pi, size=64), device=device)

    def f(X):
        flat = X.reshape(-1, dim)
        g = torch.cat([torch.cos(p @ w + b).sum(-1) for p in flat.split(1 << 18)])
        return (mean * torch.exp(0.3 * math.sqrt(2.0 / 64) * g - 0.045)).reshape(X.shape[:-1])

    return f


def _inputs(case, seed, device):
    """Coefficient functions, the vectors and the boundary data of a seed."""
    D, rng = case["dim"], np.random.default_rng([seed, 5])
    length = 0.2 if min(_cells(case)) >= 8 else 1.0  # coarse meshes do not resolve the short one
    fields = [_field(D, 2.0, length, rng, device), _field(D, 1.0, length, rng, device)]
    E = math.factorial(D) * int(np.prod(_cells(case)))
    comps = D if case["kind"] == "elasticity" else 1
    width = E * math.comb(case["degree"] + D, D) * comps
    gen = torch.Generator(device=device).manual_seed(seed + 17)
    dt = torch.float64 if case["dtype"] == "f64" else torch.float32
    X = torch.rand((2 if case["what"] == "gradient" else case["cols"], width), generator=gen, device=device, dtype=dt)
    wave = torch.tensor(rng.normal(size=(D, D)), device=device)
    return fields, X * 2.0 - 1.0, lambda P: torch.sin(P @ wave)  # facet data: one smooth value per component


def _warped(X):
    return X + 0.02 * torch.prod(torch.sin(2.0 * math.pi * X), dim=-1, keepdim=True)


# ------------------------------------------------------------------------------ the library's side
def _operator(case, degree, mesh, nodes, fields, device):
    op = T.DGOperator(mesh, T.ELASTICITY if case["kind"] == "elasticity" else T.POISSON, degree, nodes)
    P = torch.from_numpy(op.volume_points()).to(device)
    c = [f(P).cpu().numpy() for f in fields]
    op.set_material(c[0], c[1] if case["kind"] == "elasticity" else None)
    op.upload()
    return op


def prepare(case, seed):
    dev = torch.device("cuda")
    mesh = T.Mesh(*_mesh(case))
    fields, X, data = _inputs(case, seed, dev)
    what, s = case["what"], {"what": case["what"]}
    degrees = LEVELS[case["degree"]] if what == "solve" else (case["degree"],)
    ops = []
    for p in degrees:
        # the curved map of every level is the fine level's, interpolated at the level's own nodes
        nodes = torch.from_numpy(mesh.affine_nodes(p)).to(dev)
        ops.append(_operator(case, p, mesh, _warped(nodes).cpu().numpy(), fields, dev))
    op = s["op"] = ops[0]
    if what == "apply" and case["cols"] > 1:
        op.autotune(case["cols"], "fp64" if case["dtype"] == "f64" else "fp32")
    if what == "assembled":
        op.assemble()
        op.set_variant("assembled")
    if what == "jacobi":
        op.block_jacobi_build()
    if what == "wave":
        s["facet"] = data(torch.from_numpy(op.facet_points()).to(dev)).transpose(1, 2).contiguous().view(-1)
    if what == "solve":
        s["mg"] = T.PMultigrid(ops, galerkin_penalty=0)
        s["mg"].setup()
    if what == "gradient":
        s["g"] = [torch.empty(op.E * op.Nq, dtype=X.dtype, device=dev) for _ in range(2)]
    s["x"], s["y"] = X, torch.empty_like(X)
    torch.cuda.synchronize()
    return s


def run(s):
    op, x, y, what = s["op"], s["x"], s["y"], s["what"]
    if what in ("apply", "assembled"):
        return op.apply(x[0], y[0]) if x.shape[0] == 1 else op.apply_batched(x, y)
    if what == "jacobi":
        return op.block_jacobi_apply(x[0], y[0])
    if what == "gradient":
        return list(op.material_gradient(x[0], x[1], *s["g"]))
    if what == "wave":
        return op.wave_rhs(x[0], s["facet"], y[0])
    s["mg"].solve_multi(x, y)
    return y[0]


# ------------------------------------------------------------------------------ what a pass needs
def _sizes(case):
    D, N, n = case["dim"], case["degree"], _cells(case)
    E = math.factorial(D) * int(np.prod(n))
    bnd = 2 * sum(int(np.prod(n)) // k for k in n) * (2 if D == 3 else 1)
    Nq = {2: (4, 7, 15, 19, 28, 37), 3: (6, 14, 31, 57)}[D][N - 1]
    nq = N + 1 if D == 2 else (4, 7, 15, 19)[N - 1]
    return E, (E * (D + 1) + bnd) // 2, math.comb(N + D, D), math.comb(N + D - 1, D - 1), Nq, nq


def work(case):
    """Bytes: vectors and results once, and the operator as its geometry nodes, nodal coefficients,
    penalties and neighbours (or its blocks).  Flops: the reference's contractions, with the values and
    the tangential derivatives on a face taken over the face's own nodes."""
    D, r, what = case["dim"], 8 if case["dtype"] == "f64" else 4, case["what"]
    E, F, nbf, nf, Nq, nq = _sizes(case)
    Q = D if case["kind"] == "elasticity" else 1
    bs, cols = nbf * Q, case["cols"]
    plan = r * (E * nbf * (D + (2 if Q > 1 else 1)) + F) + 4 * E * 2 * (D + 1)
    on_face = (D * nf + nbf) if Q > 1 else (D + 1) * nbf  # the modal basis has no face nodes
    vol = E * (4 * D * Nq * nbf * Q + (4 * D * D * Q + 3 * D * D + 2 * D) * Nq)
    fct = F * 2 * (4 * nq * on_face * Q + 8 * D * D * nq * Q)
    if what == "apply":
        return {"bytes": plan + 2 * r * E * bs * cols, "flops": (vol + fct) * cols}
    if what == "assembled":
        return {"bytes": r * E * ((D + 2) * bs * bs + 2 * bs * cols), "flops": 2 * E * (D + 2) * bs * bs * cols}
    if what == "jacobi":
        return {"bytes": r * E * (bs * (bs + 1) // 2 + 2 * bs), "flops": 2 * E * bs * bs}
    if what == "gradient":
        return {"bytes": plan + r * E * (2 * bs + 2 * Nq), "flops": vol + fct + E * (8 * Nq * nbf + 4 * nbf * nbf)}
    if what == "wave":
        return {"bytes": plan + 2 * r * E * bs, "flops": vol + fct + E * Q * (4 * nbf * nbf + 4 * nbf * Nq)}
    # a solve: about 100 iterations of one FP64 apply and a V-cycle of 13 FP32 applies on the fine level
    return {"bytes": 100 * (plan + 2 * r * E * bs + 13 * (plan + 2 * r * E * bs) // 2), "flops": 1400 * (vol + fct)}


def tolerance(case):
    """About four times the difference from exact() that was measured over listed and drawn cases."""
    what, f64 = case["what"], case["dtype"] == "f64"
    if what == "solve":
        return {"rel": 5e-7}  # any two solutions stop at a relative residual of 1e-10: 6e-10 to 5e-8
    if not f64:
        return {"rel": 2e-6 if what == "gradient" else 1e-6}  # 3.7e-7 and 1e-7 to 2e-7
    # 5e-15 to 2e-13; the gradient adds the projection's solve
    return {"rel": 2e-12 if what == "gradient" else 8e-13}


# ------------------------------------------------------------------------------ FP64 values in plain torch
def _exponents(D, N):
    if D == 1:
        return [(a,) for a in range(N + 1)]
    if D == 2:
        return [(s - b, b) for s in range(N + 1) for b in range(s + 1)]
    return [(a - b, b - c, c) for a in range(N + 1) for b in range(a + 1) for c in range(b + 1)]


def _jacobi(n, a, x, y):
    """y^n P_n^(a,0)(x / y) by the three-term recurrence."""
    p, q = np.ones_like(x), 0.5 * a * y + (1.0 + 0.5 * a) * x
    if n == 0:
        return p
    for m in range(2, n + 1):
        c = 2.0 * m + a
        p, q = q, ((c - 1.0) * (a * a * y + c * (c - 2.0) * x) * q - 2.0 * (m + a - 1.0) * (m - 1.0) * c * y * y * p) / (
            2.0 * m * (m + a) * (c - 2.0))
    return q


def _dubiner(D, N, P):
    """The orthogonal polynomials of the reference simplex at the points P (m, D)."""
    one, out = np.ones_like(P[:, 0]), []
    for i in _exponents(D, N):
        v, rest, a = one, one, 0
        tail = [sum((P[:, k] for k in range(d, D)), 0 * one) for d in range(D + 1)]  # x_d + ... + x_(D-1)
        for d in range(D):
            v = v * _jacobi(i[d], a, P[:, d] - (one - tail[d]), one - tail[d + 1])
            a += 2 * i[d] + 1
        out.append(v)
    return np.stack(out, 1)


def _warp(N, r):
    eq = np.linspace(-1.0, 1.0, N + 1)
    inner = np.polynomial.legendre.Legendre.basis(N).deriv().roots() if N > 1 else []
    gl = np.concatenate([[-1.0], np.sort(np.real(inner)), [1.0]])
    w = np.zeros_like(r)
    for i in range(N + 1):
        w += (gl[i] - eq[i]) * np.prod([(r - eq[m]) / (eq[i] - eq[m]) for m in range(N + 1) if m != i], axis=0)
    inside = np.abs(r) < 1.0 - 1e-14
    return np.where(inside, w / np.where(inside, 1.0 - r * r, 1.0), w)


def _warp_triangle(N, alpha, L, V):
    """In-plane displacement of the nodes with barycentric coordinates L on the triangle V."""
    out = np.zeros((L.shape[0], V.shape[1]))
    for a, b, m in ((0, 1, 2), (0, 2, 1), (1, 2, 0)):
        t = (V[b] - V[a]) / np.linalg.norm(V[b] - V[a])
        blend = 4.0 * L[:, a] * L[:, b] * (1.0 + (alpha * L[:, m]) ** 2)
        out += (_warp(N, L[:, b] - L[:, a]) * blend)[:, None] * t
    return out


def _nodes(D, N):
    """Warp-and-blend nodes (T. Warburton, An explicit construction of interpolation nodes on the simplex,
    J. Eng. Math. 56, 2006) of the reference simplex."""
    L = np.array(_exponents(D, N)) / N
    L = np.concatenate([1.0 - L.sum(1, keepdims=True), L], 1)
    r3, r6 = math.sqrt(3.0), math.sqrt(6.0)
    if D == 2:
        V = np.array([[-1.0, -1.0 / r3], [1.0, -1.0 / r3], [0.0, 2.0 / r3]])
        X = L @ V + _warp_triangle(N, (0.0, 0.0, 1.4152, 0.1001, 0.2751, 0.9800)[N - 1], L, V)
    else:
        V = np.array([[-1.0, -1.0 / r3, -1.0 / r6], [1.0, -1.0 / r3, -1.0 / r6], [0.0, 2.0 / r3, -1.0 / r6],
                      [0.0, 0.0, 3.0 / r6]])
        alpha, move = (0.0, 0.0, 0.0, 0.1002)[N - 1], np.zeros((len(L), 3))
        for f in ((0, 1, 2, 3), (0, 1, 3, 2), (0, 2, 3, 1), (1, 2, 3, 0)):
            warp, lm = _warp_triangle(N, alpha, L[:, f[:3]], V[list(f[:3])]), L[:, f[3]]
            num = np.prod(L[:, f[:3]], axis=1)
            den = np.prod(L[:, f[:3]] + 0.5 * lm[:, None], axis=1)
            flat = np.abs(den) < 1e-14  # on an edge of the face the edge's own displacement stays
            s = np.where(flat, 1.0, (1.0 + (alpha * lm) ** 2) * num / np.where(flat, 1.0, den))
            move = np.where(flat[:, None], 0.0, move) + s[:, None] * warp
        X = L @ V + move
    return np.linalg.solve((V[1:] - V[0]).T, (X - V[0]).T).T


def _rule(D, order):
    """Quadrature of the reference simplex: the tabulated rules, or Gauss points where those are fewer."""
    if D == 1:
        x, w = np.polynomial.legendre.leggauss(1 + order // 2)
        return (0.5 * x + 0.5)[:, None], 0.5 * w
    if order == 3 and D == 2:  # 2 x 2 Gauss points in collapsed coordinates
        s = np.sqrt(6.0)
        x1, w1 = np.array([(4.0 + s) / 10.0, (4.0 - s) / 10.0]), np.array([(9.0 - s) / 36.0, (9.0 + s) / 36.0])
        x0, w0 = np.polynomial.legendre.leggauss(2)
        x0 = (0.5 * x0 + 0.5)[::-1]
        return (np.array([[a, b * (1.0 - a)] for a in x1 for b in x0]), np.array([a * b for a in w1 for b in 0.5 * w0]))
    best = None
    with open(RULES) as f:
        for line in f:
            if line.startswith("rule"):
                _, fam, d, o, n = line.split()
                rows = [[float(v) for v in next(f).split()] for _ in range(int(n))]
                if int(d) == D and int(o) >= order and (best is None or (int(n), fam) < best[0]):
                    best = ((int(n), fam), np.array(rows))
    (_, fam), r = best
    return (r[:, :D], r[:, D] / 6.0) if fam == "JS" else (0.5 * r[:, :D] + 0.5, r[:, D] / 2 ** D)


class _Form:
    """The interior-penalty form of a case on its mesh in FP64."""

    def __init__(self, case, fields, dev):
        D, N = case["dim"], case["degree"]
        self.D, self.el, self.Q = D, case["kind"] == "elasticity", D if case["kind"] == "elasticity" else 1
        t = lambda a: torch.tensor(np.ascontiguousarray(a), dtype=torch.float64, device=dev)
        ref = _nodes(D, N)
        inv = np.linalg.inv(_dubiner(D, N, ref))

        def tables(P):  # nodal values and gradients, then those of the solution's basis
            g = np.stack([_dubiner(D, N, P + 1e-30j * np.eye(D)[d]).imag / 1e-30 for d in range(D)], 1)
            v = _dubiner(D, N, P)
            nodal = t(v @ inv), t(g @ inv)
            return nodal + (nodal if self.el else (t(v), t(g)))

        order = 2 * N + 1
        (P, W), (Pf, wf) = _rule(D, order), _rule(D - 1, order)
        v, el, bnd, bc = _mesh(case)
        self.E, self.Nbf = len(el), len(ref)
        cor = np.concatenate([np.zeros((1, D)), np.eye(D)])
        X = _warped(t(np.einsum("pv,evi->epi", np.concatenate([1.0 - ref.sum(1, keepdims=True), ref], 1), v[el])))
        self.W, self.wf = t(W), t(wf)
        self.M, Mg, self.B, self.G = tables(P)
        self.x = torch.einsum("qk,eki->eqi", self.M, X)
        self.Ji, det = self.inverse(torch.einsum("qdk,eki->eqid", Mg, X))
        self.detW = det.abs()
        vol = (self.detW * self.W).sum(1)
        # faces: f leaves out vertex D - f; the points run over the other vertices in ascending order, so
        # those of two elements that share a face coincide
        self.fM, self.fB, self.fG, fx, fJi, fn = [], [], [], [], [], []
        for f in range(D + 1):
            keep = [k for k in range(D + 1) if k != D - f]
            pts = np.concatenate([1.0 - Pf.sum(1, keepdims=True), Pf], 1) @ cor[keep]
            m, g, b, bg = tables(pts)
            Ji, det = self.inverse(torch.einsum("qdk,eki->eqid", g, X))
            grad = np.concatenate([-np.ones((1, D)), np.eye(D)])[D - f]
            self.fM.append(m), self.fB.append(b), self.fG.append(bg)
            fx.append(torch.einsum("qk,eki->eqi", m, X)), fJi.append(Ji)
            fn.append(-det.abs()[..., None] * torch.einsum("d,eqdi->eqi", t(grad), Ji))
        self.fx, self.fJi, self.n = (torch.stack(a, 1) for a in (fx, fJi, fn))
        self.nl = self.n.norm(dim=-1)
        faces, key = _faces(el, len(v))
        o = np.argsort(key, kind="stable")
        nb = np.full(len(key), -1)
        pair = np.nonzero(key[o][1:] == key[o][:-1])[0]
        nb[o[pair]], nb[o[pair + 1]] = o[pair + 1], o[pair]
        bk = np.zeros(len(bnd), dtype=np.int64)
        for d in range(D):
            bk = bk * len(v) + bnd[:, d]
        natural = np.isin(key, bk[bc == T.BC_NATURAL])
        self.nb = torch.tensor(np.maximum(nb, 0), device=dev)
        self.two = torch.tensor(nb >= 0, device=dev).view(self.E, D + 1, 1, 1)
        self.on = torch.tensor(~natural, dtype=torch.float64, device=dev).view(self.E, D + 1, 1, 1)
        self.area = ((self.nl * self.wf).sum(-1) / vol[:, None]) * (D + 1) * N * (N - 1 + D) / D
        self.set([f(self.x) for f in (fields if self.el else fields[:1])])

    @staticmethod
    def inverse(J):
        """Inverse and determinant of J[..., i, d]; the inverse is indexed [..., d, i]."""
        if J.shape[-1] == 2:
            det = J[..., 0, 0] * J[..., 1, 1] - J[..., 0, 1] * J[..., 1, 0]
            A = torch.stack([J[..., 1, 1], -J[..., 0, 1], -J[..., 1, 0], J[..., 0, 0]], -1).view(J.shape)
        else:
            c = [torch.linalg.cross(J[..., (d + 1) % 3], J[..., (d + 2) % 3]) for d in range(3)]
            A, det = torch.stack(c, -2), (J[..., 0] * c[0]).sum(-1)
        return A / det[..., None, None], det

    def set(self, coef):
        """Coefficients at the volume points -> their L2 projection, traces and the penalty."""
        wj, D = self.W * self.detW, self.D
        mass = torch.einsum("qk,eq,ql->ekl", self.M, wj, self.M)
        rhs = torch.einsum("qk,eq,ceq->ekc", self.M, wj, torch.stack(coef))
        nodal = torch.linalg.solve(mass, rhs)
        self.c = [torch.einsum("qk,ek->eq", self.M, nodal[..., i]) for i in range(len(coef))]
        self.fc = [torch.stack([m @ nodal[..., i].T for m in self.fM], 0).permute(2, 0, 1) for i in range(len(coef))]
        lo = nodal[..., 0] if not self.el else 2.0 * nodal[..., 1]
        hi = nodal[..., 0] if not self.el else D * nodal[..., 0] + 2.0 * nodal[..., 1]
        p = self.area * (hi.amax(1) ** 2 / lo.amin(1))[:, None]
        self.pen = torch.where(self.two[..., 0, 0], 0.25 * (p + p.reshape(-1)[self.nb].view(p.shape)), p)

    def stress(self, c, g):  # g[..., r, i] = d u_r / d x_i
        if not self.el:
            return c[0][..., None, None] * g
        tr = torch.diagonal(g, dim1=-2, dim2=-1).sum(-1)
        return c[1][..., None, None] * (g + g.transpose(-1, -2)) + (c[0] * tr)[..., None, None] * torch.eye(
            self.D, dtype=g.dtype, device=g.device)

    def apply(self, x, data=None, own=False):
        """A x (minus the right-hand side of Dirichlet data at the facet points); own: only the blocks of
        the elements themselves."""
        U = x.view(self.E, self.Q, self.Nbf)
        g = torch.einsum("qdk,erk,eqdi->eqri", self.G, U, self.Ji)
        s = self.stress(self.c, g) * (self.W * self.detW)[..., None, None]
        y = torch.einsum("qdk,eqdi,eqri->erk", self.G, self.Ji, s)
        u = torch.stack([torch.einsum("qk,erk->eqr", b, U) for b in self.fB], 1)
        g = torch.stack([torch.einsum("qdk,erk->eqrd", b, U) for b in self.fG], 1)
        sn = (self.stress(self.fc, g @ self.fJi) * self.n[..., None, :]).sum(-1)
        zero = torch.zeros_like(u)
        un, sm = (zero, zero) if own else (a.reshape(-1, *a.shape[2:])[self.nb].view(a.shape) for a in (u, sn))
        given = zero if data is None else data(self.fx)[..., :self.Q]
        d = torch.where(self.two, 0.5 * (un - u), given - u)
        tau = torch.where(self.two, 0.5 * (sn - sm) - (self.pen[..., None] * self.nl)[..., None] * (u - un),
                          sn - (self.pen[..., None] * self.nl)[..., None] * (u - given))
        tau, d = (tau * self.on * self.wf[:, None], d * self.on * self.wf[:, None])
        lift = self.stress(self.fc, d[..., :, None] * self.n[..., None, :]) @ self.fJi.transpose(-1, -2)
        for f in range(self.D + 1):
            y = y - torch.einsum("qk,eqr->erk", self.fB[f], tau[:, f]) + torch.einsum("qdk,eqrd->erk", self.fG[f], lift[:, f])
        return y.reshape(-1)

    def blocks(self):
        """Diagonal block of every element, [element, row, column]."""
        bs, out = self.Q * self.Nbf, []
        for j in range(bs):
            e = torch.zeros((self.E, bs), dtype=torch.float64, device=self.W.device)
            e[:, j] = 1.0
            out.append(self.apply(e.view(-1), own=True).view(self.E, bs))
        return torch.stack(out, -1)

    def solve(self, b):
        """Block-Jacobi CG to the FP64 floor."""
        D = torch.linalg.inv(self.blocks())
        pre = lambda r: (D @ r.view(self.E, -1, 1)).reshape(-1)
        x, r = torch.zeros_like(b), b.clone()
        z = pre(r)
        p, rz = z.clone(), r @ z
        for i in range(4000):
            q = self.apply(p)
            a = rz / (p @ q)
            x, r = x + a * p, r - a * q
            z = pre(r)
            rz, old = r @ z, rz
            p = z + (rz / old) * p
            if i % 50 == 49 and float(r.norm()) < 2e-14 * float(b.norm()):
                break
        return x


def exact(case, seed):
    E, _, nbf, _, _, _ = _sizes(case)
    what, bs = case["what"], nbf * (case["dim"] if case["kind"] == "elasticity" else 1)
    # probing or inverting every block, or a CG on a larger mesh, would take too long
    if (what == "jacobi" and E * bs * bs > 1.5e8) or (what == "solve" and E * bs > 4e5):
        return None
    dev = torch.device("cuda")
    fields, X, data = _inputs(case, seed, dev)
    A, X = _Form(case, fields, dev), X.double()
    if what in ("apply", "assembled"):
        return A.apply(X[0]) if len(X) == 1 else torch.stack([A.apply(x) for x in X])
    if what == "jacobi":
        return torch.linalg.solve(A.blocks(), X[0].view(A.E, -1, 1)).reshape(-1)
    if what == "gradient":
        c = [f(A.x).requires_grad_() for f in fields]
        A.set(c)
        return list(torch.autograd.grad(X[1] @ A.apply(X[0]), c))
    if what == "wave":
        y = A.apply(X[0], data).view(A.E, A.Q, A.Nbf)
        Mi = torch.linalg.inv(A.B.T @ (A.W[:, None] * A.B)) @ A.B.T
        return -torch.einsum("kq,eq,lq,erl->erk", Mi, A.W / A.detW, Mi, y).reshape(-1)
    return A.solve(X[0])

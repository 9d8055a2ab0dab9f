"""Kernel branches at the sizes where they can go wrong, on meshes with permuted vertex ids (every pair
of local faces meets) against the CPU FP64 oracle.  Bars as in test_gpu_apply.py: relative L2 1e-12 in
FP64 (observed 1e-14), 1e-5 in FP32 (observed 2e-7)."""
import numpy as np
import pytest

import oracle_lib as O
import tandem_amd as T
from cases import BC_D, BC_N, rel_l2, smooth_coefficients, warp_nodes

pytestmark = pytest.mark.gpu


class Mixed:
    """A warped box of n cells with permuted vertex ids, a natural side and Dirichlet elsewhere."""

    def __init__(self, D, n, N, kind=0, seed=0):
        b = T.Mesh.box(D, n, 1 if D == 3 else 0, [BC_D] * (2 * D - 1) + [BC_N])
        p = np.random.default_rng(seed).permutation(len(b.vertices))
        v = np.empty_like(b.vertices)
        v[p] = b.vertices
        self.mesh = T.Mesh(v, p[b.elements], p[b.boundary_facets], b.boundary_bc)
        m = self.mesh
        self.nodes = np.ascontiguousarray(warp_nodes(m.affine_nodes(N)))
        self.op = T.DGOperator(m, kind, N, self.nodes)
        c0, c1 = smooth_coefficients(self.op.volume_points(), seed)
        self.c = (c0, c1 if kind == 0 else None)
        self.op.set_material(*self.c)
        om = O.Mesh.from_arrays(m.vertices, m.elements, m.boundary_facets, m.boundary_bc)
        self.oracle = O.Operator(kind, om, N, *self.c, nodes=self.nodes)
        self.n = self.op.n


@pytest.mark.parametrize("variant", ["auto", "mfma-element"])
@pytest.mark.parametrize("D,n,N", [(3, (1, 1, 1), 4), (3, (3, 1, 1), 4), (3, (3, 2, 1), 3), (3, (2, 2, 1), 2),
                                   (2, (3, 3), 6), (2, (5, 3), 4), (2, (4, 3), 3), (2, (4, 2), 2)])
def test_face_frame_traces(cuda, D, n, N, variant):
    """The face frame numbers the face's own nodes first and the facet kernel contracts values and
    tangential derivatives over those alone: every degree, both sides of its rule, partial groups."""
    import torch

    c = Mixed(D, n, N, seed=N)
    c.op.set_variant(variant)
    x = np.random.default_rng(2).uniform(-1.0, 1.0, c.n)
    ref = c.oracle.apply(x)
    for dt, bar in ((torch.float64, 1e-12), (torch.float32, 1e-5)):
        xd = torch.from_numpy(x).to(cuda).to(dt)
        y = torch.full_like(xd, float("nan"))
        c.op.apply(xd, y)
        assert rel_l2(y.double().cpu().numpy(), ref) <= bar


@pytest.mark.parametrize("D,n,N", [(3, (3, 1, 1), 1), (3, (1, 1, 1), 3), (2, (3, 3), 1), (2, (3, 5), 2), (2, (4, 2), 4),
                                   (2, (9, 1), 5), (3, (1, 1, 1), 5), (3, (1, 1, 1), 4), (3, (5, 5, 4), 4)])
def test_wave_rhs_degrees(cuda, D, n, N):
    """The matrix-core inverse mass at the other degrees and partial groups (3D P5 keeps the kernel with
    run-time sizes and has no apply; 3D P4 takes it up to 512 elements), in place too; the facet part added to the elements with data."""
    import torch

    c = Mixed(D, n, N, seed=N)
    rng = np.random.default_rng(4)
    x, g = rng.uniform(-1.0, 1.0, c.n), rng.uniform(-1.0, 1.0, (c.op.F, D, c.op.nq))
    xd, gd = torch.from_numpy(x).to(cuda), torch.from_numpy(g.ravel()).to(cuda)
    assert rel_l2(c.op.inverse_mass(xd).cpu().numpy(), c.oracle.inverse_mass(x)) <= 1e-12
    z = xd.clone()
    assert rel_l2(c.op.inverse_mass(z, z).cpu().numpy(), c.oracle.inverse_mass(x)) <= 1e-12
    if D == 3 and N > 4:
        return
    assert rel_l2(c.op.wave_rhs(xd, gd).cpu().numpy(), c.oracle.wave_rhs(x, g)) <= 1e-12
    b = torch.empty_like(xd)
    assert rel_l2(c.op.rhs_device(b, None, gd).cpu().numpy(), c.oracle.rhs(None, g)) <= 1e-12


@pytest.mark.parametrize("D,n,N", [(3, (1, 1, 1), 4), (3, (3, 2, 1), 4), (3, (3, 2, 1), 3), (3, (2, 2, 1), 2),
                                   (2, (3, 3), 6), (2, (5, 3), 4), (2, (3, 3), 3)])
def test_small_apply_and_explicit_shapes(cuda, D, n, N):
    """The launches of small applies (default here) and every explicitly chosen launch shape and workgroup
    order on the same mesh."""
    import torch

    c = Mixed(D, n, N, seed=N + 1)
    x = np.random.default_rng(3).uniform(-1.0, 1.0, c.n)
    ref = c.oracle.apply(x)
    for prec, dt, bar in (("fp64", torch.float64, 1e-12), ("fp32", torch.float32, 1e-5)):
        xd = torch.from_numpy(x).to(cuda).to(dt)
        for config in [None] + [(s, o) for s in range(4) for o in range(3)]:
            if config:
                c.op.set_shape(prec, *config)
            y = torch.full_like(xd, float("nan"))
            c.op.apply(xd, y)
            assert rel_l2(y.double().cpu().numpy(), ref) <= bar, config


@pytest.mark.parametrize("D,n,N,cols", [(3, (4, 4, 4), 4, 43), (2, (16, 16), 6, 33), (3, (8, 7, 7), 2, 7)])
def test_small_apply_limits(cuda, D, n, N, cols):
    """Groups x columns on both sides of the rules (384 facet groups, 1024 element groups) and of the
    one-group-a-workgroup limit (256), batched and singly; a short CG runs the fused dot on the small
    launches."""
    import torch

    c = Mixed(D, n, N, seed=5)
    X = np.random.default_rng(6).uniform(-1.0, 1.0, (cols, c.n))
    ref = np.stack([c.oracle.apply(x, nthreads=4) for x in X])
    for dt, bar in ((torch.float64, 1e-12), (torch.float32, 1e-5)):
        for k in sorted({1, 2, 3, 4, 7, min(cols, 11), cols - 1, cols}):
            Xd = torch.from_numpy(X[:k]).to(cuda).to(dt)
            Y = torch.full_like(Xd, float("nan"))
            c.op.apply_batched(Xd, Y)
            assert rel_l2(Y.double().cpu().numpy(), ref[:k]) <= bar, k
    b = torch.from_numpy(ref[0]).to(cuda)
    x = torch.zeros_like(b)
    res = c.op.solve(b, x, rtol=1e-8, mode="fp64", precond="block-jacobi", max_iter=5000)
    assert res["converged"] and rel_l2(c.oracle.apply(x.cpu().numpy()), ref[0]) <= 1e-7


@pytest.mark.parametrize("mode", ["fp64", "fp32-ru"])
@pytest.mark.parametrize("D,n,N", [(3, (1, 1, 1), 4), (3, (11, 9, 9), 3), (2, (47, 47), 4), (2, (91, 90), 6)])
def test_fused_dot_of_the_small_launches(cuda, D, n, N, mode):
    """The solvers' p.Ap from the element kernel's partial sums on the small launches, both precisions: one
    group of elements a workgroup, two (257 to 1024 groups), and near the upper end of the rule.  A wrong sum
    gives CG wrong steps; the residual is taken in FP64 by the oracle."""
    import torch

    c = Mixed(D, n, N, seed=7)
    groups = (c.op.E + 15) // 16
    assert groups == 1 or 257 <= groups <= 1024
    b = c.oracle.apply(np.random.default_rng(15).uniform(-1.0, 1.0, c.n), nthreads=8)
    bd = torch.from_numpy(b).to(cuda)
    x = torch.zeros_like(bd)
    res = c.op.solve(bd, x, rtol=1e-8, mode=mode, precond="block-jacobi", max_iter=20000)  # some 2,700 steps
    assert res["converged"]
    r = b - c.oracle.apply(x.cpu().numpy(), nthreads=8)
    assert np.linalg.norm(r) <= 1e-7 * np.linalg.norm(b)


@pytest.mark.parametrize("D,n,N", [(2, (101, 101), 2), (2, (79, 77), 3), (2, (65, 63), 4), (2, (55, 53), 5),
                                   (2, (47, 47), 6), (3, (15, 13, 14), 1), (3, (11, 10, 10), 2), (3, (9, 9, 7), 3),
                                   (3, (7, 7, 7), 4)])
def test_poisson_matrix_core_apply(cuda, D, n, N):
    """Every compiled degree of the matrix-core Poisson apply (both kernels, natural and Dirichlet faces,
    a partial last group) just above its size rule, singly, batched at a larger stride, without
    allocation; "points" agrees."""
    import ctypes as C

    import torch
    from tandem_amd._lib import lib

    c = Mixed(D, n, N, kind=1, seed=N)
    assert c.op.E % 16 != 0
    X = np.random.default_rng(8).uniform(-1.0, 1.0, (3, c.n))
    ref = np.stack([c.oracle.apply(x, nthreads=4) for x in X])
    for dt, bar in ((torch.float64, 1e-12), (torch.float32, 1e-5)):
        Xd = torch.zeros((3, c.n + 6), dtype=dt, device=cuda)
        Xd[:, :c.n] = torch.from_numpy(X).to(cuda).to(dt)
        Y = torch.full_like(Xd, float("nan"))
        c.op.apply_batched(Xd, Y)
        assert rel_l2(Y[:, :c.n].double().cpu().numpy(), ref) <= bar
        y = torch.full((c.n,), float("nan"), dtype=dt, device=cuda)
        c.op.apply(Xd[1, :c.n].contiguous(), y)
        assert torch.equal(y, Y[1, :c.n])
        if dt == torch.float64:
            z = torch.full_like(y, float("nan"))
            assert lib().tdg_mult_noalloc(c.op._h, C.c_void_p(Xd[1].contiguous().data_ptr()), C.c_void_p(z.data_ptr())) == 0
            assert torch.equal(z, y)
        c.op.set_variant("points")
        c.op.apply(Xd[1, :c.n].contiguous(), y)
        assert rel_l2(y.double().cpu().numpy(), ref[1]) <= bar
        assert not torch.equal(y, Y[1, :c.n])  # the other kernel: its sums run in another order
        c.op.set_variant("auto")


@pytest.mark.parametrize("fp32", [1, 0])
@pytest.mark.parametrize("D,n,degrees", [(3, (4, 3, 5), (2, 1)), (2, (15, 13), (2, 1)), (2, (15, 13), (3, 2))])
def test_multigrid_few_columns(cuda, D, n, degrees, fp32):
    """The coarse solver's kernels for at most two columns (assembled rows of 6 and 12, fused smoothing
    steps, a wave per block row) and, with three columns, those for many: the same solutions to 1e-10."""
    import torch

    cs = [Mixed(D, n, N, seed=9) for N in degrees]
    fine, ops = cs[0], [c.op for c in cs]
    assert ops[-1].n > 800 and ops[-1].E % 32 != 0
    B = np.random.default_rng(12).uniform(-1.0, 1.0, (3, fine.n))
    Bd = torch.zeros((3, fine.n + 4), dtype=torch.float64, device=cuda)
    Bd[:, :fine.n] = torch.from_numpy(B).to(cuda)
    mg = T.PMultigrid(ops, galerkin_penalty=0, vcycle_fp32=fp32, coarse_fp32=fp32)
    for k in (1, 2, 3):
        X = torch.zeros((k, fine.n + 4), dtype=torch.float64, device=cuda)
        res = mg.solve_multi(Bd[:k].contiguous(), X, rtol=1e-10)
        assert res["converged"]
        for c in range(k):
            r = B[c] - fine.oracle.apply(X[c, :fine.n].cpu().numpy())
            assert np.linalg.norm(r) <= 1e-9 * np.linalg.norm(B[c])
    op = ops[-1]  # assembled by the set-up: two columns at a stride equal single applies
    for dt in (torch.float64, torch.float32):
        X = torch.rand((2, op.n + 3), dtype=dt, device=cuda)
        Y = torch.full_like(X, 7.0)
        op.apply_batched(X, Y)
        for c in range(2):
            y = torch.zeros(op.n, dtype=dt, device=cuda)
            op.apply(X[c, :op.n].contiguous(), y)
            assert torch.equal(y, Y[c, :op.n])
        assert torch.all(Y[:, op.n:] == 7.0)


def test_poisson_column_ranges(cuda):
    """More columns than one range of the Poisson trace buffer (1 GiB) holds: every column as singly."""
    import torch

    c = Mixed(3, (7, 7, 7), 4, kind=1, seed=2)
    one = c.op.E * 4 * c.op.nq * 2 * 8
    cols = (1 << 30) // one + 3
    X = torch.rand((cols, c.n), dtype=torch.float64, device=cuda)
    Y = torch.full_like(X, float("nan"))
    c.op.apply_batched(X, Y)
    for k in (0, cols - 4, cols - 3, cols - 1):
        y = torch.empty(c.n, dtype=torch.float64, device=cuda)
        c.op.apply(X[k].contiguous(), y)
        assert torch.equal(y, Y[k])


@pytest.mark.parametrize("kind,D,n,N", [(1, 2, (65, 63), 4), (1, 3, (11, 10, 10), 2), (0, 3, (4, 3, 3), 3)])
def test_captured_and_on_two_streams(cuda, kind, D, n, N):
    """The matrix-core Poisson apply and the two-kernel apply captured into a graph and replayed after a larger
    batch, with eager applies between, and applies of two vectors queued on two streams in turn: the eager
    results' bits."""
    import torch

    c = Mixed(D, n, N, kind=kind, seed=3)
    c.op.upload()
    X = torch.rand((5, c.n), dtype=torch.float64, device=cuda)
    ref = torch.empty_like(X)
    for k in range(5):
        c.op.apply(X[k], ref[k])
    x, y, Y = X[0].clone(), torch.zeros_like(X[0]), torch.empty_like(X)
    s, graph = torch.cuda.Stream(), torch.cuda.CUDAGraph()
    torch.cuda.synchronize()
    with torch.cuda.graph(graph, stream=s):
        c.op.set_stream(s)
        c.op.apply(x, y)
    c.op.set_stream(None)
    c.op.apply_batched(X, Y)
    assert torch.equal(Y, ref)
    for k in (1, 4, 2):
        x.copy_(X[k])
        y.fill_(float("nan"))
        graph.replay()
        torch.cuda.synchronize()
        c.op.apply(X[k - 1], Y[0])
        torch.cuda.synchronize()
        assert torch.equal(y, ref[k]) and torch.equal(Y[0], ref[k - 1])
    Y.fill_(float("nan"))
    torch.cuda.synchronize()
    streams = [torch.cuda.Stream(), torch.cuda.Stream()]
    for i in range(40):
        c.op.set_stream(streams[i % 2])
        c.op.apply(X[i % 5], Y[i % 5])
    c.op.set_stream(None)
    torch.cuda.synchronize()
    assert torch.equal(Y, ref)


def test_multigrid_coarse_operator_changed_after_setup(cuda):
    """A coarse operator that a caller has given another variant, and a new material besides (its block rows
    are dropped), still serves one and two columns: the set-up's AMG levels precondition what it now applies."""
    import torch

    cs = [Mixed(3, (4, 3, 5), N, seed=9) for N in (2, 1)]
    fine, coarse = cs
    B = torch.from_numpy(np.random.default_rng(13).uniform(-1.0, 1.0, (2, fine.n))).to(cuda)
    mg = T.PMultigrid([c.op for c in cs], galerkin_penalty=0)
    assert mg.solve_multi(B, torch.zeros_like(B), rtol=1e-10)["converged"]
    for change in (lambda: coarse.op.set_variant("auto"), lambda: coarse.op.set_material(*coarse.c),
                   lambda: coarse.op.set_variant("assembled")):
        change()
        for k in (1, 2):
            X = torch.zeros_like(B)
            assert mg.solve_multi(B[:k].contiguous(), X[:k], rtol=1e-10)["converged"]
            for c in range(k):
                r = B[c].cpu().numpy() - fine.oracle.apply(X[c].cpu().numpy())
                assert np.linalg.norm(r) <= 1e-9 * float(torch.linalg.norm(B[c]))

"""The solver kernels at the sizes where they can go wrong: every block size of
the element inverses, restart lengths around the groups of basis vectors that a
CGS2 pass takes, instances around the reduction chunks of the packed solver,
ILU(0) sweeps over element numberings with few and many levels."""
import numpy as np
import pytest

from pdes_amd import abi, euler, linsolve, problems
from pdes_amd.batch import BatchSolver

pytestmark = pytest.mark.gpu

SHAPES = [("vortex", 1, "omega", "roe"), ("vortex", 2, "omega", "roe"), ("vortex", 3, "omega", "roe"),
          ("vortex", 4, "omega", "roe"), ("vortex", 1, "diage", "ir"), ("vortex", 2, "diage", "ir"),
          ("vortex", 3, "diage", "ir"), ("vortex", 4, "diage", "ir"), ("cube", 1, "omega", "roe"),
          ("cube", 2, "omega", "roe")]


def _problem(kind, n, p, opk, flux, shuffle=False):
    m, op, ph = problems.make_problem(kind, n, p, opk, flux, Ma=0.5, aoa_deg=2.0)
    if shuffle:
        perm = np.random.default_rng(5).permutation(m.numEl)
        place = np.argsort(perm).astype(m.interfaces.dtype)
        for a in ("coords", "dxidx", "jac", "vert_coords"):
            setattr(m, a, np.ascontiguousarray(getattr(m, a)[perm]))
        m.interfaces[:, :2] = place[m.interfaces[:, :2]]
        m.bndryfaces[:, 0] = place[m.bndryfaces[:, 0]]
    q = problems.vortex_noise_state(m, ph, seed=5) if kind == "vortex" else problems.freestream_bump_state(m, ph)
    return m, op, ph, q


@pytest.mark.parametrize("shuffle", [False, True])
@pytest.mark.parametrize("kind,p,opk,flux", SHAPES)
def test_ilu0_sweeps_agree(monkeypatch, kind, p, opk, flux, shuffle):
    """Dependency-driven sweeps, level sweeps and the unforced choice give the
    same bits, for one element layer, for sets shorter and longer than the
    largest (68 to 384 elements), numbered naturally and at random."""
    for n in (1, 5, 45) if kind == "vortex" else (1, 6):
        print(f"case {kind} n={n} p={p} {opk} {flux} shuffle={shuffle}", flush=True)
        m, op, ph, q = _problem(kind, n, p, opk, flux, shuffle)
        b = np.random.default_rng(13).standard_normal(q.shape)
        out = []
        for env in ("PDES_ILU_DEP", "PDES_ILU_LEVELS", None):
            for v in ("PDES_ILU_DEP", "PDES_ILU_LEVELS"):
                monkeypatch.delenv(v, raising=False)
            if env:
                monkeypatch.setenv(env, "1")
            e = euler.EulerData(m, op, ph)
            e.set_q(q)
            linsolve.evalJacobian(m, op, e)
            pc = linsolve.HIPILU0PC(e)
            pc.calcPC()
            x = np.zeros_like(b)
            for _ in range(2):
                pc.applyPC(m, op, e, None, 0.0, b, x)
            out.append(x)
            e.free()
        assert np.all(np.isfinite(out[0]))
        assert np.array_equal(out[0], out[1]) and np.array_equal(out[0], out[2])


@pytest.mark.parametrize("kind,p,opk,flux", SHAPES)
def test_ilu0_sweeps_agree_fp64_blocks(monkeypatch, kind, p, opk, flux):
    """The same with FP64 blocks: the same bits from both kinds of sweep over
    sets of one element, of a few and longer than the largest."""
    for n in (1, 5, 45) if kind == "vortex" else (1, 6):
        print(f"case {kind} n={n} p={p} {opk} {flux}", flush=True)
        m, op, ph, q = _problem(kind, n, p, opk, flux)
        b = np.random.default_rng(13).standard_normal(q.shape)
        out = []
        for env in ("PDES_ILU_DEP", "PDES_ILU_LEVELS"):
            monkeypatch.delenv("PDES_ILU_DEP", raising=False)
            monkeypatch.setenv(env, "1")
            e = euler.EulerData(m, op, ph)
            e.set_q(q)
            linsolve.evalJacobian(m, op, e, fp64_blocks=True)
            pc = linsolve.HIPILU0PC(e)
            pc.calcPC()
            x = np.zeros_like(b)
            for _ in range(2):
                pc.applyPC(m, op, e, None, 0.0, b, x)
            out.append(x)
            e.free()
        monkeypatch.delenv("PDES_ILU_LEVELS")
        assert np.all(np.isfinite(out[0]))
        assert np.array_equal(out[0], out[1])


@pytest.mark.parametrize("kind,p,opk,flux", SHAPES)
def test_block_inverses(kind, p, opk, flux):
    """The block-Jacobi apply solves with each element's block to what an FP32
    inverse of N unknowns allows: 8 N eps cond."""
    print(f"case {kind} p={p} {opk} {flux}", flush=True)
    m, op, ph, q = _problem(kind, 1 if kind == "cube" else 2, p, opk, flux)
    e = euler.EulerData(m, op, ph)
    e.set_q(q)
    linsolve.evalJacobian(m, op, e)
    rowptr, colind = linsolve.getSparsityPattern(e)
    vals = linsolve.getJacobianValues(e).astype(np.float64)
    pc = linsolve.HIPBJacobiPC(e)
    pc.calcPC()
    b = np.random.default_rng(3).standard_normal(q.shape)
    x = np.zeros_like(b)
    pc.applyPC(m, op, e, None, 0.0, b, x)
    Np, nd = q.shape[1:]
    N = Np * nd
    for el in range(m.numEl):
        D = np.zeros((Np, nd, Np, nd))
        for i in range(Np):
            for t in range(rowptr[el * Np + i], rowptr[el * Np + i + 1]):
                if colind[t] // Np == el:
                    D[i, :, colind[t] % Np, :] += vals[t]
        D = D.reshape(N, N)
        xe = np.linalg.solve(D, b[el].ravel())
        err = np.linalg.norm(x[el].ravel() - xe) / np.linalg.norm(xe)
        assert err <= 8 * N * 2.0 ** -24 * np.linalg.cond(D), (el, err)
    e.free()


@pytest.mark.parametrize("fp64", [False, True])
@pytest.mark.parametrize("kind,p,opk,flux", SHAPES)
def test_block_row_products(kind, p, opk, flux, fp64):
    """J x over rows of 3 to 60 blocks, some a multiple of the blocks in flight
    and some not, is numpy's sum of the same products to n rounding errors."""
    print(f"case {kind} p={p} {opk} {flux} fp64={fp64}", flush=True)
    m, op, ph, q = _problem(kind, 1 if kind == "cube" else 2, p, opk, flux, shuffle=True)
    e = euler.EulerData(m, op, ph)
    e.set_q(q)
    lo = linsolve.HIPBSRLO(e, fp64_blocks=fp64)
    lo.calcLinearOperator()
    rowptr, colind = linsolve.getSparsityPattern(e, fp64_blocks=fp64)
    vals = linsolve.getJacobianValues(e, fp64_blocks=fp64).astype(np.float64)
    x = np.random.default_rng(6).standard_normal(q.shape)
    y = np.zeros_like(x)
    lo.applyLinearOperator(m, op, e, None, None, 0.0, x, y)
    nd = q.shape[2]
    xb, yb = x.reshape(-1, nd), y.reshape(-1, nd)
    for r in range(len(rowptr) - 1):
        blk, xc = vals[rowptr[r]:rowptr[r + 1]], xb[colind[rowptr[r]:rowptr[r + 1]]]
        ref, mag = np.einsum("bij,bj->i", blk, xc), np.einsum("bij,bj->i", np.abs(blk), np.abs(xc))
        assert np.all(np.abs(yb[r] - ref) <= 2 * nd * len(blk) * 2.0 ** -53 * mag)
    e.free()


@pytest.mark.parametrize("restart", [1, 2, 7, 8, 9, 16, 17, 33, 70])
def test_gmres_cycle_is_the_least_squares_solution(restart):
    """One restart cycle of k steps reaches the least residual over
    M^-1 span(r, A M^-1 r, ...) (computed densely), and the one of the next
    cycle's two steps after it.  M^-1 rounds to FP32 in each of the k steps,
    which moves the residual by about k N 2^-24 |b| (N = 12 unknowns an
    element): below 1e-4 |b|."""
    m, op, ph, q = _problem("vortex", 3, 1, "omega", "roe")
    e = euler.EulerData(m, op, ph)
    e.set_q(q)
    lo, pc = linsolve.HIPBSRLO(e, fp64_blocks=True), linsolve.HIPBJacobiPC(e)
    ndof = q.size
    b = np.random.default_rng(4).standard_normal(q.shape)
    linsolve.StandardLinearSolver(pc, lo).calcPCandLO()
    A, Minv = np.zeros((ndof, ndof)), np.zeros((ndof, ndof))
    for i in range(ndof):
        u, v = np.zeros(ndof), np.zeros(q.shape)
        u[i] = 1.0
        lo.applyLinearOperator(m, op, e, None, None, 0.0, u.reshape(q.shape), v)
        A[:, i] = v.ravel()
        pc.applyPC(m, op, e, None, 0.0, u.reshape(q.shape), v)
        Minv[:, i] = v.ravel()
    K, x_ref = A @ Minv, np.zeros(ndof)
    for cycle, steps in enumerate((restart, 2)):
        r = b.ravel() - A @ x_ref
        V = [r / np.linalg.norm(r)]
        for _ in range(min(steps, restart) - 1):
            w = K @ V[-1]
            for _ in range(2):
                for v in V:
                    w = w - (v @ w) * v
            V.append(w / np.linalg.norm(w))
        Z = np.stack(V, axis=1)
        y = np.linalg.lstsq(K @ Z, r, rcond=None)[0]
        x_ref = x_ref + Minv @ (Z @ y)
        total = restart + cycle * min(2, restart)
        ls = linsolve.StandardLinearSolver(pc, lo, reltol=1e-14, restart=restart, itermax=total)
        x = np.zeros_like(b)
        assert ls.linearSolve(b, x) == total
        got = np.linalg.norm(b.ravel() - A @ x.ravel())
        ref = np.linalg.norm(b.ravel() - A @ x_ref)
        print(restart, total, got / np.linalg.norm(b), ref / np.linalg.norm(b), flush=True)
        assert abs(got - ref) <= 1e-4 * np.linalg.norm(b)
    e.free()


def test_gmres_cycle_longer_than_the_coefficients_in_lds():
    """A cycle of 1,100 unpreconditioned steps, whose coefficients no longer go
    to LDS, reaches the least residual over its Krylov space (numpy, CGS2), to
    the k N eps |A| |x| that a backward stable method allows; the problem is so
    stiff that the residual is still falling there (from 1 to 0.1)."""
    m, op, ph, q = _problem("vortex", 3, 4, "diage", "roe")
    e = euler.EulerData(m, op, ph)
    e.set_q(q)
    lo, pc = linsolve.HIPBSRLO(e, fp64_blocks=True), linsolve.PCNone(e)
    linsolve.StandardLinearSolver(pc, lo).calcPCandLO()
    ndof, k = q.size, 1100
    rowptr, colind = linsolve.getSparsityPattern(e, fp64_blocks=True)
    vals = linsolve.getJacobianValues(e, fp64_blocks=True)
    nd = q.shape[2]
    A4 = np.zeros((ndof // nd, nd, ndof // nd, nd))
    for r in range(len(rowptr) - 1):
        for t in range(rowptr[r], rowptr[r + 1]):
            A4[r, :, colind[t], :] += vals[t]
    A = A4.reshape(ndof, ndof)
    b = np.random.default_rng(4).standard_normal(q.shape)
    V, H = np.zeros((k + 1, ndof)), np.zeros((k + 1, k))
    V[0] = b.ravel() / np.linalg.norm(b)
    for j in range(k):
        w = A @ V[j]
        for _ in range(2):
            h = V[:j + 1] @ w
            w -= V[:j + 1].T @ h
            H[:j + 1, j] += h
        H[j + 1, j] = np.linalg.norm(w)
        V[j + 1] = w / H[j + 1, j]
    g = np.zeros(k + 1)
    g[0] = np.linalg.norm(b)
    x_ref = V[:k].T @ np.linalg.lstsq(H, g, rcond=None)[0]
    ref = np.linalg.norm(b.ravel() - A @ x_ref)
    ls = linsolve.StandardLinearSolver(pc, lo, reltol=1e-14, restart=k, itermax=k)
    x = np.zeros_like(b)
    assert ls.linearSolve(b, x) == k
    got = np.linalg.norm(b.ravel() - A @ x.ravel())
    print(got, ref, flush=True)
    assert ref > 1e-2 * np.linalg.norm(b)
    assert abs(got - ref) <= 2 * k * ndof * 2.0 ** -53 * np.linalg.norm(A, 2) * np.linalg.norm(x_ref)
    e.free()


@pytest.mark.parametrize("kind,p,opk,flux", SHAPES)
def test_jacobian_matches_coloring_at_the_smallest_meshes(kind, p, opk, flux):
    """The element-wise assembly equals the colouring one where the last
    workgroup is part empty: one layer of elements, and two."""
    for n in (1, 2):
        print(f"case {kind} n={n} p={p} {opk} {flux}", flush=True)
        m, op, ph, q = _problem(kind, n, p, opk, flux, shuffle=True)
        e = euler.EulerData(m, op, ph)
        e.set_q(q)
        linsolve.evalJacobian(m, op, e, fp64_blocks=True)
        a = linsolve.getJacobianValues(e, fp64_blocks=True).copy()
        linsolve.calcJacobianSparse(m, op, e, fp64_blocks=True)
        c = linsolve.getJacobianValues(e, fp64_blocks=True)
        assert np.abs(a - c).max() <= 1e-12 * np.abs(a).max()
        e.free()


@pytest.mark.parametrize("pc_kind", [abi.PDES_PC_BJACOBI, abi.PDES_PC_ILU0])
def test_packed_instances_at_the_chunk_edges(pc_kind):
    """Instances of one element pair, of exactly six reduction chunks, of one
    chunk and a bit, and (ILU(0)) of more chunks than a workgroup adds up
    itself solve as they do alone: both end below the tolerance, and the
    states of these coarse meshes agree to 1e-7 (what that tolerance fixes)."""
    opts = linsolve.NewtonOptions(res_abstol=1e-10, krylov_reltol=1e-4, itermax=20, pc_kind=pc_kind)
    sizes = [16, 1, 7] + ([105] if pc_kind == abi.PDES_PC_ILU0 else [])
    inst = [_problem("vortex", n, 1, "omega", "roe") for n in sizes]
    bs = BatchSolver([(m, op, ph) for m, op, ph, q in inst])
    for i, (m, op, ph, q) in enumerate(inst):
        bs.set_state(i, q)
    reps = bs.solve(opts)
    for i, (m, op, ph, q) in enumerate(inst):
        assert reps[i].converged == 1 and reps[i].res_norm < 1e-10
        e = euler.EulerData(m, op, ph)
        e.set_q(q)
        assert linsolve.newton(m, op, e, opts).converged
        alone, packed = e.get_q(), bs.get_state(i)
        e.set_q(packed)
        euler.evalResidual_device(e)
        assert euler.calcNorm(e) < 1e-10
        diff = np.abs(packed - alone).max() / np.abs(alone).max()
        print(sizes[i], reps[i].iterations, diff, flush=True)
        if sizes[i] <= 16:
            assert diff <= 1e-7
        e.free()
    bs.free()


@pytest.mark.parametrize("restart", [33, 62])
def test_packed_cycles_longer_than_a_group_of_vectors(restart):
    """Packed cycles of more basis vectors than a CGS2 pass keeps in registers
    (32), up to the longest: the linear systems of one Newton step run to their
    iteration limit, a whole cycle and two steps more, and end at the residual
    of the single solve.  Block-Jacobi rounds to FP32 in each of the k steps,
    which moves the residual by about k N 2^-24 |b| (N = 24 unknowns an
    element): below 1e-4 |b|."""
    total = restart + 2
    opts = linsolve.NewtonOptions(res_abstol=1e-13, krylov_reltol=1e-14, krylov_itermax=total, itermax=1,
                                  gmres_restart=restart, pc_kind=abi.PDES_PC_BJACOBI, fp64_blocks=True)
    inst = [_problem("vortex", n, 2, "omega", "roe") for n in (20, 6, 14)]
    bs = BatchSolver([(m, op, ph) for m, op, ph, q in inst])
    for i, (m, op, ph, q) in enumerate(inst):
        bs.set_state(i, q)
    reps = bs.solve(opts)
    for i, (m, op, ph, q) in enumerate(inst):
        e = euler.EulerData(m, op, ph)
        e.set_q(q)
        euler.evalResidual(m, op, e)
        b = -e.res.copy()
        alone = linsolve.newton(m, op, e, opts)
        assert reps[i].total_krylov_iters == alone.total_krylov_iters == total
        steps = [e.get_q() - q, bs.get_state(i) - q]
        e.set_q(q)
        lo = linsolve.HIPBSRLO(e, fp64_blocks=True)
        lo.calcLinearOperator(m, op, e)
        r = []
        for dq in steps:
            y = np.zeros_like(dq)
            lo.applyLinearOperator(m, op, e, None, None, 0.0, dq, y)
            r.append(np.linalg.norm(b - y) / np.linalg.norm(b))
        print(restart, i, r, flush=True)
        assert abs(r[0] - r[1]) <= 1e-4
        if i == 0:
            assert r[0] > 1e-3   # still falling: the vectors beyond 32 count
        e.free()
    bs.free()

"""Row tiles of the multi-right-hand-side PCG where they end: fewer rows than a tile, one row past it, a row of
more entries than a tile stages (2049 and more), every column group (1, 2, 4, 8) with empty columns.

Each column is compared with a direct FP64 solve. The stopping test bounds the residual of every column,
r^T D^-1 r <= tol^2 b^T D^-1 b, and x - x* = A^-1 r, so |x - x*|_2 <= |A^-1|_2 max(D)^(1/2) tol (b^T D^-1 b)^(1/2);
to that come the rounding of the recurrence and of the direct solve, 100 cond(A) eps |x*| together.
"""
import time

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def wheel(ctx, spokes):
    """the matrix of a fan of triangles, every fifth rim node held: its hub's row has spokes + 1 entries"""
    from gpupfem2_amd import capi
    t = 2 * np.pi * np.arange(spokes) / spokes
    xy = np.ascontiguousarray(np.concatenate([[[0.0, 0.0]], np.stack([np.cos(t), np.sin(t)], 1)]))
    k = np.arange(spokes)
    tri = np.ascontiguousarray(np.stack([0 * k, 1 + k, 1 + (k + 1) % spokes], 1).astype(np.int32))
    n = spokes + 1
    m = capi.Mesh2D(ctx, xy, tri)
    a, rhs = capi.CSR(ctx, mesh=m), ctx.zeros(n)
    capi.assemble_poisson2d(m, a, rhs, coeff=1.0, rhs_kind=2, rhs_param=0.0)
    fixed = np.arange(1, n, 5, dtype=np.int32)
    capi.Dirichlet(ctx, n, fixed, np.zeros(fixed.size)).apply(a, rhs, 1)
    return m, a, fixed


@pytest.mark.parametrize("mixed", [False, True])
@pytest.mark.parametrize("nrhs", [1, 2, 3, 5, 8])
@pytest.mark.parametrize("spokes", [7, 127, 128, 511, 512, 2046, 2300])
def test_multi_tiles(ctx, oracle, spokes, nrhs, mixed):
    from gpupfem2_amd import capi
    print("multi tiles", spokes, nrhs, mixed, flush=True)
    m, a, fixed = wheel(ctx, spokes)
    n = spokes + 1
    rp, col, val = a.download()
    A = np.zeros((n, n))
    A[np.repeat(np.arange(n), np.diff(rp)), col] = val
    B = np.random.default_rng(spokes + nrhs).standard_normal((nrhs, n))
    B[:, fixed] = 0.0
    tol = 1e-10
    s = capi.Solver(a, capi.SOLVER_CG, tol, 4000, 0, capi.TOL_RELATIVE, capi.Preconditioner(a, capi.PRECOND_JACOBI))
    if mixed:
        s.set_precision(capi.PRECISION_MIXED)
    X = ctx.zeros(nrhs * n)
    stats = s.solve_multi(a, X, ctx.to_device(B.ravel()), nrhs)
    Xh = X.download().reshape(nrhs, n)
    free = np.setdiff1d(np.arange(n), fixed)
    Af, d = A[np.ix_(free, free)], np.diag(A)[free]
    w = np.linalg.eigvalsh(Af)
    for j in range(nrhs):
        assert stats[j].converged, j
        want = np.linalg.solve(Af, B[j, free])
        bound = (d.max() ** 0.5 / w[0] * tol * (B[j, free] ** 2 / d).sum() ** 0.5
                 + 100 * w[-1] / w[0] * 2.3e-16 * np.linalg.norm(want))
        assert np.linalg.norm(Xh[j, free] - want) <= bound, (j, np.linalg.norm(Xh[j, free] - want), bound)
        assert not Xh[j, fixed].any()


@pytest.mark.parametrize("mixed", [False, True])
def test_multi_long_row_cost(ctx, mixed):
    """a row of 2001 entries is staged, one of 5001 is not: walked by one lane it took 600 us a product"""
    from gpupfem2_amd import capi
    took = []
    for spokes in (2000, 5000):
        m, a, fixed = wheel(ctx, spokes)
        b = np.random.default_rng(1).standard_normal(spokes + 1)
        b[fixed] = 0.0
        d = ctx.to_device(b)
        s = capi.Solver(a, capi.SOLVER_CG, 1e-30, 60, 0, capi.TOL_RELATIVE, capi.Preconditioner(a, capi.PRECOND_JACOBI))
        if mixed:
            s.set_precision(capi.PRECISION_MIXED)
        best = np.inf
        for _ in range(4):
            x = ctx.zeros(spokes + 1)
            ctx.sync()
            t = time.perf_counter()
            st = s.solve_multi(a, x, d, 1)
            ctx.sync()
            best = min(best, (time.perf_counter() - t) / max(st[0].iterations, 1))
        took.append(best)
    print("multi long row", mixed, took, flush=True)
    assert took[1] < 2 * took[0], took

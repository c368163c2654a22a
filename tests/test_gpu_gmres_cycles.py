"""GPU: GMRES cycles at the lengths where its kernels change form (eight coefficients to a workgroup, eight basis
vectors loaded together, up to 64 unknowns of the small system in LDS), alone and as a pair: the pair's bits are the
single solves', and the solution agrees with the oracle's modified Gram-Schmidt GMRES as the library's GMRES test
asks (relative L2 <= 1e-10 at tolerance 1e-12)."""
import numpy as np
import pytest

from conftest import rel_l2

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("restart", [5, 7, 8, 9, 16, 17, 63, 64, 65, 200])
def test_gmres_cycles(ctx, oracle, restart):
    from gpupfem2_amd import capi, meshgen
    print("gmres cycles", restart, flush=True)
    xy, tri = meshgen.unit_square(20)
    n = xy.shape[0]
    m = capi.Mesh2D(ctx, xy, tri)
    a, rhs = capi.CSR(ctx, mesh=m), ctx.zeros(n)
    capi.assemble_poisson2d(m, a, rhs, rhs_kind=2, rhs_param=1.0)
    rp, col, val = a.download()
    rng = np.random.default_rng(restart)
    rows = np.repeat(np.arange(n), np.diff(rp))
    # the second of a pair converges well before the first
    vals = [val + np.where(col == rows, d, 0.2 * rng.uniform(-1, 1, col.size) * np.abs(val)) for d in (0.3, 3.0)]
    mats = [capi.CSR(ctx, like=a) for _ in vals]
    bs = [rng.standard_normal(n) for _ in vals]
    single, solvers = [], []
    for mt, v, b in zip(mats, vals, bs):
        mt.upload_values(v)
        s = capi.Solver(mt, capi.SOLVER_GMRES, 1e-12, 3000, restart, capi.TOL_RELATIVE,
                        capi.Preconditioner(mt, capi.PRECOND_JACOBI))
        x = ctx.zeros(n)
        st = s.solve(mt, x, ctx.to_device(b))
        assert st.converged
        single.append((st.iterations, x.download()))
        solvers.append(s)
        xr = np.zeros(n)
        assert oracle.gmres(rp, col, v, xr, b, 1e-12, 3000, restart, 1, "jacobi").converged
        assert rel_l2(single[-1][1], xr) < 1e-10
    assert single[0][0] > single[1][0]
    x = [ctx.zeros(n) for _ in bs]
    st = solvers[0].solve_pair(mats[0], x[0], ctx.to_device(bs[0]), solvers[1], mats[1], x[1], ctx.to_device(bs[1]))
    for k in range(2):
        assert st[k].converged and st[k].iterations == single[k][0]
        assert np.array_equal(x[k].download(), single[k][1])

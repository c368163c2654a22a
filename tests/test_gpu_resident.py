"""GPU: the single-launch (resident) PCG against the launch-per-kernel PCG (SOLVER_OPT_SINGLE_LAUNCH 0), and against a
single launch given up for it (a zero spin limit fails every wait that is not satisfied at once): the same bits of
the solution and the same iteration count, since both add the same partials in the same order. The solver's
counts tell which path each solve took."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


# single launches, launch per kernel, single launches given up
WAYS = ((1, 1 << 16), (0, 1 << 16), (1, 0))


def check_way(s, way, rows):
    """the path that the solver's solves took; systems of up to 1024 rows are one workgroup, which never waits"""
    taken, given_up = s.single_launches()
    if way == WAYS[0]:
        assert taken >= 1 and given_up == 0, (taken, given_up)
    elif way == WAYS[1]:
        assert (taken, given_up) == (0, 0)
    elif rows > 1024:
        assert taken == 0 and given_up >= 1, (taken, given_up)
    else:
        assert taken >= 1 and given_up == 0, (taken, given_up)


def poisson(ctx, nx, ny, seed, jitter=0.2):
    from gpupfem2_amd import capi, meshgen
    xy, tri = meshgen.rectangle(0.0, 2.0, 0.0, 1.0, nx, ny, jitter=jitter, seed=seed)
    m = capi.Mesh2D(ctx, xy, tri, fill_neighbors=False)
    a = capi.CSR(ctx, mesh=m)
    n = xy.shape[0]
    scratch = ctx.zeros(n)
    capi.assemble_poisson2d(m, a, scratch, coeff=1.0, rhs_kind=2, rhs_param=0.0)
    left = np.nonzero(xy[:, 0] < 1e-9)[0].astype(np.int32)
    capi.Dirichlet(ctx, n, left, np.zeros(left.size)).apply(a, scratch)
    b = np.random.default_rng(seed).standard_normal(n)
    b[left] = 0.0
    return m, a, b


# rows: one workgroup, 1024 and one more (a second workgroup with one row), one tile short of and past a
# workgroup, many workgroups, more than 256 tiles (several slots per lane)
@pytest.mark.parametrize("nx,ny", [(1, 1), (15, 15), (31, 31), (40, 24), (63, 19), (100, 50), (400, 100), (361, 361)])
@pytest.mark.parametrize("kind,precision", [(1, 0), (0, 0), (1, 1)])
def test_resident_same_bits(ctx, nx, ny, kind, precision):
    from gpupfem2_amd import capi
    print("resident", nx, ny, kind, precision, flush=True)
    m, a, b = poisson(ctx, nx, ny, seed=nx + ny)
    n = a.n
    start = np.random.default_rng(5).standard_normal(n) * 1e-3
    out = []
    for way in WAYS:
        pc = capi.Preconditioner(a, kind)
        pc.set_spin_limit(way[1])
        s = capi.Solver(a, capi.SOLVER_CG, 1e-11, 8000, 0, capi.TOL_RELATIVE, pc)
        s.set_option(capi.SOLVER_OPT_SINGLE_LAUNCH, way[0])
        if precision:
            s.set_precision(precision, 1e-5, 30)
        x = ctx.to_device(start)
        d = ctx.to_device(b)
        st = s.solve(a, x, d)
        assert st.converged and not st.nan_detected
        check_way(s, way, n)
        out.append((x.download(), st.iterations, st.final_residual, st.refinements))
    assert out[0][1:] == out[1][1:] == out[2][1:]
    assert np.array_equal(out[0][0], out[1][0]) and np.array_equal(out[0][0], out[2][0])


def test_resident_iteration_limit_and_zero(ctx):
    """stopped by the iteration limit: the iterate of that many steps; a zero right-hand side stops at once"""
    from gpupfem2_amd import capi
    m, a, b = poisson(ctx, 60, 60, seed=2)
    out = []
    for way in WAYS:
        pc = capi.Preconditioner(a, 1)
        pc.set_spin_limit(way[1])
        s = capi.Solver(a, capi.SOLVER_CG, 1e-11, 17, 0, capi.TOL_RELATIVE, pc)
        s.set_option(capi.SOLVER_OPT_SINGLE_LAUNCH, way[0])
        x = ctx.zeros(a.n)
        st = s.solve(a, x, ctx.to_device(b))
        assert not st.converged and st.iterations == 17
        out.append(x.download())
        st = s.solve(a, ctx.zeros(a.n), ctx.zeros(a.n))
        assert st.converged and st.iterations == 0
        check_way(s, way, a.n)
    assert np.array_equal(out[0], out[1]) and np.array_equal(out[0], out[2])


@pytest.mark.parametrize("precision", [0, 1])
def test_resident_batch(ctx, precision):
    """systems of one row tile to many workgroups: in FP64 the bits of the launch-per-kernel path; in mixed
    precision both solve to the tolerance with the true residual in the stopping test"""
    from gpupfem2_amd import capi, cases
    case = cases.batched_poisson_case(nmesh=14, tmin=60, tmax=30000, seed=8)
    mesh, a, b = cases.build_batched_poisson(ctx, case)
    rows, n = case["sys_rows"], case["sys_rows"][-1]
    out = []
    for way in WAYS:
        pc = capi.Preconditioner(a, 1)
        pc.set_spin_limit(way[1])
        s = capi.Solver(a, capi.SOLVER_CG, 1e-11, 20000, 0, capi.TOL_RELATIVE, pc)
        s.set_option(capi.SOLVER_OPT_SINGLE_LAUNCH, way[0])
        if precision:
            s.set_precision(precision, 1e-5, 30)
        x = ctx.zeros(n)
        st, ms = s.solve_batched(a, rows, x, b)
        assert all(q.converged and not q.nan_detected for q in st)
        assert (ms > 0).all()
        check_way(s, way, n)
        out.append((x.download(), [q.iterations for q in st], [q.refinements for q in st]))
    if precision:
        assert all(r >= 1 for r in out[0][2])
        assert np.linalg.norm(out[0][0] - out[1][0]) < 1e-8 * np.linalg.norm(out[1][0])
        assert out[1][1] == out[2][1] and np.array_equal(out[1][0], out[2][0])
    else:
        assert out[0][1] == out[1][1] == out[2][1]
        assert np.array_equal(out[0][0], out[1][0]) and np.array_equal(out[0][0], out[2][0])


def test_stepper_counts(ctx):
    """the stepper reports its solvers' single launches: every solve of a small channel step is one"""
    from gpupfem2_amd import cases
    mesh, ph, stepper = cases.build_gpu(ctx, cases.poiseuille_case(nx=40, ny=10, ppc=4, dt=1e-2))
    assert stepper.single_launches() == (0, 0)
    stepper.step()
    first = stepper.single_launches()
    stepper.step()
    assert first[0] > 0 and first[1] == 0 and stepper.single_launches()[0] > first[0]


def test_resident_halo(ctx):
    """nodes numbered at random: a workgroup's rows use more columns of others than it can hold, in all but the last of
    the workgroups. The first launch sees it and none is tried again; in a batch with a system that fits the plan does
    """
    from gpupfem2_amd import capi, meshgen
    xy, tri = meshgen.rectangle(0.0, 2.0, 0.0, 1.0, 100, 50, jitter=0.2, seed=3)
    n = xy.shape[0]
    new = np.random.default_rng(5).permutation(n)
    shuffled = np.empty_like(xy)
    shuffled[new] = xy
    other, other_tri = meshgen.rectangle(0.0, 2.0, 2.0, 3.0, 60, 40, jitter=0.2, seed=4)
    for batch in (False, True):
        p, t = shuffled, new[tri]
        if batch:
            p, t = np.concatenate([p, other]), np.concatenate([t, other_tri + n])
        m = capi.Mesh2D(ctx, np.ascontiguousarray(p), np.ascontiguousarray(t.astype(np.int32)), fill_neighbors=False)
        a = capi.CSR(ctx, mesh=m)
        scratch = ctx.zeros(a.n)
        capi.assemble_poisson2d(m, a, scratch, coeff=1.0, rhs_kind=2, rhs_param=0.0)
        left = np.nonzero(p[:, 0] < 1e-9)[0].astype(np.int32)
        capi.Dirichlet(ctx, a.n, left, np.zeros(left.size)).apply(a, scratch)
        b = np.random.default_rng(1).standard_normal(a.n)
        b[left] = 0.0
        d = ctx.to_device(b)
        s = capi.Solver(a, capi.SOLVER_CG, 1e-9, 4000, 0, capi.TOL_RELATIVE, capi.Preconditioner(a, 1))
        for _ in range(2 if batch else 66):
            x = ctx.zeros(a.n)
            st = s.solve_batched(a, [0, n, a.n], x, d)[0] if batch else [s.solve(a, x, d)]
            assert all(q.converged for q in st)
        assert s.single_launches() == (0, 0)

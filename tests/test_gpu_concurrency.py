"""Two contexts (two streams) on one GPU solving at the same time from two host threads: the multicolour IC0-PCG as
single launches, and as fused launches (single-pass sweeps that wait on values published by earlier workgroups of
their own launch), and the blocked one, each interleaved on the device with the other's launches. Each solve must
give the bits and iteration count it gives alone: a sweep only ever waits on workgroups of its own grid, which
were dispatched before it whatever else the device runs, and a single launch runs only where all its workgroups
fit the device beside those of the others.
"""
import threading
import time

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def pressure_system(ctx, case):
    from gpupfem2_amd import capi
    n = case.xy.shape[0]
    m = capi.Mesh2D(ctx, case.xy, case.tri, fill_neighbors=False)
    a = capi.CSR(ctx, mesh=m)
    rhs = ctx.zeros(n)
    capi.assemble_poisson2d(m, a, rhs, coeff=1.0, rhs_kind=2, rhs_param=1.0)
    capi.Dirichlet(ctx, n, case.bcp_node, case.bcp_val).apply(a, rhs, capi.DIRICHLET_MASK)
    return m, a, rhs


@pytest.mark.parametrize("single", [1, 0])
@pytest.mark.parametrize("orderings", [(1, 1), (1, 2)])
def test_concurrent_solves_two_streams(orderings, single):
    from gpupfem2_amd import capi, cases
    print("concurrent solves", orderings, single, flush=True)
    case = cases.cylinder_case(h=1.0 / 56)
    n = case.xy.shape[0]
    ctxs = [capi.Context(0), capi.Context(0)]
    systems = [pressure_system(c, case) for c in ctxs]

    def make(k):
        c = ctxs[k]
        m, a, rhs = systems[k]
        s = capi.Solver(a, capi.SOLVER_CG, 1e-12, 20000, 0, capi.TOL_RELATIVE,
                        capi.Preconditioner(a, capi.PRECOND_IC0, orderings[k]))
        s.set_option(capi.SOLVER_OPT_SINGLE_LAUNCH, single)
        return s

    def solve(k, s, out):
        c = ctxs[k]
        m, a, rhs = systems[k]
        x = c.zeros(n)
        st = s.solve(a, x, rhs)
        out[k] = (st.converged, st.iterations, x.download())

    solvers = [make(0), make(1)]
    alone = {}
    for k in range(2):
        solve(k, solvers[k], alone)
        assert alone[k][0]
    for rep in range(3):
        together = {}
        threads = [threading.Thread(target=solve, args=(k, solvers[k], together)) for k in range(2)]
        for t in threads:
            t.start()
        for t in threads:
            t.join(timeout=120)
        assert not any(t.is_alive() for t in threads)
        for k in range(2):
            assert together[k][0] and together[k][1] == alone[k][1], (rep, k, together[k][1], alone[k][1])
            assert np.array_equal(together[k][2], alone[k][2]), (rep, k)
    for k in range(2):
        assert solvers[k].single_launches() == (4 if single and orderings[k] == 1 else 0, 0)
    for c in ctxs:
        c.sync()
    # the handles before the contexts they were made on
    del solvers, systems, together, threads
    for c in ctxs:
        c.close()


def test_concurrent_steppers_with_graphs():
    """Two PFEM-2 steppers (the small cylinder and the small Poiseuille channel) on two contexts, stepped
    at the same time from two host threads with the step graphs on: one thread captures its graphs (a
    thread-local capture) while the other launches, allocates and synchronises. Each gives, step by
    step, the forces, fields, iteration counts and particle counts it gives alone."""
    from gpupfem2_amd import capi, cases
    print("concurrent steppers", flush=True)
    case_list = [cases.cylinder_case(h=1.0 / 8, ppc=6, dt=2e-3), cases.poiseuille_case(nx=40, ny=10, ppc=9, dt=2e-3)]
    ctxs = [capi.Context(0), capi.Context(0)]
    steps = 5

    def run(k, out):
        mesh, ph, stepper = cases.build_gpu(ctxs[k], case_list[k], precision=k, inner_tol=1e-5)
        stepper.set_graphs(True)
        res = []
        for s in range(steps):
            f = stepper.step()
            res.append((f.copy(), stepper.fields(), stepper.iterations().copy(), ph.count()))
        out[k] = res
        del stepper, ph, mesh

    alone = {}
    for k in range(2):
        run(k, alone)
    together = {}
    threads = [threading.Thread(target=run, args=(k, together)) for k in range(2)]
    for t in threads:
        t.start()
    for t in threads:
        t.join(timeout=200)
    assert not any(t.is_alive() for t in threads)
    for k in range(2):
        assert k in together, k
        for s, (a, b) in enumerate(zip(alone[k], together[k])):
            assert np.array_equal(a[0], b[0]), (k, s)
            for f in a[1]:
                assert np.array_equal(a[1][f], b[1][f]), (k, s, f)
            assert np.array_equal(a[2], b[2]) and a[3] == b[3], (k, s)
    for c in ctxs:
        c.sync()
    del together, alone, threads
    for c in ctxs:
        c.close()


@pytest.mark.parametrize("kind,order,nx,ny", [(1, 0, 100, 50), (2, 1, 100, 50), (1, 0, 511, 255)])
def test_concurrent_single_launches(kind, order, nx, ny):
    """Four threads' single-launch solves of 6 workgroups each wait rather than compute, and fit the device many
    times over: together they take well under the time of one thread after the other (the same while one solve at a
    time was let onto the device), with the bits each gives alone. Of 128 workgroups each, two fit at a time."""
    from gpupfem2_amd import capi, meshgen
    print("concurrent single launches", kind, nx, flush=True)
    threads, reps = 4, 10 if nx == 100 else 3
    xy, tri = meshgen.rectangle(0.0, 2.0, 0.0, 1.0, nx, ny, jitter=0.2, seed=3)
    left = np.nonzero(xy[:, 0] < 1e-9)[0].astype(np.int32)
    n = xy.shape[0]
    b = np.random.default_rng(1).standard_normal(n)
    b[left] = 0.0
    ctxs = [capi.Context(0) for _ in range(threads)]
    held = []
    for c in ctxs:
        m = capi.Mesh2D(c, xy, tri, fill_neighbors=False)
        a, scratch = capi.CSR(c, mesh=m), c.zeros(n)
        capi.assemble_poisson2d(m, a, scratch, coeff=1.0, rhs_kind=2, rhs_param=0.0)
        capi.Dirichlet(c, n, left, np.zeros(left.size)).apply(a, scratch, 1)
        s = capi.Solver(a, capi.SOLVER_CG, 1e-11, 8000, 0, capi.TOL_RELATIVE, capi.Preconditioner(a, kind, order))
        held.append((m, a, s, c.to_device(b), c.zeros(n)))
        del m, a, s, scratch

    def work(k, out):
        m, a, s, d, x = held[k]
        for _ in range(reps):
            x.zero()
            assert s.solve(a, x, d).converged
        out[k] = x.download()

    out = [{}, {}]
    for k in range(threads):
        work(k, out[0])
    t = time.perf_counter()
    for k in range(threads):
        work(k, out[0])
    alone = time.perf_counter() - t
    ts = [threading.Thread(target=work, args=(k, out[1])) for k in range(threads)]
    t = time.perf_counter()
    for q in ts:
        q.start()
    for q in ts:
        q.join(timeout=60)
    together = time.perf_counter() - t
    assert not any(q.is_alive() for q in ts)
    print("one after the other", alone, "together", together, flush=True)
    for k in range(threads):
        assert np.array_equal(out[0][k], out[0][0]) and np.array_equal(out[1][k], out[0][0])
        assert held[k][2].single_launches() == (3 * reps, 0)
    held.clear()
    for c in ctxs:
        c.close()
    assert together < (0.85 if nx == 100 else 1.2) * alone

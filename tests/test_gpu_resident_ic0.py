"""GPU: the multicolour IC0-PCG whose iterations run as one launch, against the launch-per-kernel iterations
(fusion level 3, whose sweeps are tagged, and level 0): the same operations but for the grouping of the two sums, the
tags and the reciprocal of the factor's diagonal with its correction. Compared as the library's other
reorderings are: iteration counts within 3, relative L2 <= 1e-10 at tolerance 1e-12; two solves of one system are the
same bits. The solver's counts tell which path each solve took."""
import numpy as np
import pytest

from conftest import rel_l2

pytestmark = pytest.mark.gpu


def system(ctx, xy, tri, seed):
    from gpupfem2_amd import capi
    m = capi.Mesh2D(ctx, xy, tri, fill_neighbors=False)
    a = capi.CSR(ctx, mesh=m)
    n = xy.shape[0]
    scratch = ctx.zeros(n)
    capi.assemble_poisson2d(m, a, scratch, coeff=1.0, rhs_kind=2, rhs_param=0.0)
    left = np.nonzero(xy[:, 0] < 1e-9)[0].astype(np.int32)
    capi.Dirichlet(ctx, n, left, np.zeros(left.size)).apply(a, scratch, 1)
    b = np.random.default_rng(seed).standard_normal(n)
    b[left] = 0.0
    return m, a, b


def compare(ctx, a, b, precision, bits, fits=True):
    from gpupfem2_amd import capi
    n = b.size
    d_b = ctx.to_device(b)
    out = []
    for fuse, single, reps in ((3, 1, 2), (3, 0, 2), (0, 1, 1)):
        pc = capi.Preconditioner(a, capi.PRECOND_IC0, capi.ORDER_MULTICOLOR)
        if bits:
            pc.set_factor_bits(bits)
        s = capi.Solver(a, capi.SOLVER_CG, 1e-12, 6000, 0, capi.TOL_RELATIVE, pc)
        if precision:
            s.set_precision(precision, 1e-5, 20)
        s.set_option(capi.SOLVER_OPT_FUSE, fuse)
        s.set_option(capi.SOLVER_OPT_SINGLE_LAUNCH, single)
        for _ in range(reps):
            x = ctx.to_device(np.linspace(-1.0, 1.0, n) * (b != 0))
            st = s.solve(a, x, d_b)
            assert st.converged and not st.nan_detected
            out.append((st.iterations, x.download()))
        assert s.single_launches() == (reps if fits and fuse == 3 and single else 0, 0)
    for k in (0, 2):
        assert out[k][0] == out[k + 1][0] and np.array_equal(out[k][1], out[k + 1][1])
        assert abs(out[k][0] - out[4][0]) <= 3, (k, out[k][0], out[4][0])
        assert rel_l2(out[k][1], out[4][1]) <= 1e-10


# one workgroup, exactly 1024 rows, one row into a second, several, a long strip, more rows than one pass of 64
@pytest.mark.parametrize("nx,ny", [(2, 1), (31, 31), (40, 24), (63, 31), (300, 5), (140, 90), (361, 361)])
@pytest.mark.parametrize("precision,bits", [(0, 0), (2, 32), (2, 16)])
def test_resident_ic0(ctx, nx, ny, precision, bits):
    from gpupfem2_amd import meshgen
    print("resident ic0", nx, ny, precision, bits, flush=True)
    xy, tri = meshgen.rectangle(0.0, 2.0, 0.0, 1.0, nx, ny, jitter=0.2, seed=3)
    m, a, b = system(ctx, xy, tri, nx + ny)
    compare(ctx, a, b, precision, bits)


# nodes numbered at random; two parts without a common node; rows of 9 to 12 and of more neighbours (the latter
# take the other path)
@pytest.mark.parametrize("form", ["shuffled", "parts", "hub10", "hub12", "hub13"])
def test_resident_ic0_meshes(ctx, form):
    from gpupfem2_amd import meshgen
    print("resident ic0", form, flush=True)
    xy, tri = meshgen.rectangle(0.0, 2.0, 0.0, 1.0, 70, 40, jitter=0.2, seed=5)
    n = xy.shape[0]
    rng = np.random.default_rng(9)
    if form == "shuffled":
        new = rng.permutation(n)
        shuffled = np.empty_like(xy)
        shuffled[new] = xy
        xy, tri = shuffled, new[tri].astype(np.int32)
    else:
        k = 30 if form == "parts" else int(form[3:])
        if form == "parts":
            xy2, tri2 = meshgen.rectangle(0.0, 1.0, 2.0, 3.0, k, k, jitter=0.2, seed=6)
        else:
            t = 2 * np.pi * np.arange(k) / k
            xy2 = np.concatenate([[[1.0, 4.0]], np.stack([1.0 + np.cos(t), 4.0 + np.sin(t)], 1)])
            xy2[1 + np.argmin(np.cos(t)), 0] = 0.0     # held
            q = np.arange(k)
            tri2 = np.stack([0 * q, 1 + q, 1 + (q + 1) % k], 1)
        xy = np.concatenate([xy, xy2])
        tri = np.concatenate([tri, tri2 + n]).astype(np.int32)
    m, a, b = system(ctx, np.ascontiguousarray(xy), np.ascontiguousarray(tri), 4)
    compare(ctx, a, b, 0, 0, fits=form != "hub13")


def test_fused_iterations_in_graphs(ctx):
    """launch per kernel at level 3: batches replayed from a HIP graph, with an odd poll interval too and eager work
    between the solves, are the same bits as the kernels one by one"""
    from gpupfem2_amd import capi, meshgen
    xy, tri = meshgen.rectangle(0.0, 2.0, 0.0, 1.0, 70, 40, jitter=0.2, seed=5)
    m, a, b = system(ctx, xy, tri, 4)
    d_b = ctx.to_device(b)
    first = None
    for graph, poll in ((0, 8), (1, 8), (1, 3), (1, 8)):
        s = capi.Solver(a, capi.SOLVER_CG, 1e-12, 6000, 0, capi.TOL_RELATIVE,
                        capi.Preconditioner(a, capi.PRECOND_IC0, capi.ORDER_MULTICOLOR))
        for option, value in ((capi.SOLVER_OPT_SINGLE_LAUNCH, 0), (capi.SOLVER_OPT_GRAPH, graph), (capi.SOLVER_OPT_POLL, poll)):
            s.set_option(option, value)
        for _ in range(3):
            x = ctx.zeros(a.n)
            st = s.solve(a, x, d_b)
            assert st.converged
            now = (st.iterations, x.download())
            first = first or now
            assert now[0] == first[0] and np.array_equal(now[1], first[1]), (graph, poll)
            a.spmv(d_b, x)
            ctx.sync()

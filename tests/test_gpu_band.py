"""GPU: the single-pass sweeps of natural-order IC0/ILU0 factors, in bands (many small levels) and in chunks (what the
bands do not take), against the per-level solves (one launch per level, selected with set_sweep): the same bits."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def square(ctx, n, jitter=0.2):
    from gpupfem2_amd import capi, meshgen
    xy, tri = meshgen.unit_square(n, jitter=jitter, seed=n)
    m = capi.Mesh2D(ctx, xy, tri, fill_neighbors=False)
    a = capi.CSR(ctx, mesh=m)
    rhs = ctx.zeros(a.n)
    capi.assemble_poisson2d(m, a, rhs, coeff=1.0, rhs_kind=2, rhs_param=1.0)
    edge = (np.abs(xy - 0.5) > 0.5 - 1e-9).any(axis=1)
    nodes = np.nonzero(edge)[0].astype(np.int32)
    capi.Dirichlet(ctx, a.n, nodes, np.zeros(nodes.size)).apply(a, rhs)
    return a, m


def box(ctx, n):
    from gpupfem2_amd import capi, meshgen
    xyz, tet = meshgen.box3d(n)
    m = capi.Mesh3D(ctx, xyz, tet)
    a = capi.CSR(ctx, mesh=m)
    rhs = ctx.zeros(a.n)
    capi.assemble_poisson3d(m, a, rhs, coeff=1.0, rhs_kind=2, rhs_param=1.0)
    nodes = np.nonzero(xyz[:, 0] < 1e-9)[0].astype(np.int32)
    capi.Dirichlet(ctx, a.n, nodes, np.zeros(nodes.size)).apply(a, rhs)
    return a, m


def chain(ctx, n):
    """tridiagonal: every row a level of its own, one value passed from band to band"""
    from gpupfem2_amd import capi
    i = np.arange(n)
    col = np.stack([i - 1, i, i + 1], 1)
    val = np.stack([np.full(n, -1.0), 2.5 + 0.1 * np.sin(i), np.full(n, -1.0)], 1)
    keep = (col >= 0) & (col < n)
    rowptr = np.concatenate([[0], np.cumsum(keep.sum(1))]).astype(np.int32)
    return capi.CSR(ctx, rowptr=rowptr, col=col[keep].astype(np.int32), val=val[keep]), None


CASES = {"square_1": (square, 1), "square_40": (square, 40), "square_89": (square, 89), "square_90": (square, 90),
         "square_200": (square, 200), "box_12": (box, 12), "box_22": (box, 22), "chain_8192": (chain, 8192),
         "chain_20001": (chain, 20001)}


@pytest.mark.parametrize("kind", [2, 3])
@pytest.mark.parametrize("name", CASES)
def test_band_sweeps_same_bits(ctx, name, kind):
    from gpupfem2_amd import capi
    print("band sweeps", name, kind, flush=True)
    make, size = CASES[name]
    a, keep = make(ctx, size)
    r = np.random.default_rng(1).standard_normal(a.n)
    # magnitudes at both ends of the range in which a quotient is formed from the reciprocal, and zeros
    r[::7] *= 1e-170
    r[3::11] *= 1e160
    r[5::13] = 0.0
    out = []
    for sweep in (True, False):
        pc = capi.Preconditioner(a, kind, capi.ORDER_NATURAL)
        pc.set_sweep(sweep)
        pc.initialize(a)
        src = ctx.to_device(r)
        z = ctx.zeros(a.n)
        for _ in range(3):      # the published buffers are re-armed between applies
            pc.apply(z, src)
        first = z.download()
        pc.apply(src, src)      # in place
        assert np.array_equal(src.download(), first)
        out.append(first)
    assert np.array_equal(out[0], out[1])


def shuffled(ctx, n):
    """a mesh numbered at random: few levels, each of a good part of the rows"""
    from gpupfem2_amd import capi, meshgen
    xy, tri = meshgen.unit_square(n, jitter=0.2, seed=n)
    new = np.random.default_rng(4).permutation(xy.shape[0])
    q = np.empty_like(xy)
    q[new] = xy
    m = capi.Mesh2D(ctx, q, np.ascontiguousarray(new[tri].astype(np.int32)), fill_neighbors=False)
    a = capi.CSR(ctx, mesh=m)
    rhs = ctx.zeros(a.n)
    capi.assemble_poisson2d(m, a, rhs, coeff=1.0, rhs_kind=2, rhs_param=1.0)
    edge = np.nonzero((np.abs(q - 0.5) > 0.5 - 1e-9).any(axis=1))[0].astype(np.int32)
    capi.Dirichlet(ctx, a.n, edge, np.zeros(edge.size)).apply(a, rhs)
    return a, m


def wide(ctx, n):
    """17 entries on either side of the diagonal, one more than a slice of a band holds"""
    from gpupfem2_amd import capi
    off = np.concatenate([-np.arange(17, 0, -1) * 3, [0], np.arange(1, 18) * 3])
    col = np.arange(n)[:, None] + off[None, :]
    val = np.where(off == 0, 40.0, -1.0)[None, :] + 0.1 * np.sin(np.arange(n))[:, None] * (off == 0)
    keep = (col >= 0) & (col < n)
    rowptr = np.concatenate([[0], np.cumsum(keep.sum(1))]).astype(np.int32)
    return capi.CSR(ctx, rowptr=rowptr, col=col[keep].astype(np.int32), val=val[keep]), None


def far(ctx, n):
    """coupled to rows up to 6000 away: more columns of other bands than a band holds, in many levels"""
    from gpupfem2_amd import capi
    i = np.repeat(np.arange(n), 2)
    j = i - np.random.default_rng(6).integers(1, 6000, i.size)
    lower = sorted(set(zip(i[j >= 0].tolist(), j[j >= 0].tolist())))
    rows = [[] for _ in range(n)]
    for p, q in lower:
        rows[p].append(q)
        rows[q].append(p)
    col, val, rowptr = [], [], [0]
    for p in range(n):
        r = sorted(rows[p] + [p])
        col += r
        val += [float(len(r)) if q == p else -1.0 for q in r]
        rowptr.append(len(col))
    return capi.CSR(ctx, rowptr=np.array(rowptr, np.int32), col=np.array(col, np.int32), val=np.array(val)), None


# what the bands do not take: chunks of the whole factor's levels
CHUNKED = {"shuffled_40": (shuffled, 40), "shuffled_200": (shuffled, 200), "wide_300": (wide, 300), "wide_3000": (wide, 3000),
           "far_30000": (far, 30000)}


@pytest.mark.parametrize("kind", [2, 3])
@pytest.mark.parametrize("name", CHUNKED)
def test_chunked_sweeps_same_bits(ctx, name, kind):
    from gpupfem2_amd import capi
    print("chunked sweeps", name, kind, flush=True)
    make, size = CHUNKED[name]
    a, keep = make(ctx, size)
    r = np.random.default_rng(1).standard_normal(a.n)
    out = []
    for sweep in (True, False):
        pc = capi.Preconditioner(a, kind, capi.ORDER_NATURAL)
        pc.set_sweep(sweep)
        pc.initialize(a)
        src = ctx.to_device(r)
        z = ctx.zeros(a.n)
        for _ in range(3):
            pc.apply(z, src)
        out.append(z.download())
    assert np.array_equal(out[0], out[1])


@pytest.mark.parametrize("kind,solver", [(2, 0), (3, 1)])
@pytest.mark.parametrize("precision", [0, 1, 2])
def test_band_solves(ctx, kind, solver, precision):
    """solves over band sweeps in every precision agree with the FP64 per-level ones"""
    from gpupfem2_amd import capi
    a, keep = square(ctx, 120)
    b = np.random.default_rng(2).standard_normal(a.n)
    x = []
    for sweep in (False, True):
        pc = capi.Preconditioner(a, kind, capi.ORDER_NATURAL)
        s = capi.Solver(a, solver, 1e-11, 2000, 50, capi.TOL_RELATIVE, pc)
        if sweep and precision:
            s.set_precision(precision, 1e-5, 40)
        pc.set_sweep(sweep)
        d = ctx.zeros(a.n)
        st = s.solve(a, d, ctx.to_device(b))
        assert st.converged
        x.append(d.download())
    assert np.linalg.norm(x[1] - x[0]) < 1e-8 * np.linalg.norm(x[0])


@pytest.mark.parametrize("kind", [2, 3])
def test_band_long_chain(ctx, kind):
    """200000 levels in 25 bands that all start together: the last band waits 30 ms for its first value, more than the
    default spin limit of one wait"""
    from gpupfem2_amd import capi
    print("band long chain", kind, flush=True)
    a, keep = chain(ctx, 200000)
    src = ctx.to_device(np.random.default_rng(3).standard_normal(a.n))
    out = []
    pc = capi.Preconditioner(a, kind, capi.ORDER_NATURAL)
    pc.initialize(a)
    for sweep in (True, False):
        pc.set_sweep(sweep)
        z = ctx.zeros(a.n)
        pc.apply(z, src)
        out.append(z.download())
    assert np.array_equal(out[0], out[1])


def test_band_memory(ctx):
    """a chain of 2.6M rows: its slices would take 24 GB (the tables alone took 10); the sweeps take the form whose
    tables are the factor's size"""
    from gpupfem2_amd import capi
    from test_gpu_resources import free_bytes
    a, keep = chain(ctx, 2600000)
    ctx.sync()
    before = free_bytes()
    pc = capi.Preconditioner(a, 2, capi.ORDER_NATURAL)
    ctx.sync()
    took = (before - free_bytes()) / 1e9
    print("band memory", took, "GB", flush=True)
    assert took < 1.0


def test_large_levels_cost(ctx):
    """half bandwidths 2000 and 2001: 100 levels of 2000 rows, none of which overlaps another. A band would take
    such a level 64 rows at a time (1.3 ms an apply); one launch per triangle must not be slower than one per
    level, with the same bits"""
    import time
    from gpupfem2_amd import capi
    n = 200000
    i = np.arange(n)
    col = np.stack([i - 2001, i - 2000, i, i + 2000, i + 2001], 1)
    val = np.tile([-1.0, -1.0, 4.5, -1.0, -1.0], (n, 1))
    keep = (col >= 0) & (col < n)
    rowptr = np.concatenate([[0], np.cumsum(keep.sum(1))]).astype(np.int32)
    a = capi.CSR(ctx, rowptr=rowptr, col=col[keep].astype(np.int32), val=val[keep])
    pc = capi.Preconditioner(a, 2, capi.ORDER_NATURAL)
    pc.initialize(a)
    src = ctx.to_device(np.random.default_rng(1).standard_normal(n))
    took, out = [], []
    for sweep in (True, False):
        pc.set_sweep(sweep)
        z = ctx.zeros(n)
        best = np.inf
        for _ in range(5):
            ctx.sync()
            t = time.perf_counter()
            pc.apply(z, src)
            ctx.sync()
            best = min(best, time.perf_counter() - t)
        took.append(best)
        out.append(z.download())
    print("large levels", took, flush=True)
    assert took[0] < took[1], took
    assert np.array_equal(out[0], out[1])

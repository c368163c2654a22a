"""GPU: the reorder of an advection step where it can go wrong: cells with no, one, and more particles than a
workgroup orders in LDS (1024), counts around its tile of 1024 places, particles that change cell in bulk.
Every array must be the oracle's, bit for bit."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("per_cell", [(0, 1, 3), (1023, 1024, 1025), (5000, 0, 40), (16, 16, 16), (2, 2500, 1100)])
@pytest.mark.parametrize("speed", [0.05, 0.9])
def test_reorder_bits(ctx, oracle, per_cell, speed):
    from gpupfem2_amd import capi, meshgen
    print("reorder", per_cell, speed, flush=True)
    xy, tri = meshgen.rectangle(0.0, 2.0, 0.0, 1.0, 8, 4, jitter=0.2, seed=1)
    area, invJ = oracle.geometry2d(xy, tri)
    off, idx = oracle.neighbors_bruteforce(tri)
    rng = np.random.default_rng(7)
    count = np.array([per_cell[c % 3] for c in range(tri.shape[0])])
    cell = np.repeat(np.arange(tri.shape[0]), count).astype(np.int32)
    n = cell.size
    lam = rng.dirichlet([1.0, 1.0, 1.0], n)
    lam[:, 2] = 1.0 - lam[:, 0] - lam[:, 1]
    pos = np.einsum("pi,pid->pd", lam, xy[tri[cell]])
    state = dict(cell=cell, lam=lam, pos=pos, vel=rng.standard_normal((n, 2)), id=np.arange(n, dtype=np.uint32))
    m = capi.Mesh2D(ctx, xy, tri)
    ph = capi.Particles(m, 4)
    ph.set(state, n)
    oph = oracle.Particles(xy, tri, invJ, off, idx, 4)
    oph.set(state, n)
    u = speed * np.cos(3.0 * xy[:, 1])
    v = 0.3 * speed * np.sin(2.0 * xy[:, 0])
    d0, d1 = ctx.to_device(u), ctx.to_device(v)
    for _ in range(3):
        ph.advect(d0, d1, 0.1, 2)
        oph.advect(u, v, 0.1, 2)
        a, b = ph.get(), oph.get()
        assert a["cell"].size == b["cell"].size
        for k in ("cell", "lam", "pos", "vel", "id"):
            assert np.array_equal(a[k], b[k]), k
        w = [ctx.zeros(xy.shape[0]), ctx.zeros(xy.shape[0])]
        ph.project(w[0], w[1])
        p0, p1 = oph.project(xy.shape[0])
        assert np.array_equal(w[0].download(), p0) and np.array_equal(w[1].download(), p1)

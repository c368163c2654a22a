"""Assembly tiles at their edges: row counts around 256, rows of 255 to 257 entries (the widest that a row's
byte places hold is 256), workgroups with more entries than their LDS sums hold, each face rule. Bit for bit
against the oracle's sequential element loop."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def fan(spokes, extra):
    """A closed fan of `spokes` triangles about node 0, and a strip of `extra` more nodes."""
    t = 2 * np.pi * np.arange(spokes) / spokes
    xy = [np.zeros((1, 2)), np.stack([np.cos(t), np.sin(t)], 1)]
    tri = [np.stack([np.zeros(spokes, int), 1 + np.arange(spokes), 1 + (np.arange(spokes) + 1) % spokes], 1)]
    if extra:
        k = np.arange(extra)
        xy.append(np.stack([3.0 + 0.25 * (k // 2), 1.0 * (k % 2) + 0.01 * k], 1))
        a = 1 + spokes + np.arange(extra - 2)
        tri.append(np.where((np.arange(extra - 2) % 2 == 0)[:, None], np.stack([a, a + 2, a + 1], 1),
                            np.stack([a, a + 1, a + 2], 1)))
    return np.ascontiguousarray(np.concatenate(xy)), np.ascontiguousarray(np.concatenate(tri).astype(np.int32))


@pytest.mark.parametrize("spokes,extra,quad", [(254, 0, 1), (255, 0, 1), (256, 0, 1), (255, 257, 1), (300, 700, 1),
                                               (5, 249, 0), (5, 250, 2), (5, 251, 3), (6, 506, 4)])
def test_assembly_tiles_2d(ctx, oracle, spokes, extra, quad):
    from gpupfem2_amd import capi
    xy, tri = fan(spokes, extra)
    nv = xy.shape[0]
    print("assembly", spokes, extra, quad, flush=True)
    m = capi.Mesh2D(ctx, xy, tri)
    edges = np.full(3 * tri.shape[0], -1, np.int32)
    edges[1:3 * spokes:3] = 2
    m.set_edge_ids(edges)
    normals = np.zeros((8, 2))
    normals[2] = (0.6, 0.8)
    prm_g = capi.make_params(1.3, 0.01, 0.05, 1, 4, normals, face_quad=quad)
    prm_o = oracle.make_params(1.3, 0.01, 0.05, 1, 4, normals, face_quad=quad)
    area, invJ = oracle.geometry2d(xy, tri)
    rp, col = oracle.csr_pattern(nv, tri)
    rng = np.random.default_rng(spokes + extra)
    f = [rng.standard_normal(nv) for _ in range(5)]
    d = [ctx.to_device(v) for v in f]
    a0 = capi.CSR(ctx, mesh=m)
    a1 = capi.CSR(ctx, like=a0)
    r0, r1 = ctx.empty(nv), ctx.empty(nv)

    def same(mats, rhss, ref):
        for got, want in zip([a.download()[2] for a in mats] + [r.download() for r in rhss], ref):
            assert np.array_equal(got, want)

    capi.assemble_poisson2d(m, a0, r0, coeff=0.7, rhs_kind=2, rhs_param=1.5, quad=quad)
    same([a0], [r0], oracle.assemble_poisson2d(xy, tri, area, invJ, rp, col, coeff=0.7, rhs_kind=2, rhs_param=1.5, quad=quad))
    capi.assemble_prediction(m, a0, a1, r0, r1, *d, prm_g)
    same([a0, a1], [r0, r1], oracle.assemble_prediction(xy, tri, area, invJ, edges, rp, col, *f, prm_o))
    capi.assemble_pressure(m, a0, r0, d[0], d[1], d[2], prm_g)
    same([a0], [r0], oracle.assemble_pressure(tri, area, invJ, rp, col, f[0], f[1], f[2], prm_o))
    capi.assemble_correction(m, a0, r0, r1, *d[:4], prm_g)
    same([a0], [r0, r1], oracle.assemble_correction(tri, area, invJ, rp, col, *f[:4], prm_o))


@pytest.mark.parametrize("ring", [253, 254, 255, 600])
def test_assembly_tiles_3d(ctx, oracle, ring):
    """Tetrahedra about one edge: its two nodes' rows hold ring + 2 entries."""
    from gpupfem2_amd import capi
    print("assembly 3d", ring, flush=True)
    t = 2 * np.pi * np.arange(ring) / ring
    xyz = np.concatenate([[[0, 0, 0], [0, 0, 1]], np.stack([np.cos(t), np.sin(t), 0.3 + 0.1 * np.sin(5 * t)], 1)])
    k = np.arange(ring)
    tet = np.ascontiguousarray(np.stack([0 * k, 2 + k, 2 + (k + 1) % ring, 0 * k + 1], 1).astype(np.int32))
    vol, invJ = oracle.geometry3d(xyz, tet)
    rp, col = oracle.csr_pattern(xyz.shape[0], tet)
    m = capi.Mesh3D(ctx, xyz, tet)
    a, rhs = capi.CSR(ctx, mesh=m), ctx.empty(xyz.shape[0])
    capi.assemble_poisson3d(m, a, rhs, coeff=1.0, rhs_kind=2, rhs_param=2.0)
    val, r = oracle.assemble_poisson3d(xyz, tet, vol, invJ, rp, col, 1.0, 2, 2.0)
    assert np.array_equal(a.download()[2], val) and np.array_equal(rhs.download(), r)

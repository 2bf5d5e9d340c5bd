"""The four-wide walk's box tests at their edges: trees of one to nine
primitives (nodes with unused children), and rays that leave the regular
range of the biased test -- zero, tiny, subnormal, huge, infinite and NaN
components, origins on box planes, axis-parallel rays along shared edges of an
axis-aligned grid.  Hit records and occlusion bits equal the oracle's, whose
walk tests every box of the binary tree with the plain slab test."""
import numpy as np
import pytest

import test_gpu_traversal as trav
import wpt

pytestmark = pytest.mark.gpu


def grid_triangles(n, size, material=0):
    """A flat n x n grid at y = 0 of unit cells (flat leaf boxes whose planes
    are the cells' edges) under a row of steps."""
    tris = []
    for i in range(n):
        for k in range(n):
            h = size * ((i + k) % 3 == 0)
            a, b, c, d = ((i + dx - n / 2, h, k + dz - n / 2) for dx, dz in ((0, 0), (1, 0), (1, 1), (0, 1)))
            tris += [wpt.make_triangle(a, b, c, material), wpt.make_triangle(a, c, d, material)]
    return tris


def edge_rays(n, seed, extent):
    rng = np.random.default_rng(seed)
    rays = np.empty((6, n), np.float32)
    rays[0:3] = rng.uniform(-extent, extent, (3, n))
    on_planes = rng.random((3, n)) < 0.5
    rays[0:3][on_planes] = np.round(rays[0:3][on_planes])
    d = rng.normal(size=(3, n))
    rays[3:6] = d / np.linalg.norm(d, axis=0)
    kind = rng.integers(0, 8, n)
    special = rng.random((3, n)) < 0.5
    for k, value in enumerate((0.0, -0.0, 1e-12, 1e-19, 1e-30, 1e-41)):
        where = special & (kind == k)
        rays[3:6][where] = value
    rays[3:6, kind == 6] *= rng.choice(np.float32([1e-25, 1e-10, 1e10, 1e25]), (kind == 6).sum())
    rays[0:3, kind == 7] *= np.float32(1e20)
    return rays


def check(torch, oracle, scene, name, rays):
    want = oracle.trace(rays)
    trav.assert_hits_equal(name, trav.gpu_trace(torch, scene, rays), want)
    hit = want["kind"] != wpt.HIT_NONE
    limits = np.where(hit, want["t"], 1000.0).astype(np.float32)
    for tmax in (limits * np.float32(0.5), limits * np.float32(1.5)):
        assert np.array_equal(trav.gpu_occluded(torch, scene, rays, tmax), oracle.occluded(rays, tmax)), name


@pytest.mark.parametrize("count", [1, 2, 3, 4, 5, 8, 18])
@pytest.mark.parametrize("accel", [wpt.FLAT_SAH_BVH2, wpt.FLAT_MEDIAN_BVH2])
def test_small_flat_trees(torch_cuda, oracle_mod, accel, count):
    b = wpt.SceneBuilder()
    b.material(wpt.make_material(wpt.DIFFUSE, (0.5, 0.5, 0.5)))
    b.flat_triangles = grid_triangles(3, 0.5)[:count]
    b.flat_accelerator = accel
    scene = wpt.Scene(b.desc(), device=True, owner=b)
    check(torch_cuda, oracle_mod.Oracle(scene), scene, f"{count} flat triangles", edge_rays(20000, count, 3.0))


@pytest.mark.parametrize("spheres", [0, 1, 3, 7])
@pytest.mark.parametrize("cells", [1, 2, 9])
def test_instances_and_spheres(torch_cuda, oracle_mod, cells, spheres):
    b = wpt.SceneBuilder()
    b.material(wpt.make_material(wpt.DIFFUSE, (0.5, 0.5, 0.5)))
    mesh = b.mesh(grid_triangles(cells, 0.5))
    b.instance(mesh, wpt.scaled_transform((0, 0, 0), 1))
    b.instance(mesh, wpt.scaled_transform((1, 1, 0), 0.5))
    b.instance(mesh, wpt.scaled_transform((0, -2, 1), axis_scales=(2.0, 1e-3, 0.25)))
    for k in range(spheres):
        b.sphere((k - 3, 1, (k % 3) - 1), 0.5, 0)
    scene = wpt.Scene(b.desc(), device=True, owner=b)
    check(torch_cuda, oracle_mod.Oracle(scene), scene, f"{cells} cells, {spheres} spheres",
          edge_rays(30000, 10 * cells + spheres, 6.0))


def test_non_finite_rays_hit_nothing(torch_cuda):
    b = wpt.SceneBuilder()
    b.material(wpt.make_material(wpt.DIFFUSE, (0.5, 0.5, 0.5)))
    mesh = b.mesh(grid_triangles(5, 0.5))
    b.instance(mesh, wpt.scaled_transform((0, 0, 0), 1))
    b.instance(mesh, wpt.scaled_transform((0, 2, 0), 1))
    scene = wpt.Scene(b.desc(), device=True, owner=b)
    rays = edge_rays(6 * 64, 5, 3.0)
    for component in range(6):
        rays[component, 64 * component:64 * component + 64] = [np.nan, np.inf, -np.inf, np.nan] * 16
    hits = trav.gpu_trace(torch_cuda, scene, rays)
    assert np.all(hits["kind"] == wpt.HIT_NONE)
    assert not trav.gpu_occluded(torch_cuda, scene, rays, np.full(rays.shape[1], 10.0, np.float32)).any()


def bumpy_grid(n, bump, seed):
    """An n x n grid of unit cells whose heights vary by `bump`, as vertices."""
    h = np.random.default_rng(seed).uniform(-bump, bump, (n + 1, n + 1)) if bump else np.zeros((n + 1, n + 1))
    tris = []
    for i in range(n):
        for k in range(n):
            a, b, c, d = ((x - n / 2, h[x, z], z - n / 2) for x, z in ((i, k), (i + 1, k), (i + 1, k + 1), (i, k + 1)))
            tris += [(a, b, c), (a, c, d)]
    return np.array(tris, np.float32)


def aimed_rays(verts, n, seed):
    """Rays at points of the triangles' edges, more than half of them grazing."""
    rng = np.random.default_rng(seed)
    tri = verts[rng.integers(0, len(verts), n)].astype(np.float64)
    e, s = rng.integers(0, 3, n), rng.random((n, 1))
    a, b = tri[np.arange(n), e], tri[np.arange(n), (e + 1) % 3]
    d = rng.normal(size=(n, 3))
    graze = rng.random(n) < 0.6
    d[graze, 1] *= np.exp(rng.uniform(np.log(1e-5), 0, graze.sum()))
    d /= np.linalg.norm(d, axis=1)[:, None]
    origin = (a + (b - a) * s - d * np.exp(rng.uniform(np.log(0.05), np.log(600.0), (n, 1)))).astype(np.float32)
    d = a + (b - a) * s - origin
    d /= np.maximum(np.linalg.norm(d, axis=1), 1e-30)[:, None]
    return np.concatenate([origin.T, d.T]).astype(np.float32)


@pytest.mark.parametrize("accel", [wpt.FLAT_SAH_BVH2, wpt.FLAT_MEDIAN_BVH2, wpt.FLAT_SPATIAL_SPLIT_BVH2,
                                   wpt.FLAT_WIDE8])
@pytest.mark.parametrize("bump", [0.0, 0.3])
def test_rays_at_edges_of_flat_trees(torch_cuda, oracle_mod, accel, bump):
    """Trees of whole triangles: the hits of the oracle's binary walk, in whose
    order the four-wide one goes.  Clipped leaf boxes reach out of the boxes
    around them by rounding, where only a binary walk notices: on the bumpy
    grid the neighbour may be hit instead, at nearly the same distance."""
    verts = bumpy_grid(40, bump, 3)
    b = wpt.SceneBuilder()
    b.material(wpt.make_material(wpt.DIFFUSE, (0.5, 0.5, 0.5)))
    b.flat_triangles = [wpt.make_triangle(*t.tolist(), 0) for t in verts]
    b.flat_accelerator = accel
    scene = wpt.Scene(b.desc(), device=True, owner=b)
    oracle, rays = oracle_mod.Oracle(scene), aimed_rays(verts, 400000, 1)
    if bump == 0.0 or accel != wpt.FLAT_SPATIAL_SPLIT_BVH2:
        check(torch_cuda, oracle, scene, f"accelerator {accel}, bump {bump}", rays)
        return
    want, got = oracle.trace(rays), trav.gpu_trace(torch_cuda, scene, rays)
    assert np.array_equal(got["kind"], want["kind"])
    assert np.allclose(got["t"], want["t"], rtol=1e-3)
    for p, q in zip(*(h["primitive"][got["primitive"] != want["primitive"]] for h in (got, want))):
        assert len(set(map(tuple, verts[p])) & set(map(tuple, verts[q]))) > 0, (p, q)


def test_spill_columns_are_sized_to_the_scene(torch_cuda):
    """A scene of twelve triangles has no deep walks: a regenerating renderer,
    which has no path queues, takes a frame and little else, where 80 stack
    entries for each of its threads alone would be 1 GB."""
    host = wpt.HostScene("cornell-box")
    scene = wpt.Scene(host.desc(), device=True, owner=host)
    torch_cuda.cuda.synchronize()
    before = torch_cuda.cuda.mem_get_info()[0]
    r = wpt.Renderer(scene, host.camera(1920, 1080),
                     wpt.render_config(1920, 1080, spp=1, max_depth=4, mode=wpt.MODE_REGENERATE))
    used = before - torch_cuda.cuda.mem_get_info()[0]
    r.close()
    assert used < 1 << 28, used

"""Ray queries at the sizes where the persistent query kernel changes course: a
single ray, a wavefront and a block with and without a remainder, more rays
than one host piece of 2^20 (whose later pieces must keep the global ray index
as the alpha test's key), occlusion against closest hits, and the device query
of a context that has no traversal stacks yet. All paths run the same traversal
on the same keys, so whole answers are compared bit for bit; the traversal's
agreement with the oracle is covered by the parity tests."""

import numpy as np
import pytest

import vkrt_amd as V
from vkrt_amd import scenes

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


def box_rays(n, seed):
    rng = np.random.default_rng(seed)
    rays = np.zeros((n, 8), np.float32)
    rays[:, 0:3] = rng.uniform(0.02, 0.98, (n, 3))
    d = rng.normal(size=(n, 3))
    rays[:, 4:7] = d / np.linalg.norm(d, axis=1, keepdims=True)
    rays[:, 3], rays[:, 7] = 1e-3, 1e4
    rays[n // 2:, 0:3] += 50.0 * rays[n // 2:, 4:7]  # half start outside the box's bounds and look away
    return rays


def renderer(scene):
    r = V.Renderer(64, 64)
    scenes.load(r, scene)
    r.configure(spp=1, max_depth=4, min_depth=4, mode=V.RENDER_MODE_RGB, rng=V.RNG_PCG32, seed=1)
    r.start(64, 64, 0)
    return r


def device_query(r, rays):
    n = len(rays)
    d = torch.from_numpy(rays).cuda()
    mesh, prim = (torch.empty(n, dtype=torch.int32, device="cuda") for _ in range(2))
    t, bary = torch.empty(n, device="cuda"), torch.empty((n, 2), device="cuda")
    torch.cuda.synchronize()
    r.trace_rays_device_noalloc(d.data_ptr(), n, mesh.data_ptr(), prim.data_ptr(), t.data_ptr(), bary.data_ptr())
    return mesh.cpu().numpy().view(np.uint32), prim.cpu().numpy().view(np.uint32), t.cpu().numpy(), bary.cpu().numpy()


def same(a, b):
    for x, y in zip(a, b):
        assert np.array_equal(x.view(np.uint32), y.view(np.uint32))


@pytest.mark.parametrize("n", [1, 15, 63, 64, 65, 255, 257, 98_303, 393_217, (1 << 20) + 77])
def test_host_and_device_queries_agree(n):
    r = renderer(scenes.alpha_cornell())
    try:
        rays = box_rays(n, n)
        host = r.trace_rays(rays)
        same(host, device_query(r, rays))
        # any prefix of the rays has the same answers (the key is the ray's index)
        part = r.trace_rays(rays[: max(1, n // 3)])
        same([x[: len(part[0])] for x in host], part)
        vis = r.trace_shadow_rays(rays)
        # a ray that no accepted triangle stops is visible, and the other way round
        assert np.array_equal(vis == 1, host[0] == V.VKRT_INVALID_INDEX)
    finally:
        r.close()


def test_device_query_before_the_context_has_traversal_stacks():
    r = renderer(scenes.displaced_sphere(24))
    try:
        rays = box_rays(70_001, 5)
        rays[:, 0:3] -= 0.5
        r.export()  # uploads the scene and builds the tree, and traces nothing
        first = device_query(r, rays)
        host = r.trace_rays(rays)
        assert 0.2 < np.mean(host[0] != V.VKRT_INVALID_INDEX) < 0.9
        same(first, host)
    finally:
        r.close()


def test_queries_without_geometry_miss():
    r = renderer(scenes.Scene())
    try:
        rays = box_rays(321, 9)
        mesh, prim, t, _ = r.trace_rays(rays)
        assert np.all(mesh == V.VKRT_INVALID_INDEX) and np.all(prim == V.VKRT_INVALID_INDEX) and np.all(t == 0.0)
        assert np.all(r.trace_shadow_rays(rays) == 1)
    finally:
        r.close()


@pytest.mark.parametrize("axes", [(0,), (1,), (2,), (0, 1), (1, 2), (0, 2)])
def test_rays_parallel_to_axis_planes_find_every_hit(axes):
    """Directions with components of exactly (plus or minus) zero, from origins
    between the triangles, on their vertices' coordinates and on the scene's
    box: the closest hits of a brute-force search in 64 bits over the same 32-bit
    coordinates, and an occlusion query that agrees."""
    rng = np.random.default_rng(17)
    n = 3000
    pos = (rng.random((n, 1, 3)) + rng.normal(size=(n, 3, 3)) * 0.04).reshape(-1, 3).astype(np.float32)
    count = 600
    rays = np.zeros((count, 8), np.float32)
    d = rng.normal(size=(count, 3))
    d[:, list(axes)] = 0.0
    d /= np.linalg.norm(d, axis=1, keepdims=True)
    d[::2, list(axes)] = -0.0
    rays[:, 4:7] = d
    rays[:, :3] = rng.uniform(0.1, 0.9, (count, 3)) - 3.0 * d
    # a third of the origins lie exactly at a vertex's coordinate, a few at the box's faces
    for a in axes:
        rays[: count // 3, a] = pos[rng.integers(0, len(pos), count // 3), a]
        rays[count // 3: count // 3 + 5, a] = pos[:, a].min()
        rays[count // 3 + 5: count // 3 + 10, a] = pos[:, a].max()
    rays[:, 3], rays[:, 7] = 1e-3, 1e4
    s = scenes.Scene()
    s.materials = [scenes.lambert((0.5, 0.5, 0.5))]
    s.meshes.append(scenes.MeshData(V.make_vertices(pos, np.tile([[0.0, 0.0, 1.0]], (len(pos), 1))),
                                    np.arange(3 * n, dtype=np.uint32).reshape(-1, 3), 0))
    r = renderer(s)
    try:
        mesh, prim, t, _ = r.trace_rays(rays)
        vis = r.trace_shadow_rays(rays)
        v = pos.astype(np.float64).reshape(-1, 3, 3)
        e1, e2 = v[:, 1] - v[:, 0], v[:, 2] - v[:, 0]
        nrm = np.cross(e1, e2)
        want = np.full(count, np.inf)
        for i, ray in enumerate(rays.astype(np.float64)):
            o, dd = ray[:3], ray[4:7]
            ao = o - v[:, 0]
            dao = np.cross(ao, dd)
            with np.errstate(divide="ignore", invalid="ignore"):
                det = -(nrm @ dd)
                tt = (nrm * ao).sum(1) / det
                u, w = (e2 * dao).sum(1) / det, -(e1 * dao).sum(1) / det
                ok = (u >= 0) & (w >= 0) & (u + w <= 1) & (tt > ray[3]) & (tt < ray[7])
            if ok.any():
                want[i] = tt[ok].min()
        hit = mesh != V.VKRT_INVALID_INDEX
        # edges within 32-bit rounding may go either way, as for any ray (see test_gpu_build)
        assert np.mean(hit != np.isfinite(want)) <= 5e-3
        both = hit & np.isfinite(want)
        assert both.mean() > 0.5 and np.mean(np.abs(t[both] - want[both]) > 1e-4) <= 5e-3
        assert np.array_equal(vis == 1, ~hit)
    finally:
        r.close()


def triangle_scene(pos, indices=None):
    s = scenes.Scene()
    s.materials = [scenes.lambert((0.5, 0.5, 0.5))]
    if indices is None:
        indices = np.arange(len(pos), dtype=np.uint32).reshape(-1, 3)
    s.meshes.append(scenes.MeshData(V.make_vertices(np.asarray(pos, np.float32), np.tile([[0.0, 0.0, 1.0]], (len(pos), 1))),
                                    indices, 0))
    return s


def test_hits_behind_the_origin_of_a_thin_scene():
    """A query's interval may begin before its origin. The scene is thinner than the
    1e-5 of a distance by which a frame's rays are tested against its box."""
    pos = [[0.0, 0.0, 0.0], [1.0, 0.0, 3e-4], [0.0, 1.0, 3e-4]]
    rays = np.tile(np.float32([0.2, 0.2, 100.0, -1000.0, 0.0, 0.0, 1.0, 1000.0]), (70, 1))
    rays[1::2, 2] = -100.0
    r = renderer(triangle_scene(pos))
    try:
        mesh, prim, t, _ = host = r.trace_rays(rays)
        assert np.all(mesh == 0) and np.all(prim == 0)
        # z = 3e-4 * (u + v), rounded to the last place of 100
        assert np.allclose(t[::2], -100.0 + 1.2e-4, rtol=0.0, atol=2e-5) and np.all(t[1::2] > 100.0)
        same(host, device_query(r, rays))
        assert np.all(r.trace_shadow_rays(rays) == 0)
    finally:
        r.close()


def test_directions_too_short_for_a_reciprocal_still_slope():
    """(2e-39, 4e-39, 0): 1 / 2e-39 is infinite, as for a ray parallel to the plane
    x = 0, but the ray climbs half as fast in x as in y."""
    pos = [[0.3, 1.0, -0.2], [0.7, 1.0, -0.2], [0.5, 1.0, 0.4]]
    rays = np.zeros((3, 8), np.float32)
    rays[:, 4], rays[:, 5], rays[:, 7] = 2e-39, 4e-39, 3.4e38
    rays[1, 0] = 0.1  # ends at x = 0.6
    rays[2, 0] = 0.25  # passes the triangle
    r = renderer(triangle_scene(pos))
    try:
        mesh, _, t, _ = host = r.trace_rays(rays)
        assert np.array_equal(mesh == 0, [True, True, False])
        # the directions hold 21 bits
        assert np.allclose(t[:2], np.float32(1.0) / rays[:2, 5], rtol=1e-5)
        same(host, device_query(r, rays))
        assert np.array_equal(r.trace_shadow_rays(rays) == 0, mesh == 0)
    finally:
        r.close()


def test_a_device_query_cut_off_by_its_visit_limit_fails():
    """A direction that is not a number meets every box and no triangle, here 4,205,000
    leaves: more than the 2^22 visits a traversal may make, in a tree too shallow to
    overflow the stack. The query has not looked everywhere, and says so."""
    k = 1451
    x, y = np.meshgrid(np.linspace(0.0, 1.0, k), np.linspace(0.0, 1.0, k), indexing="ij")
    pos = np.stack([x, y, 0.1 * np.sin(9.0 * x) * np.cos(7.0 * y)], axis=-1).reshape(-1, 3)
    i = (np.arange(k - 1, dtype=np.uint32)[:, None] * np.uint32(k) + np.arange(k - 1, dtype=np.uint32)).reshape(-1)
    tris = np.concatenate([np.stack([i, i + 1, i + k], 1), np.stack([i + 1, i + k + 1, i + k], 1)]).astype(np.uint32)
    rays = np.float32([[0.5, 0.5, 9.0, 1e-3, np.nan, np.nan, np.nan, 20.0], [0.3, 0.6, 9.0, 1e-3, 0.0, 0.0, -1.0, 20.0]])
    r = renderer(triangle_scene(pos, tris))
    try:
        host = r.trace_rays(rays[1:])
        assert host[0][0] == 0
        assert r.stats().bvhMaxDepth <= 18  # 18 levels of at most 7 pushes: 128 entries hold them
        same(host, device_query(r, rays[1:]))
        with pytest.raises(V.VkrtError):
            device_query(r, rays)
    finally:
        r.close()


def test_a_tree_of_too_many_levels_is_refused():
    """30,000 coincident triangles cluster into a chain: over 4,200 levels of eight
    children, more than the build follows. Nothing may be traced through what is left
    unwritten; the scene without them is traced again."""
    pos = [[0.0, 0.0, 0.0], [1.0, 0.0, 0.0], [0.0, 1.0, 0.0]]
    ray = np.float32([[0.2, 0.2, 1.0, 1e-3, 0.0, 0.0, -1.0, 10.0]])
    s = triangle_scene(pos)
    s.meshes.append(triangle_scene(pos, np.tile(np.uint32([[0, 1, 2]]), (30_000, 1))).meshes[0])
    r = renderer(s)
    try:
        for trace in (lambda: r.trace_rays(ray), lambda: r.trace_shadow_rays(ray), lambda: device_query(r, ray),
                      lambda: r.primary_hits(0), r.draw):
            with pytest.raises(V.VkrtError):
                trace()
        assert r.export().triangleCount == 30_001
        assert r.lib.VKRT_removeMesh(r.h, 1) == 0
        mesh, prim, t, _ = r.trace_rays(ray)
        assert (mesh[0], prim[0], t[0]) == (0, 0, 1.0)
    finally:
        r.close()

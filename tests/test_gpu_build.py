"""The BVH build at the sizes where it changes course (a leaf root, one node, the
switch to the one-workgroup clustering at 2048, several levels), coincident
triangles among them, against a brute-force search; and scene edits, whose device-side
placement must give exactly the scene that was never edited."""

import numpy as np
import pytest

import vkrt_amd as V
from vkrt_amd import scenes

pytestmark = pytest.mark.gpu


def soup(n, seed):
    rng = np.random.default_rng(seed)
    c = rng.random((n, 3))
    pos = (c[:, None, :] + rng.normal(size=(n, 3, 3)) * 0.03).reshape(-1, 3)
    if n > 40:
        pos[30:60] = np.tile(pos[:3], (10, 1))  # coincident triangles: equal Morton codes and zero merged growth
    return pos.astype(np.float32)


def brute_force(pos, rays):
    """Closest hits in 64 bits: t (inf for a miss) by testing every triangle."""
    v = pos.astype(np.float64).reshape(-1, 3, 3)
    e1, e2 = v[:, 1] - v[:, 0], v[:, 2] - v[:, 0]
    n = np.cross(e1, e2)
    out = np.full(len(rays), np.inf)
    for i, r in enumerate(rays.astype(np.float64)):
        o, d = r[:3], r[4:7]
        det = -(n @ d)
        ao = o - v[:, 0]
        dao = np.cross(ao, d)
        with np.errstate(divide="ignore", invalid="ignore"):
            t = (n * ao).sum(1) / det
            u, w = (e2 * dao).sum(1) / det, -(e1 * dao).sum(1) / det
            ok = (u >= 0) & (w >= 0) & (u + w <= 1) & (t > r[3]) & (t < r[7])
        if ok.any():
            out[i] = t[ok].min()
    return out


@pytest.mark.parametrize("n", [1, 2, 3, 8, 9, 65, 2047, 2048, 2049, 5003])
def test_small_builds_find_every_closest_hit(n):
    pos = soup(n, n)
    rng = np.random.default_rng(n + 1)
    rays = np.zeros((1500, 8), np.float32)
    target = pos[rng.integers(0, len(pos), 1500)] + rng.normal(size=(1500, 3)) * 0.01
    o = rng.normal(size=(1500, 3)) * 2.0
    d = target - o
    rays[:, :3], rays[:, 4:7] = o, d / np.linalg.norm(d, axis=1, keepdims=True)
    rays[:, 3], rays[:, 7] = 1e-3, 1e4
    r = V.Renderer(16, 16)
    try:
        s = scenes.Scene()
        s.materials = [scenes.lambert((0.5, 0.5, 0.5))]
        s.meshes.append(scenes.MeshData(V.make_vertices(pos, np.tile([[0.0, 0.0, 1.0]], (len(pos), 1))),
                                        np.arange(3 * n, dtype=np.uint32).reshape(-1, 3), 0))
        scenes.load(r, s)
        mesh, _, t, _ = r.trace_rays(rays)
        want = brute_force(pos, rays)
        hit = mesh != V.VKRT_INVALID_INDEX
        # rays within rounding of an edge may go either way: 32-bit edge functions of
        # coordinates up to 3 have errors of 1e-6, edges of 0.03: under 1 in 1000
        assert np.mean(hit != np.isfinite(want)) <= 2e-3
        both = hit & np.isfinite(want)
        assert both.any() and np.mean(np.abs(t[both] - want[both]) > 1e-4) <= 2e-3
    finally:
        r.close()


def moved_scene(step):
    s = scenes.cornell_box()
    for i, a in ((3, 0.3 * step), (4, -0.2 * step), (5, 0.1 * step)):  # both boxes and the light
        m = np.eye(4)
        m[:2, :2] = [[np.cos(a), -np.sin(a)], [np.sin(a), np.cos(a)]]
        m[:3, 3] = [0.05 * step, 0.02 * step, -0.01 * step]
        s.meshes[i].transform = m
    return s


def draw(r):
    r.start(64, 48, 0)
    r.draw()
    return r.accumulation()


def renderer(scene):
    r = V.Renderer(64, 48)
    scenes.load(r, scene)
    r.configure(spp=4, max_depth=6, min_depth=4, mode=V.RENDER_MODE_RGB, rng=V.RNG_PCG32, seed=2)
    return r


def test_moved_meshes_and_changed_materials_match_a_fresh_scene():
    r = renderer(moved_scene(0))
    try:
        r.add_texture_rgba32f(scenes.sky_environment(32, 16))
        draw(r)
        for step in (1, 2, 3):
            s = moved_scene(step)
            for i, mesh in enumerate(s.meshes):
                m = np.eye(4) if mesh.transform is None else mesh.transform
                r.set_mesh_transform_matrix(i, np.ascontiguousarray(m.T, dtype=np.float32).reshape(-1))
            if step == 2:  # a material between two moves, and an alpha test that comes and goes
                s.meshes[2].opacity = 0.5
                r.set_mesh_opacity(2, 0.5)
                s.materials[1].baseColor[:] = (0.2, 0.3, 0.9)
                r.set_material(2, s.materials[1])
            if step == 3:
                s.materials[1].baseColor[:] = (0.2, 0.3, 0.9)
                r.set_mesh_opacity(2, 1.0)
                r.set_environment_texture(0)
                r.set_environment_light((1.0, 1.0, 1.0), 1.0)
            fresh = renderer(s)
            if step == 3:
                fresh.add_texture_rgba32f(scenes.sky_environment(32, 16))
                fresh.set_environment_texture(0)
                fresh.set_environment_light((1.0, 1.0, 1.0), 1.0)
            want = draw(fresh)
            a, b = r.export(), fresh.export()
            n = a.triangleCount * 9
            assert np.array_equal(np.ctypeslib.as_array(a.worldTriangles, (n,)),
                                  np.ctypeslib.as_array(b.worldTriangles, (n,)))
            fresh.close()
            assert np.array_equal(draw(r), want)
            assert np.array_equal(draw(r), want)
    finally:
        r.close()


def placed_scene():
    """Meshes turned, stretched, mirrored, sheared, moved far and shrunk to thin slivers."""
    rng = np.random.default_rng(23)
    s = scenes.Scene()
    s.materials = [scenes.lambert((0.5, 0.5, 0.5))]
    linear = [np.eye(3), np.diag([0.3, 2.0, 1.1]), np.diag([-1.0, 1.0, 0.7]), np.diag([1.0, 1e-3, 1.0])]
    linear += [rng.normal(size=(3, 3)) for _ in range(4)]
    for k, a in enumerate(linear):
        q = np.linalg.qr(rng.normal(size=(3, 3)))[0]
        m = np.eye(4)
        m[:3, :3] = q @ a
        m[:3, 3] = [2.0 * (k % 4) + (100.0 if k == 7 else 0.0), 2.0 * (k // 4), 0.3 * k]
        count = 70 + 57 * k  # not whole blocks, and meshes that share one
        pos = soup(count, k)
        index = rng.permutation(3 * count).astype(np.uint32).reshape(-1, 3)
        s.meshes.append(scenes.MeshData(V.make_vertices(pos, np.tile([[0.0, 0.0, 1.0]], (len(pos), 1))), index, 0, m))
    return s


def test_the_device_places_the_triangles_that_an_export_shows():
    """The same rays through a scene of transformed meshes, whose triangles the device
    places, and through the exported triangles themselves as meshes that are not
    transformed: the same hits to the last bit. Corners one last place further off
    are told apart."""
    s = placed_scene()
    r = renderer(s)
    try:
        exported = r.export()
        n = exported.triangleCount
        tris = np.ctypeslib.as_array(exported.worldTriangles, (n * 9,)).copy().reshape(n, 3, 3)
        rng = np.random.default_rng(24)
        w = rng.dirichlet([1.0, 1.0, 1.0], n)[:, :, None].astype(np.float32)
        target = np.repeat((tris * w).sum(1), 3, axis=0)
        d = rng.normal(size=target.shape)
        d /= np.linalg.norm(d, axis=1, keepdims=True)
        rays = np.zeros((len(d), 8), np.float32)
        rays[:, :3], rays[:, 4:7], rays[:, 3], rays[:, 7] = target - 3.0 * d, d, 1e-3, 1e4
        placed = r.trace_rays(rays)
        assert np.mean(placed[0] != V.VKRT_INVALID_INDEX) > 0.5
    finally:
        r.close()

    def flat(corners):
        f, first = scenes.Scene(), 0
        f.materials = s.materials
        for mesh in s.meshes:
            pos = corners[first:first + len(mesh.indices)].reshape(-1, 3)
            first += len(mesh.indices)
            f.meshes.append(scenes.MeshData(V.make_vertices(pos, np.tile([[0.0, 0.0, 1.0]], (len(pos), 1))),
                                            np.arange(len(pos), dtype=np.uint32).reshape(-1, 3), 0))
        g = renderer(f)
        try:
            return g.trace_rays(rays)
        finally:
            g.close()

    for a, b in zip(placed, flat(tris)):
        assert np.array_equal(a.view(np.uint32), b.view(np.uint32))
    assert np.mean(placed[2] != flat(np.nextafter(tris, np.float32(np.inf)))[2]) > 0.1

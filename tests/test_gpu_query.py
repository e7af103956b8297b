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

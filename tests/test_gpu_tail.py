"""The fused tail kernel on the GPU: once it takes over a frame's last depths,
the image and the ray counts must be exactly those of the per-depth launches
(every path keeps its random stream and its arithmetic), in every render mode.
A frame picks the tail's first depth from the queue lengths of the previous
frame of the same size, so each case draws two frames and compares the second.
"""

import numpy as np
import pytest

import oracle as O
import vkrt_amd as V
from vkrt_amd import scenes

pytestmark = pytest.mark.gpu


def render_two_frames(scene, w, h, spp, depth, mode, spectral, tail_rays, nee=None, seed=3):
    r = V.Renderer(w, h)
    scenes.load(r, scene)
    r.configure(spp=spp, max_depth=depth, min_depth=4, mode=mode, spectral=spectral, rng=V.RNG_PCG32, seed=seed,
                nee=nee)
    r.set_fused_tail(tail_rays)
    r.start(w, h, 0)
    r.draw()
    first = r.stats()
    r.draw()
    second = r.stats()
    img = r.accumulation()
    r.close()
    return img, first, second


def sphere_scene():
    s = scenes.displaced_sphere(24)
    s.environment = scenes.sky_environment(256, 128)
    return s


def cornell_without_nee():
    return scenes.cornell_box()


CASES = [
    ("sphere hero spectral", sphere_scene, 96, 54, 16, 12, V.RENDER_MODE_SPECTRAL, V.SPECTRAL_HERO, None),
    ("sphere single wavelength", sphere_scene, 64, 36, 16, 12, V.RENDER_MODE_SPECTRAL, V.SPECTRAL_SINGLE, None),
    ("cornell rgb, nee off", cornell_without_nee, 64, 64, 8, 8, V.RENDER_MODE_RGB, V.SPECTRAL_HERO, False),
]


@pytest.mark.parametrize("name,make,w,h,spp,depth,mode,spectral,nee", CASES, ids=[c[0] for c in CASES])
@pytest.mark.parametrize("start", ["depth 1", "short queues"])
def test_fused_tail_gives_the_same_frame(name, make, w, h, spp, depth, mode, spectral, nee, start):
    """A threshold of 2^30 rays hands every depth from 1 on to the tail (long
    queues); a quarter of the frame's paths only the shorter queues of later depths."""
    tail_rays = 1 << 30 if start == "depth 1" else w * h * spp // 4
    ref, _, ref2 = render_two_frames(make(), w, h, spp, depth, mode, spectral, 0, nee)
    img, first, second = render_two_frames(make(), w, h, spp, depth, mode, spectral, tail_rays, nee)
    print(f"{name}: tail from depth {second.tailStartDepth}, {second.tailRays} of {second.extensionRays} rays, "
          f"{second.tailMs:.3f} ms")
    assert ref2.tailStartDepth == 0 and first.tailStartDepth == 0  # no tail: turned off / no previous frame
    assert second.tailStartDepth >= 1 and second.tailLaunches == 1
    if tail_rays == 1 << 30:
        assert second.tailStartDepth == 1
    assert second.extensionRays == ref2.extensionRays
    assert second.tailRays > 0 and second.raysBeforeTail + second.tailRays == second.extensionRays
    assert np.array_equal(img, ref)


def test_fused_tail_frames_match_the_oracle():
    """Two frames of the hero sphere, the second with the tail from depth 1,
    against the FP32 oracle's accumulation of the same two frames."""
    w, h, spp = 48, 27, 8
    r = V.Renderer(w, h)
    scenes.load(r, sphere_scene())
    r.configure(spp=spp, max_depth=12, min_depth=4, mode=V.RENDER_MODE_SPECTRAL, spectral=V.SPECTRAL_HERO,
                rng=V.RNG_PCG32, seed=3)
    r.set_fused_tail(1 << 30)
    r.start(w, h, 0)
    acc, total = None, 0
    for frame in range(2):
        orc = O.OracleScene(r.export(), use_bvh=True)
        r.draw()
        acc, bounces = orc.render(w, h, accum=acc, precision=32)
        orc.close()
        total += bounces
    st = r.stats()
    gpu = r.accumulation()
    r.close()
    assert st.tailStartDepth == 1
    err = O.relmse(gpu[..., :3], acc[..., :3])
    print(f"2-frame relMSE against the oracle {err:.3e}; frame 2: {st.tailRays} of {st.extensionRays} rays in the tail")
    assert np.all(gpu[..., 3] == 2 * spp)
    # measured 6.3e-11, the same with the tail off (the images are identical);
    # the hero sphere's hits on shared edges of the displaced mesh differ
    # between the GPU and the oracle BVH in a few paths
    assert err < 6e-10


def test_statistics_frame_records_the_rays_before_the_tail():
    """With traversal statistics the depths stay separate launches; the frame
    still reports the rays, nodes and triangles before the tail's depth."""
    r = V.Renderer(64, 36)
    scenes.load(r, sphere_scene())
    r.configure(spp=16, max_depth=12, min_depth=4, mode=V.RENDER_MODE_SPECTRAL, spectral=V.SPECTRAL_HERO,
                rng=V.RNG_PCG32, seed=3)
    r.set_fused_tail(4096)
    r.start(64, 36, 0)
    r.draw()
    r.set_traversal_statistics(True)
    r.draw()
    s = r.stats()
    r.close()
    assert s.tailStartDepth == 0 and s.tailRays == 0
    assert 0 < s.raysBeforeTail < s.extensionRays
    assert 0 < s.nodeVisitsBeforeTail < s.nodeVisits and 0 < s.triangleTestsBeforeTail < s.triangleTests


def shadowed_frames(scene, w, h, spp, mode, spectral, tail_rays, env, frames=2):
    r = V.Renderer(w, h)
    scenes.load(r, scene)
    r.configure(spp=spp, max_depth=9, min_depth=4, mode=mode, spectral=spectral, rng=V.RNG_PCG32, seed=5,
                env_importance=env)
    r.set_fused_tail(tail_rays)
    r.start(w, h, 0)
    for _ in range(frames):
        r.draw()
    st, img = r.stats(), r.accumulation()
    r.close()
    return img, st


def lit_glass_under_sky():
    """A light, a sky, dispersive and absorbing glass: both kinds of shadow ray,
    unsupported occluders and collapsed hero wavelengths."""
    s = scenes.cornell_box()
    glass = V.default_material(baseColor=(0.9, 0.95, 0.9), roughness=0.05, metallic=0.0, specular=0.5)
    glass.transmission, glass.ior, glass.abbeNumber = 1.0, 1.5, 30.0
    glass.absorptionCoefficient = 0.5
    glass.attenuationColor[:] = (0.7, 0.9, 0.8)
    s.materials.append(glass)
    s.meshes[4].material = len(s.materials) - 1
    s.environment = scenes.sky_environment(128, 64, sun_radiance=50.0)
    return s


@pytest.mark.parametrize("mode,spectral", [(V.RENDER_MODE_RGB, V.SPECTRAL_HERO),
                                           (V.RENDER_MODE_SPECTRAL, V.SPECTRAL_SINGLE),
                                           (V.RENDER_MODE_SPECTRAL, V.SPECTRAL_HERO)])
@pytest.mark.parametrize("env", [False, True], ids=["light", "light and sky"])
@pytest.mark.parametrize("w,h,spp", [(5, 3, 1), (65, 63, 1), (512, 513, 1), (96, 54, 64)])
def test_fused_tail_with_shadow_rays_gives_the_same_frame(mode, spectral, env, w, h, spp):
    """Whole frames (up to 2^18 paths; 512 x 513 is just above) and tails from a
    later depth against the launches per depth, to the last bit."""
    ref, off = shadowed_frames(lit_glass_under_sky(), w, h, spp, mode, spectral, 0, env)
    assert off.tailLaunches == 0 and off.shadowRays > 0
    paths = w * h * spp
    for rays in (1 << 20, paths // 2):
        if rays == 0:
            continue
        img, st = shadowed_frames(lit_glass_under_sky(), w, h, spp, mode, spectral, rays, env)
        whole = paths <= min(rays, 1 << 18)
        # the second frame always ends in a tail: the queue of depth 1 is below 2^19 in
        # every case, and half of half the paths are left after a few depths
        assert st.tailLaunches == 1
        assert st.tailStartDepth == 0 if whole else st.tailStartDepth == 1 if rays == 1 << 20 else st.tailStartDepth > 1
        assert st.tailRays > 0 or paths < 100
        assert st.extensionRays == off.extensionRays and st.shadowRays == off.shadowRays
        assert st.raysBeforeTail + st.tailRays == st.extensionRays
        assert np.array_equal(img, ref)


def test_depths_that_a_tail_carried_have_no_known_length():
    """A frame whose tail began at depth 0 has counted no later queue: with a limit
    below its paths the next frame starts no tail, and the ones after it start where
    the lengths counted in between allow."""
    w = h = 64
    depth, limit = 9, 1600
    r = V.Renderer(w, h)
    scenes.load(r, scenes.cornell_box())
    r.configure(spp=1, max_depth=depth, min_depth=4, mode=V.RENDER_MODE_RGB, rng=V.RNG_PCG32, seed=5)
    r.start(w, h, 0)
    stats = []
    for rays in (1 << 20, limit, limit, limit // 4):
        r.set_fused_tail(rays)
        r.draw()
        stats.append(r.stats())
    r.close()
    whole, unknown, known, later = stats
    assert whole.tailLaunches == 1 and whole.tailStartDepth == 0
    assert unknown.tailLaunches == 0
    # shadow rays halve the limit; a tail of n paths traces at most n rays a depth, and the
    # counts are those of the frame before (a quarter more than 5 of their deviations)
    assert known.tailLaunches == 1 and known.tailStartDepth > 1
    assert 0 < known.tailRays <= 1.25 * (limit // 2) * (depth - known.tailStartDepth)
    # deeper queues keep the lengths of the frame that counted them
    assert later.tailLaunches == 1 and later.tailStartDepth > known.tailStartDepth
    assert 0 < later.tailRays <= 1.25 * (limit // 8) * (depth - later.tailStartDepth)

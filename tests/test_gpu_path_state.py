"""What the path tracer keeps per path: the pixel and sample of a path index, and
hero radiance across the collapse to one wavelength."""

import numpy as np
import pytest

import oracle as O
import vkrt_amd as V
from vkrt_amd import scenes

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


def same_seed(scene, w, h, spp, mode, depth=6):
    r = V.Renderer(w, h)
    try:
        scenes.load(r, scene)
        r.configure(spp=spp, max_depth=depth, min_depth=4, mode=mode, spectral=V.SPECTRAL_HERO, rng=V.RNG_PCG32, seed=4)
        r.start(w, h, 0)
        orc = O.OracleScene(r.export(), use_bvh=False)
        r.draw()
        return r.accumulation()[..., :3], orc.render(w, h, precision=32)[0][..., :3]
    finally:
        r.close()


@pytest.mark.parametrize("w,h", [(1, 1), (1, 67), (129, 1), (33, 31), (128, 2)])
@pytest.mark.parametrize("mode", [V.RENDER_MODE_RGB, V.RENDER_MODE_SPECTRAL])
def test_every_path_finds_its_pixel(w, h, mode):
    gpu, ref = same_seed(scenes.cornell_box(), w, h, 5, mode)
    # a path of another pixel or sample has another random stream: nothing would agree
    # (the bound of the same-seed parity tests, where a decision flips once in 1e6 vertices)
    assert np.mean(np.abs(gpu - ref) <= 1e-4 * (1.0 + np.abs(ref))) > 0.999


def test_lights_seen_past_a_collapse_count():
    """Dispersive glass collapses a hero path; the next-event contributions of its
    later vertices, the last one included, belong to the collapsed radiance."""
    s = scenes.cornell_box()
    s.materials.append(V.default_material(baseColor=(1.0, 1.0, 1.0), roughness=0.3, metallic=0.0, specular=0.0,
                                          transmission=1.0, ior=1.5, abbeNumber=20.0))
    for i in (3, 4):  # both boxes
        s.meshes[i].material = len(s.materials) - 1
    # three vertices: the collapse, one after it, and no long chain through glass, which
    # turns last-place differences into other paths with or without dispersion
    gpu, ref = same_seed(s, 64, 64, 16, V.RENDER_MODE_SPECTRAL, depth=3)
    # the bound of the same-seed parity tests (a lost contribution shows in 3 of 12,288 values)
    assert np.mean(np.abs(gpu - ref) <= 1e-4 * (1.0 + np.abs(ref))) > 0.9999


@pytest.mark.parametrize("mode,spectral,nee,size", [
    # random state, flags, throughput, radiance, medium, hit, sample, two queues of two 16-byte records
    (V.RENDER_MODE_RGB, V.SPECTRAL_HERO, False, 164),
    (V.RENDER_MODE_SPECTRAL, V.SPECTRAL_SINGLE, False, 180),  # and the wavelength
    (V.RENDER_MODE_SPECTRAL, V.SPECTRAL_HERO, False, 228),  # and collapsed state and radiance, pdfs
    (V.RENDER_MODE_SPECTRAL, V.SPECTRAL_HERO, True, 324),  # and the last vertex's pdfs, shadow rays
])
def test_a_path_takes_the_memory_that_its_mode_uses(mode, spectral, nee, size):
    r = V.Renderer(256, 256)
    try:
        scenes.load(r, scenes.cornell_box())
        r.configure(spp=1, max_depth=3, min_depth=2, mode=mode, spectral=spectral, rng=V.RNG_PCG32, seed=4, nee=nee)
        r.start(256, 256, 0)
        r.draw()
        before = torch.cuda.mem_get_info()[0]
        r.configure(spp=65)
        r.draw()
        grown = before - torch.cuda.mem_get_info()[0]
        # some twenty allocations, of whole pages; a record of 16 bytes per path is 65 MiB
        assert abs(grown - 65 * 256 * 256 * size) < 16 << 20
    finally:
        r.close()

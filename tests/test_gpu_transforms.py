"""Shading under mesh transforms against the FP32 oracle: the rotation and scale
terms of a mesh are computed once per upload and read by every hit."""

import numpy as np
import pytest

import oracle as O
import vkrt_amd as V
from vkrt_amd import scenes

pytestmark = pytest.mark.gpu


def rotation(ax, ay, az):
    c, s = np.cos([ax, ay, az]), np.sin([ax, ay, az])
    x = np.array([[1, 0, 0], [0, c[0], -s[0]], [0, s[0], c[0]]])
    y = np.array([[c[1], 0, s[1]], [0, 1, 0], [-s[1], 0, c[1]]])
    z = np.array([[c[2], -s[2], 0], [s[2], c[2], 0], [0, 0, 1]])
    return z @ y @ x


@pytest.mark.parametrize("mode,spectral", [(V.RENDER_MODE_RGB, V.SPECTRAL_HERO),
                                           (V.RENDER_MODE_SPECTRAL, V.SPECTRAL_SINGLE),
                                           (V.RENDER_MODE_SPECTRAL, V.SPECTRAL_HERO)])
@pytest.mark.parametrize("scale", [(0.7, 0.7, 0.7), (0.5, 1.2, 0.8), (-0.8, 0.6, 0.9), (0.9, 0.9, 1e-7)])
def test_transformed_meshes_match_the_oracle(mode, spectral, scale):
    w = h = 64
    s = scenes.cornell_box()
    for i in (3, 4):  # both boxes
        m = np.eye(4) if s.meshes[i].transform is None else np.array(s.meshes[i].transform, dtype=np.float64)
        t = np.eye(4)
        t[:3, :3] = rotation(0.1 * i, -0.07, 0.3 * i) @ np.diag(scale)
        s.meshes[i].transform = m @ t
    r = V.Renderer(w, h)
    try:
        scenes.load(r, s)
        r.configure(spp=8, max_depth=6, min_depth=4, mode=mode, spectral=spectral, rng=V.RNG_PCG32, seed=5)
        r.start(w, h, 0)
        orc = O.OracleScene(r.export(), use_bvh=True)
        r.draw()
        gpu = r.accumulation()
        ref, bounces = orc.render(w, h, precision=32)
        # the two sides' sines may differ in the last place, which moves a decision of a
        # diffuse path (roulette, a shadow edge) about once in a million vertices; a pixel
        # has some 40
        assert abs(r.stats().extensionRays - bounces) <= max(8, 1e-4 * bounces)
        assert np.mean(np.abs(gpu[..., :3] - ref[..., :3]) <= 1e-4 * (1.0 + np.abs(ref[..., :3]))) > 0.999
    finally:
        r.close()

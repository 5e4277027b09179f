"""Exact-ray raster tiles in their bins (gfx950) at image sizes around a bin and a raster tile and at
camera counts that leave the last round of bins ragged, scales from far below a pixel to several
bins wide (rays beside, on and inside a splat's support), against the CPU oracle.
"""

from __future__ import annotations

import pytest

from gpu_helpers import compare_images, render_oracle, render_service
from vgr_amd import synthetic

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("tile_size", [16, 8])
@pytest.mark.parametrize("width,height,cameras", [(1, 1, 1), (31, 33, 3), (32, 32, 2), (65, 17, 5), (129, 97, 1)])
@pytest.mark.parametrize("scale", [0.02, 1.0, 20.0])
def test_ragged_ray_images_match_the_oracle(tile_size, width, height, cameras, scale):
    scene = synthetic.gaussian_scene(1500, seed=width, sh_degree=1)
    scene.scales = scene.scales * scale
    rig = synthetic.orbit_rig(cameras, width, height, 0.9 * width, seed=height, radius=(9.0, 12.0))
    gpu, _ = render_service([(0, scene)], rig, [0] * cameras, ray_gaussian_evaluation=True, tile_size=tile_size)
    compare_images(gpu, render_oracle([(0, scene)], rig, [0] * cameras, sh_degree=1, tile_size=tile_size,
                                      ray_evaluation=True))

"""Needle-shaped splats against the compositor's test of which 8x8 blocks a splat reaches (gfx950): conics
of condition from 10 to beyond 1e5, where the test gives up and keeps the splat, means inside the image and
far outside it, against the CPU oracle, which tests every pixel.  A splat left out of a block that it reaches
changes alpha by 1/255 or more there.
"""

from __future__ import annotations

import math

import pytest
import torch

from gpu_helpers import compare_images, render_oracle, render_service
from vgr_amd import synthetic

pytestmark = pytest.mark.gpu


def needles(count: int, size: int, condition: float, epsilon: float, outside: float) -> synthetic.SyntheticScene:
    """Needles in the image plane: the screen variances are ``condition`` x and 1 x a minor one of about
    ``epsilon`` + 0.1; means over ``outside`` times the image."""
    g = torch.Generator().manual_seed(int(condition) + size)
    z = 4.0 + 4.0 * torch.rand(count, generator=g)
    minor = epsilon + 0.1
    long_px = (condition * minor) ** 0.5 * (0.7 + 0.3 * torch.rand(count, generator=g))
    per_px = z / size
    scales = torch.stack([long_px * per_px, 0.1 ** 0.5 * per_px, torch.full_like(z, 1.0e-4)], dim=1)
    angle = math.pi * torch.rand(count, generator=g)
    rotations = torch.stack([torch.cos(angle / 2), torch.zeros(count), torch.zeros(count), torch.sin(angle / 2)], dim=1)
    xy = outside * (torch.rand((count, 2), generator=g) - 0.5) * z[:, None]
    opacity = 1.0 / 255.0 * 10.0 ** (2.4 * torch.rand(count, generator=g))
    return synthetic.SyntheticScene(
        torch.cat((xy, z[:, None]), dim=1).contiguous(), scales.contiguous(), rotations.contiguous(), opacity,
        torch.rand((count, 3), generator=g), torch.arange(count, dtype=torch.int64))


@pytest.mark.parametrize("epsilon", [0.3, 0.001])
@pytest.mark.parametrize("outside", [1.0, 6.0])
@pytest.mark.parametrize("condition", [10.0, 1.0e3, 3.0e4, 9.0e4, 3.0e5])
@pytest.mark.parametrize("size,tile_size", [(96, 16), (96, 8), (592, 16)])  # by block, by block, whole tiles
def test_needles_match_the_oracle(size, tile_size, condition, outside, epsilon):
    scene = needles(400, size, condition, epsilon, outside)
    rig = synthetic.single_camera(size, size, float(size))
    rig.viewmats[:] = torch.eye(4)
    options = dict(tile_size=tile_size, covariance_epsilon=epsilon)
    gpu, backend = render_service([(0, scene)], rig, [0], max_intersections=3_000_000, max_visible_records=400, **options)
    assert backend.read_counters()["visible_gaussians"] > 0
    compare_images(gpu, render_oracle([(0, scene)], rig, [0], **options))

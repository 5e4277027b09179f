"""Long tiles rendered by a workgroup per 8x8 block (gfx950): list lengths around its batch (256),
step (24) and row store (384), beside short tiles that take the ordinary way, at ragged image sizes,
faint (no pixel ends) and opaque (pixels end inside a step), against the CPU oracle.
"""

from __future__ import annotations

import pytest
import torch

from gpu_helpers import compare_images, render_oracle, render_service
from vgr_amd import synthetic

pytestmark = pytest.mark.gpu


def scene_of(count: int, opacity: float) -> synthetic.SyntheticScene:
    """``count`` Gaussians in one small patch of the view and 40 over all of it."""
    g = torch.Generator().manual_seed(count)
    total = count + 40
    z = 4.0 + 4.0 * torch.rand(total, generator=g)
    spread = torch.cat((torch.full((count,), 0.06), torch.full((40,), 0.5)))
    xy = (2.0 * torch.rand((total, 2), generator=g) - 1.0) * spread[:, None] * z[:, None]
    return synthetic.SyntheticScene(
        torch.cat((xy, z[:, None]), dim=1).contiguous(), torch.full((total, 3), 0.05),
        torch.tensor([1.0, 0.0, 0.0, 0.0]).repeat(total, 1), torch.full((total,), opacity),
        torch.rand((total, 3), generator=g), torch.arange(total, dtype=torch.int64))


@pytest.mark.parametrize("width,height,tile_size", [(16, 16, 16), (75, 53, 16), (75, 53, 8)])
@pytest.mark.parametrize("count", [1, 23, 25, 256, 257, 385, 769, 3000])
@pytest.mark.parametrize("opacity", [0.008, 0.6])
def test_long_lists_match_the_oracle(width, height, tile_size, count, opacity):
    scene = scene_of(count, opacity)
    rig = synthetic.single_camera(width, height, float(width))
    rig.viewmats[:] = torch.eye(4)
    gpu, _ = render_service([(0, scene)], rig, [0], tile_size=tile_size)
    compare_images(gpu, render_oracle([(0, scene)], rig, [0], tile_size=tile_size))
    rgb, _ = render_service([(0, scene)], rig, [0], tile_size=tile_size, outputs=("rgb",))
    assert (rgb["rgb"] == gpu["rgb"]).all()

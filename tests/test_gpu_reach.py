"""Grids whose long tiles are told by how far they are composited (gfx950; 769 to 1,280 tiles of 16x16 with
lists of 5,000 entries and more on average): the choice is one of schedule, so images are those of the render
that counts evaluations, which gives every tile to one workgroup, and of the CPU oracle.

7,500 wide splats make most tiles opaque early (faint: after 2,000 entries; opaque: after a few); where they
end, patches of small ones lie that stay open to the end of lists past the sampled span.
"""

from __future__ import annotations

import numpy as np
import pytest
import torch

from gpu_helpers import compare_images, device, render_oracle
from vgr_amd import CustomHipBackend, RendererService, synthetic
from vgr_amd.autograd import DifferentiableRenderer
from vgr_amd.batched import BatchedRenderer, CameraSpec

pytestmark = pytest.mark.gpu

NAMES = ("rgb", "depth", "alpha", "semantic_id")


def open_edge(opacity: float) -> synthetic.SyntheticScene:
    """Wide splats on the left of the view; patches of 9000, 3000, 600 and 500 small ones on its right."""
    g = torch.Generator().manual_seed(int(1000 * opacity))
    counts = torch.tensor([7500, 9000, 3000, 600, 500])
    part = torch.repeat_interleave(torch.arange(5), counts)
    total = int(counts.sum())
    z = 4.0 + 4.0 * torch.rand(total, generator=g)
    centres = torch.tensor([[-0.48, 0.0], [0.47, -0.3], [0.46, 0.1], [0.47, 0.35], [0.2, 0.2]])
    spread = torch.tensor([0.01, 0.008, 0.02, 0.01, 0.01])
    scale = torch.tensor([0.9, 0.004, 0.004, 0.004, 0.004])
    xy = (centres[part] + (2.0 * torch.rand((total, 2), generator=g) - 1.0) * spread[part, None]) * z[:, None]
    order = torch.randperm(total, generator=g)
    return synthetic.SyntheticScene(
        torch.cat((xy, z[:, None]), dim=1)[order].contiguous(), (scale[part] * z)[order, None].repeat(1, 3),
        torch.tensor([1.0, 0.0, 0.0, 0.0]).repeat(total, 1), torch.full((total,), opacity),
        torch.rand((total, 3), generator=g), torch.arange(total, dtype=torch.int64))


def view(width: int, height: int):
    rig = synthetic.single_camera(width, height, float(width))
    rig.viewmats[:] = torch.eye(4)
    return rig


def render(scene, rig, *, counting: bool):
    dev = device()
    backend = CustomHipBackend(output_srgb=False, max_intersections=24_000_000, max_visible_records=30_000)
    if counting:
        backend.statistics = torch.zeros(4, dtype=torch.int64, device=dev)
    service = RendererService(backend, height=rig.heights[0], width=rig.widths[0], max_views=1)
    service.initialize(stage=None, device=dev)
    service.load_scene(0, **scene.to(dev).as_kwargs())
    out = service.render(rig.viewmats.to(dev), rig.intrinsics.to(dev), torch.zeros(1, dtype=torch.int64, device=dev))
    service.synchronize()
    return {name: out[name].cpu().numpy() for name in NAMES}, backend


@pytest.mark.parametrize("width,height", [(445, 437), (512, 512), (573, 565)])  # 784, 1,024 and 1,296 tiles
@pytest.mark.parametrize("opacity", [0.006, 0.05, 0.7])
def test_images_do_not_depend_on_the_reach(width, height, opacity):
    scene, rig = open_edge(opacity), view(width, height)
    got, backend = render(scene, rig, counting=False)
    lengths = backend.workspace["tile_ends"] - backend.workspace["tile_starts"]
    assert backend.read_counters()["tile_intersections"] >= 5000 * lengths.numel()
    assert backend.read_counters()["intersection_overflow"] == 0
    whole, _ = render(scene, rig, counting=True)
    for name in NAMES:
        np.testing.assert_array_equal(got[name], whole[name], err_msg=name)
    if width == 445:
        compare_images(got, render_oracle([(0, scene)], rig, [0]))


def test_uneven_resolutions():
    scene = open_edge(0.05)
    dev = device()
    specs = [CameraSpec(0, 333, 251), CameraSpec(0, 160, 120), CameraSpec(0, 401, 303)]  # 910 tiles
    views = torch.eye(4, device=dev).repeat(3, 1, 1)
    intrinsics = torch.cat([synthetic.pinhole(1, s.width, s.height, float(s.width)) for s in specs]).to(dev)
    renderer = BatchedRenderer(device=dev, ordering="global")
    renderer.register_scene(0, **scene.to(dev).as_kwargs())
    renderer.plan(specs, visible_capacity=90_000, intersection_capacity=24_000_000)
    renderer.set_cameras(views, intrinsics)
    out = {name: tensor.clone() for name, tensor in renderer.render().items()}
    assert renderer.check_capacity()["tile_intersections"] >= 5000 * renderer.total_tiles
    offset = 0
    for spec in specs:
        whole, _ = render(scene, view(spec.width, spec.height), counting=True)
        for name, tensor in whole.items():
            rows = out[name][offset:offset + spec.width * spec.height].cpu().numpy()
            np.testing.assert_array_equal(rows.reshape(tensor.shape), tensor, err_msg=name)
        offset += spec.width * spec.height


@pytest.mark.parametrize("opacity", [0.02, 0.6])
def test_training_slots(opacity):
    scene, rig = open_edge(opacity), view(512, 480)  # 960 tiles
    dev = device()
    renderer = DifferentiableRenderer(height=480, width=512, device=dev, visible_capacity=30_000,
                                      intersections_per_visible=800.0)
    log_scales, logits = torch.log(scene.scales).to(dev), torch.logit(scene.opacities).to(dev)
    out = renderer.render(scene.means.to(dev).requires_grad_(), log_scales, scene.rotations.to(dev), logits,
                          scene.features.to(dev), rig.viewmats.to(dev), rig.intrinsics.to(dev), sh_degree=0)
    # exp / sigmoid as the renderer evaluates them, so both renders see the same bits.
    scene.scales, scene.opacities = torch.exp(log_scales).cpu(), torch.sigmoid(logits).cpu()
    whole, _ = render(scene, rig, counting=True)
    for name in ("rgb", "depth", "alpha"):
        np.testing.assert_array_equal(out[name].detach().cpu().numpy(), whole[name], err_msg=name)

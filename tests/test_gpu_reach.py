"""Grids whose long tiles are told by how far they are composited (gfx950; 769 to 1,280 tiles of 16x16 and
room for long lists): the choice is one of schedule, so images, checkpoints and gradients are those of a
render whose workspace has no room for long lists, and of the CPU oracle.

Faint and opaque patches (never and early opaque), a list longer than the sampled span, ragged edges.
"""

from __future__ import annotations

import numpy as np
import pytest
import torch

from gpu_helpers import compare_images, device, render_oracle, render_service
from vgr_amd import synthetic
from vgr_amd.autograd import DifferentiableRenderer
from vgr_amd.batched import BatchedRenderer, CameraSpec

pytestmark = pytest.mark.gpu


def patches(opacity: float, counts=(9000, 3000, 600, 500)) -> synthetic.SyntheticScene:
    """A patch of each count in one part of the view, and 3000 over all of it."""
    g = torch.Generator().manual_seed(int(1000 * opacity))
    total = sum(counts) + 3000
    z = 4.0 + 4.0 * torch.rand(total, generator=g)
    centres = torch.tensor([[-0.3, -0.3], [0.31, -0.2], [0.05, 0.35], [-0.46, 0.46], [0.0, 0.0]])
    spread = torch.tensor([0.012, 0.02, 0.01, 0.01, 0.5])
    part = torch.repeat_interleave(torch.arange(5), torch.tensor([*counts, 3000]))
    xy = (centres[part] + (2.0 * torch.rand((total, 2), generator=g) - 1.0) * spread[part, None]) * z[:, None]
    order = torch.randperm(total, generator=g)
    return synthetic.SyntheticScene(
        torch.cat((xy, z[:, None]), dim=1)[order].contiguous(), torch.full((total, 3), 0.03),
        torch.tensor([1.0, 0.0, 0.0, 0.0]).repeat(total, 1), torch.full((total,), opacity),
        torch.rand((total, 3), generator=g), torch.arange(total, dtype=torch.int64))


def view(width: int, height: int):
    rig = synthetic.single_camera(width, height, float(width))
    rig.viewmats[:] = torch.eye(4)
    return rig


@pytest.mark.parametrize("width,height", [(445, 437), (512, 512), (573, 565)])  # 784, 1,024 and 1,296 tiles
@pytest.mark.parametrize("opacity", [0.006, 0.05, 0.7])
def test_images_do_not_depend_on_the_reach(width, height, opacity):
    scene, rig = patches(opacity), view(width, height)
    roomy, backend = render_service([(0, scene)], rig, [0], max_intersections=4_000_000, max_visible_records=20_000)
    lengths = backend.workspace["tile_ends"] - backend.workspace["tile_starts"]
    assert int(lengths.max()) > 8192 or lengths.numel() > 1280  # past the span, where the reach is used
    tight, _ = render_service([(0, scene)], rig, [0], max_intersections=400_000, max_visible_records=20_000)
    for name in roomy:
        np.testing.assert_array_equal(roomy[name], tight[name], err_msg=name)
    compare_images(roomy, render_oracle([(0, scene)], rig, [0]))


def test_uneven_resolutions():
    scene = patches(0.05)
    dev = device()
    specs = [CameraSpec(0, 333, 251), CameraSpec(0, 160, 120), CameraSpec(0, 401, 303)]  # 910 tiles
    views = torch.eye(4, device=dev).repeat(3, 1, 1)
    intrinsics = torch.cat([synthetic.pinhole(1, s.width, s.height, float(s.width)) for s in specs]).to(dev)
    renderer = BatchedRenderer(device=dev, ordering="global")
    renderer.register_scene(0, **scene.to(dev).as_kwargs())
    renderer.plan(specs, visible_capacity=60_000, intersection_capacity=4_000_000)
    renderer.set_cameras(views, intrinsics)
    out = {name: tensor.clone() for name, tensor in renderer.render().items()}
    offset = 0
    for spec in specs:
        single, _ = render_service([(0, scene)], view(spec.width, spec.height), [0], max_intersections=400_000,
                                   max_visible_records=20_000)
        for name, tensor in single.items():
            rows = out[name][offset:offset + spec.width * spec.height].cpu().numpy()
            np.testing.assert_array_equal(rows.reshape(tensor.shape), tensor, err_msg=name)
        offset += spec.width * spec.height


@pytest.mark.parametrize("opacity", [0.02, 0.6])
def test_training_slots(opacity):
    scene, rig = patches(opacity), view(512, 480)  # 960 tiles
    dev = device()
    results = []
    for per_visible in (200.0, 25.0):
        renderer = DifferentiableRenderer(height=480, width=512, device=dev, visible_capacity=20_000,
                                          intersections_per_visible=per_visible)
        means, quats = scene.means.to(dev).requires_grad_(), scene.rotations.to(dev)
        out = renderer.render(means, torch.log(scene.scales).to(dev), quats, torch.logit(scene.opacities).to(dev),
                              scene.features.to(dev), rig.viewmats.to(dev), rig.intrinsics.to(dev), sh_degree=0)
        (out["rgb"].sum() + out["alpha"].sum()).backward()
        results.append((*(out[name].detach() for name in ("rgb", "depth", "alpha", "semantic_id")), means.grad))
        assert int(renderer.intersection_capacity) == int(20_000 * per_visible)
    for a, b in zip(*results):
        assert torch.equal(a, b)

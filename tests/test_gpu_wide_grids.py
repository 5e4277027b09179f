"""More workgroups than one dispatch holds (2^32 threads; gfx950): batches of single-pixel cameras just
past the limit of the compositors' grids.  Every camera sees the same, so every pixel is that of a render
of one camera.
"""

from __future__ import annotations

import pytest
import torch

from vgr_amd import native

pytestmark = pytest.mark.gpu


def render_pixels(cameras: int, *, ray: bool, **options) -> list[torch.Tensor]:
    dev = torch.device("cuda", 0)
    module = native.load_native_module()
    scene = [torch.tensor([[0.1, -0.2, 4.0]], device=dev), torch.tensor([[0.5, 0.0, 0.0, 0.4, 0.0, 0.3]], device=dev),
             torch.tensor([0.6], device=dev), torch.tensor([[0.2, 0.5, 0.9]], device=dev),
             torch.tensor([7], dtype=torch.int64, device=dev), torch.zeros(1, dtype=torch.int64, device=dev),
             torch.tensor([0, 1], dtype=torch.int64, device=dev)]
    views = torch.eye(4, device=dev).repeat(cameras, 1, 1)
    intrinsics = torch.tensor([[1.0, 0.0, 0.5], [0.0, 1.0, 0.5], [0.0, 0.0, 1.0]], device=dev).repeat(cameras, 1, 1)
    camera_list = [views, intrinsics, views.clone(), torch.zeros(cameras, dtype=torch.int64, device=dev),
                   torch.empty(0, dtype=torch.int64, device=dev)]
    outputs = [torch.full((cameras, 1, 1, 3), 9.0, device=dev), torch.full((cameras, 1, 1, 1), 9.0, device=dev),
               torch.full((cameras, 1, 1, 1), 9.0, device=dev),
               torch.full((cameras, 1, 1, 1), 9, dtype=torch.int64, device=dev)]
    scratch = module.scratch_bytes(max_views=cameras, height=1, width=1, gaussians=1, intersection_capacity=cameras,
                                   tile_size=16, near_plane=0.01, far_plane=100.0)
    workspace = [torch.empty((cameras, native.RECORD_FLOATS), device=dev),
                 *(torch.empty(cameras, dtype=torch.uint64, device=dev) for _ in range(2)),
                 *(torch.empty(cameras, dtype=torch.int32, device=dev) for _ in range(2)),
                 *(torch.empty(cameras, dtype=torch.int32, device=dev) for _ in range(2)),
                 torch.zeros(native.COUNTER_SLOTS, dtype=torch.int64, device=dev),
                 torch.empty(scratch, dtype=torch.uint8, device=dev)]
    extra = {"ray_records": torch.empty((cameras, native.RAY_RECORD_FLOATS), device=dev)} if ray else {}
    module.render(scene, camera_list, outputs, workspace, 1, 1, 1, 0.01, 100.0, 3.33, 0.3, False, 0.01, ray, 16, 4096,
                  64, False, False, False, False, True, True, False, **extra, **options)
    torch.cuda.synchronize()
    assert int(workspace[7][1]) == cameras and int(workspace[7][5]) == 0
    return outputs


@pytest.mark.parametrize("ray,cameras", [(False, (1 << 24) + 33), (True, (1 << 22) + 33)])
def test_every_camera_of_a_batch_past_one_dispatch_is_rendered(ray, cameras):
    # 2^24 workgroups of 256 threads; with exact rays a 32x32 bin takes four.
    options = {} if ray else {"persistent_composite": 1280}
    expected = render_pixels(1, ray=ray)
    assert 0.1 < float(expected[2]) < 0.9
    for name, got, want in zip(("rgb", "depth", "alpha", "semantic_id"),
                               render_pixels(cameras, ray=ray, **options), expected):
        assert bool((got == want).all()), name
    torch.cuda.empty_cache()

"""Depth order inside every tile (gfx950), at the sizes where the tile sort changes its way:
list lengths around a wave and its share of the LDS, one bin per thread, the LDS capacities (512, 2048 and 8192 entries)
and the lists spread over depth bins in global memory; depths spread, all equal, half equal, and
in a few float steps beside one far outlier.

Every list must hold each of its records once, in strictly ascending (depth bits, Gaussian ID)
order, with the keys of those records.
"""

from __future__ import annotations

import numpy as np
import pytest
import torch

from vgr_amd import CustomHipBackend, RendererService, native, synthetic
from vgr_amd.batched import BatchedRenderer, CameraSpec

pytestmark = pytest.mark.gpu

DEPTHS = ("spread", "equal", "half", "steps")


def column_scene(count: int, depths: str, seed: int = 5) -> synthetic.SyntheticScene:
    """``count`` small Gaussians in front of an identity camera, near its axis."""
    rng = np.random.default_rng(seed)
    z = rng.uniform(4.0, 8.0, count)
    if depths == "equal":
        z[:] = 5.0
    elif depths == "half":
        z[rng.permutation(count)[: count // 2]] = 5.0
    elif depths == "steps":
        # 64 consecutive floats, and one far Gaussian that stretches the range of the depths.
        z = (np.float32(2.0).view(np.int32) + rng.integers(0, 64, count)).astype(np.int32).view(np.float32)
        z = z.astype(np.float64)
        z[0] = 50.0
    xy = rng.uniform(-0.2, 0.2, (count, 2)) * z[:, None]
    means = torch.tensor(np.concatenate([xy, z[:, None]], axis=1), dtype=torch.float32)
    return synthetic.SyntheticScene(
        means, torch.full((count, 3), 0.05), torch.tensor([1.0, 0.0, 0.0, 0.0]).repeat(count, 1),
        torch.full((count,), 0.3), torch.rand((count, 3), generator=torch.Generator().manual_seed(seed)),
        torch.arange(count, dtype=torch.int64))


def identity_rig(size: int):
    intrinsics = synthetic.pinhole(1, size, size, float(size))
    return torch.eye(4).unsqueeze(0).contiguous(), intrinsics


def check_lists(backend) -> int:
    counters = backend.read_counters()
    assert not counters["sort_lookback_failures"] and not counters["intersection_overflow"]
    ws = backend.workspace
    total = counters["tile_intersections"]
    starts, ends = ws["tile_starts"].cpu().numpy(), ws["tile_ends"].cpu().numpy()
    keys = ws["keys_out"][:total].cpu().numpy()
    values = ws["values_out"][:total].cpu().numpy()
    depth_bits = ws["visible_depths"].cpu().numpy().view(np.uint32)
    ids = ws["visible_gaussian_ids"].cpu().numpy()
    covered, longest = 0, 0
    for tile in np.flatnonzero(ends > starts):
        part = values[starts[tile]:ends[tile]]
        bits, part_ids = depth_bits[part].astype(np.uint64), ids[part].astype(np.int64)
        np.testing.assert_array_equal(keys[starts[tile]:ends[tile]], (np.uint64(tile) << np.uint64(32)) | bits)
        step = np.diff(bits.astype(np.int64))
        assert np.all((step > 0) | ((step == 0) & (np.diff(part_ids) > 0)))
        assert np.unique(part).size == part.size
        covered += part.size
        longest = max(longest, part.size)
    assert covered == total
    return longest


def render(scene, size: int, **knobs):
    dev = torch.device("cuda", 0)
    backend = CustomHipBackend(output_srgb=False, **knobs)
    service = RendererService(backend, height=size, width=size, max_views=1)
    service.initialize(stage=None, device=dev)
    service.load_scene(0, **scene.to(dev).as_kwargs())
    viewmats, intrinsics = identity_rig(size)
    out = service.render(viewmats.to(dev), intrinsics.to(dev), torch.zeros(1, dtype=torch.int64, device=dev))
    service.synchronize()
    return backend, out


@pytest.mark.parametrize("depths", DEPTHS)
@pytest.mark.parametrize("count", [1, 2, 64, 255, 257, 2047, 2048, 2049, 8191, 8192, 8193, 30_000])
def test_one_tile_lists(count, depths):
    backend, _ = render(column_scene(count, depths), 16)
    assert check_lists(backend) == count  # every Gaussian is in the image's one tile


@pytest.mark.parametrize("depths", DEPTHS)
@pytest.mark.parametrize("count", [63, 512, 513, 3000])
def test_one_pixel_lists(count, depths):
    scene = column_scene(count, depths)
    scene.scales = torch.full_like(scene.scales, 4.0)  # wide enough to reach every pixel
    backend, _ = render(scene, 4, tile_size=1, deterministic=True)
    assert check_lists(backend) == count


@pytest.mark.parametrize("depths", DEPTHS)
@pytest.mark.parametrize("counts", [(0, 1, 512, 513), (2048, 300, 2049, 64), (400, 0, 0, 8193), (257, 256, 9000, 1)])
def test_neighbouring_small_tiles_of_different_lengths(counts, depths):
    """Four neighbouring 4x4 tiles share a workgroup: each wave's own list, then the longer and the
    crowded ones together.  Sixteen tiles, every list in its own order of lengths."""
    size, tiles = 16, 16
    counts = np.array(counts * 4)
    scene = column_scene(int(counts.sum()), depths)
    tile = np.random.default_rng(1).permutation(np.repeat(np.arange(tiles), counts))
    z = scene.means[:, 2].numpy().astype(np.float64)
    centre = np.stack([tile % 4, tile // 4], axis=1) * 4.0 + 2.0
    scene.means[:, :2] = torch.tensor((centre - size / 2) * z[:, None] / size, dtype=torch.float32)
    scene.scales = torch.full_like(scene.scales, 1.0e-4)
    scene.opacities = torch.full_like(scene.opacities, 0.006)  # reaches one pixel
    backend, _ = render(scene, size, tile_size=4)
    check_lists(backend)
    lengths = (backend.workspace["tile_ends"] - backend.workspace["tile_starts"]).cpu().numpy()
    np.testing.assert_array_equal(lengths[:tiles], counts)


@pytest.mark.parametrize("depths", ["equal", "half", "steps"])
@pytest.mark.parametrize("count", [300, 2500, 9000])
def test_ties_of_a_spatially_ordered_scene(count, depths):
    """Records of a Morton-ordered scene are not in Gaussian order: ties go by the record's ID."""
    dev = torch.device("cuda", 0)
    renderer = BatchedRenderer(device=dev, ordering="global")
    renderer.register_scene(0, **column_scene(count, depths).to(dev).as_kwargs())
    renderer.plan([CameraSpec(0, 16, 16)])
    viewmats, intrinsics = identity_rig(16)
    renderer.calibrate(viewmats.to(dev), intrinsics.to(dev))
    out = {name: tensor.clone() for name, tensor in renderer.render().items()}
    plain = renderer.render_plain()[0]["outputs"]
    torch.cuda.synchronize()
    for name, tensor in out.items():
        assert torch.equal(tensor.view(plain[name].shape), plain[name]), name


def sorted_list(scene, size: int, *, capacity: int, gaussian_ids=None, near: float = 0.01, far: float = 100.0,
                sort_digit_bits: int = 0):
    """One identity camera through the native entry point; (keys, values, records) of its lists."""
    dev = torch.device("cuda", 0)
    module = native.load_native_module()
    scene = scene.to(dev)
    count = scene.count
    covariances = torch.empty((count, 6), device=dev)
    module.precompute_covariances(scene.scales, scene.rotations, covariances)
    viewmats, intrinsics = identity_rig(size)
    tiles = ((size + 15) // 16) ** 2
    outputs = [torch.empty((1, size, size, 3), device=dev), torch.empty((1, size, size, 1), device=dev),
               torch.empty((1, size, size, 1), device=dev), torch.empty((1, size, size, 1), dtype=torch.int64, device=dev)]
    scratch = module.scratch_bytes(max_views=1, height=size, width=size, gaussians=count,
                                   intersection_capacity=capacity, tile_size=16, near_plane=near, far_plane=far,
                                   sort_digit_bits=sort_digit_bits)
    keys = [torch.zeros(capacity, dtype=torch.uint64, device=dev) for _ in range(2)]
    values = [torch.full((capacity,), -1, dtype=torch.int32, device=dev) for _ in range(2)]
    records = torch.empty((count, native.RECORD_FLOATS), device=dev)
    counters = torch.zeros(native.COUNTER_SLOTS, dtype=torch.int64, device=dev)
    workspace = [records, *keys, *values, torch.empty(tiles, dtype=torch.int32, device=dev),
                 torch.empty(tiles, dtype=torch.int32, device=dev), counters,
                 torch.empty(scratch, dtype=torch.uint8, device=dev)]
    selector = module.render(
        [scene.means, covariances, scene.opacities, scene.features, scene.semantic_ids,
         torch.zeros(1, dtype=torch.int64, device=dev), torch.tensor([0, count], dtype=torch.int64, device=dev)],
        [viewmats.to(dev), intrinsics.to(dev), torch.eye(4, device=dev).unsqueeze(0).contiguous(),
         torch.zeros(1, dtype=torch.int64, device=dev), torch.empty(0, dtype=torch.int64, device=dev)],
        outputs, workspace, size, size, count, near, far, 3.33, 0.3, False, 0.01, False, 16, 4096, 64, False, False, False,
        False, True, True, False, gaussian_ids=None if gaussian_ids is None else gaussian_ids.to(dev),
        sort_digit_bits=sort_digit_bits)
    torch.cuda.synchronize()
    total = int(counters[1])
    assert int(counters[3]) == 0 and int(counters[5]) == 0
    return keys[selector][:total].cpu().numpy(), values[selector][:total].cpu().numpy(), records.cpu().numpy()


@pytest.mark.parametrize("distinct_ids", [1, 3])
@pytest.mark.parametrize("around", [0, 2000])
def test_more_equal_depths_and_ids_than_the_lds_holds(around, distinct_ids):
    """Nothing tells these entries apart but the record: 10,000 at each of two neighbouring depths, alone
    (crowded in the first spread's result) or with others around (crowded in the second's)."""
    crowd = 10_000
    scene = column_scene(2 * crowd + around, "spread")
    rng = np.random.default_rng(9)
    z = rng.uniform(2.0, 2.1, 2 * crowd + around).astype(np.float32)
    z[:crowd] = np.float32(2.0)
    z[crowd:2 * crowd] = np.nextafter(np.float32(2.0), np.float32(3.0))
    order = rng.permutation(z.size)
    scene.means = torch.tensor(np.stack([0.01 * rng.uniform(-1, 1, z.size), 0.01 * rng.uniform(-1, 1, z.size),
                                         z[order]], axis=1), dtype=torch.float32)
    ids = torch.arange(z.size, dtype=torch.int32) % distinct_ids
    keys, values, records = sorted_list(scene, 16, capacity=z.size, gaussian_ids=ids)
    assert keys.size == z.size and np.unique(values).size == z.size
    listed = records[values]
    np.testing.assert_array_equal(keys.astype(np.uint32), listed[:, 6].view(np.uint32))  # depth bits
    record_ids = listed[:, 10].view(np.int32).astype(np.int64)
    tie = record_ids * (1 << 32) + values
    step = np.diff(keys.astype(np.int64))
    assert np.all((step > 0) | ((step == 0) & (np.diff(tie) > 0)))


@pytest.mark.parametrize("depths", ["equal", "mixed"])
def test_more_crowded_lists_than_queue_places(depths):
    """Four-bit digits over a 20-bit key leave 19 places per sort tile of 8192 entries; 256 tiles with 300
    entries at one or two depths each, and one with 20,000 over the whole depth range, want more."""
    size, per_tile, extra = 256, 300, 20_000
    rng = np.random.default_rng(3)
    near, far = np.float32(4.0), np.float32(4.001)
    tile = np.concatenate([np.repeat(np.arange(256), per_tile), np.full(extra, 77)])
    z = np.full(tile.size, np.float32(4.0005), dtype=np.float32)
    if depths == "mixed":
        z[rng.permutation(256 * per_tile)[:5000]] = np.float32(4.0002)
    z[256 * per_tile:] = rng.uniform(4.0001, 4.0009, extra).astype(np.float32)
    order = rng.permutation(tile.size)
    tile, z = tile[order], z[order]
    centre = np.stack([tile % 16, tile // 16], axis=1) * 16.0 + 8.0
    xy = (centre - size / 2) * z[:, None].astype(np.float64) / size
    scene = column_scene(tile.size, "spread")
    scene.means = torch.tensor(np.concatenate([xy, z[:, None]], axis=1), dtype=torch.float32)
    scene.scales = torch.full_like(scene.scales, 0.001)
    keys, values, records = sorted_list(scene, size, capacity=tile.size, near=float(near), far=float(far),
                                        sort_digit_bits=4)
    assert keys.size == tile.size and np.unique(values).size == tile.size
    listed = records[values]
    np.testing.assert_array_equal((keys >> np.uint64(32)).astype(np.int64), tile[listed[:, 10].view(np.int32)])
    np.testing.assert_array_equal(keys.astype(np.uint32), listed[:, 6].view(np.uint32))  # depth bits
    step = np.diff(keys.astype(np.int64))
    assert np.all((step > 0) | ((step == 0) & (np.diff(values) > 0)))


@pytest.mark.parametrize("copies", [2, 40])
@pytest.mark.parametrize("count,depths", [(1, "equal"), (200, "equal"), (200, "steps"), (5000, "equal"), (5000, "spread")])
def test_a_camera_active_more_than_once(count, depths, copies):
    """Its lists hold every Gaussian once per copy: longer than the scene, sorted all the same."""
    dev = torch.device("cuda", 0)
    backend = CustomHipBackend(output_srgb=False, max_visible_records=count * copies,
                               max_intersections=count * copies)
    service = RendererService(backend, height=16, width=16, max_views=copies)
    service.initialize(stage=None, device=dev)
    service.load_scene(0, **column_scene(count, depths).to(dev).as_kwargs())
    viewmats, intrinsics = identity_rig(16)
    service.render(viewmats.to(dev).repeat(copies, 1, 1), intrinsics.to(dev).repeat(copies, 1, 1),
                   torch.zeros(copies, dtype=torch.int64, device=dev),
                   active_camera_ids=torch.ones(copies, dtype=torch.int64, device=dev))
    service.synchronize()
    counters = backend.read_counters()
    assert counters["tile_intersections"] == count * copies and not counters["intersection_overflow"]
    keys = backend.workspace["keys_out"][: count * copies].cpu().numpy()
    values = backend.workspace["values_out"][: count * copies].cpu().numpy()
    depth_bits = backend.workspace["visible_depths"].cpu().numpy().view(np.uint32)
    assert np.unique(values).size == values.size
    np.testing.assert_array_equal(keys, (np.uint64(1) << np.uint64(32)) | depth_bits[values].astype(np.uint64))
    step = np.diff(keys.astype(np.int64))
    assert np.all((step > 0) | ((step == 0) & (np.diff(values) > 0)))

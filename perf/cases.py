"""Performance cases of the renderer: what its users have it do, through the public entry points.

Every case is a dict of plain values.  ``kind`` selects the entry point:

* ``service``  - ``RendererService.render`` over ``CustomHipBackend`` (the simulator's camera loop);
* ``batched``  - ``BatchedRenderer.render`` as a captured graph (robot fleets, mixed resolutions);
* ``pose``     - ``BatchedRenderer.render_pose`` + backward to 6-DoF twists (camera tracking);
* ``train``    - ``DifferentiableRenderer.render`` + backward to every scene parameter and the pose.

Scenes and cameras follow the distributions of the package's synthetic workloads: an open cloud
("normal", cameras on an orbit looking at it) and a closed room ("room", cameras moving inside).
"""

from __future__ import annotations

import math
import os
import random
import sys
from typing import Any

import torch

_PACKAGE = os.path.join(os.getcwd(), "vectorized-gaussian-renderer-public_amd")
if _PACKAGE not in sys.path:
    sys.path.insert(0, _PACKAGE)

from vgr_amd import CustomHipBackend, RendererService, synthetic  # noqa: E402
from vgr_amd.autograd import DifferentiableRenderer, compose_pose  # noqa: E402
from vgr_amd.batched import BatchedRenderer, CameraSpec  # noqa: E402

DEVICE = "cuda:0"


def _case(name: str | None, kind: str, **fields: Any) -> dict[str, Any]:
    case = {"kind": kind, "cameras": 1, "width": 640, "height": 480, "gaussians": 100_000, "scenes": 1, "sh": 0,
            "layout": "normal", "tile": 16, "full": True, "antialiased": False, "srgb": False, "ray": False,
            "deterministic": False, "physical": 0, "uneven": False}
    case.update(fields)
    if name is not None:
        case["name"] = name
    return case


def listed() -> list[dict[str, Any]]:
    return [
        # One low-resolution preview camera over a small scene: the latency of a single call.
        _case("service_preview", "service", width=128, height=96, gaussians=20_000, sh=1),
        # One VGA sensor over a 100k-Gaussian scene, all outputs: a simulator's single camera.
        _case("service_vga", "service", gaussians=100_000),
        # A few odd-sized display views of two scenes, RGB only, antialiased, sRGB, 8x8 tiles.
        _case("service_ragged_rgb", "service", cameras=6, width=333, height=251, gaussians=150_000, scenes=2, sh=2,
              tile=8, full=False, antialiased=True, srgb=True),
        # The headline batch: 64 VGA sensors around a million SH3 Gaussians, all outputs.
        _case("service_orbit64", "service", cameras=64, gaussians=1_000_000, sh=3, deterministic=True),
        # A logical batch rendered as bounded physical submissions (fixed memory), inside a room.
        _case("service_chunked_room", "service", cameras=48, width=160, height=120, gaussians=1_000_000, sh=1,
              layout="room", physical=16),
        # The dense per-pixel path with its depth cutoff inside a large room.
        _case("dense_room", "service", cameras=8, width=128, height=128, gaussians=5_000_000, sh=1, layout="room",
              tile=1),
        # Exact-ray sensors (wide-angle accuracy) over the headline scene.
        _case("ray_orbit16", "service", cameras=16, gaussians=1_000_000, sh=3, ray=True, deterministic=True),
        # The robot fleet: 1024 small cameras along trajectories in a five-million-Gaussian room.
        _case("batched_robotics", "batched", cameras=1024, width=160, height=120, gaussians=5_000_000, sh=1,
              layout="room"),
        # Cameras of four resolutions over four scenes of different sizes in one graph.
        _case("batched_uneven", "batched", cameras=256, gaussians=2_000_000, scenes=4, sh=3, uneven=True),
        # Camera tracking: pose gradients of a batch of small cameras in a room.
        _case("pose_tracking", "pose", cameras=256, width=160, height=120, gaussians=2_000_000, sh=1, layout="room"),
        # A small fit (few pixels, few Gaussians): launch and host latency of a training step.
        _case("train_small", "train", cameras=2, width=97, height=71, gaussians=5_000, sh=1),
        # The training workload: 16 views of 512x512 and 500k SH3 Gaussians.
        _case("train_step", "train", cameras=16, width=512, height=512, gaussians=500_000, sh=3),
    ]


def _log(rng: random.Random, low: float, high: float) -> int:
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def draw(rng: random.Random) -> dict[str, Any]:
    kind = rng.choice(("service", "service", "service", "dense", "ray", "batched", "pose", "train", "train"))
    if kind == "service":
        case = _case(None, "service", cameras=_log(rng, 1, 64), width=_log(rng, 64, 640), height=_log(rng, 48, 480),
                     gaussians=_log(rng, 5_000, 1_000_000), scenes=rng.choice((1, 1, 2)), sh=rng.randint(0, 3),
                     tile=rng.choice((8, 16, 16)), full=rng.random() < 0.75, antialiased=rng.random() < 0.3,
                     srgb=rng.random() < 0.3, deterministic=rng.random() < 0.5)
        if rng.random() < 0.3:
            case.update(layout="room", scenes=1, cameras=min(case["cameras"], 32), width=min(case["width"], 320),
                        height=min(case["height"], 240))
        return case
    if kind == "dense":
        return _case(None, "service", cameras=rng.randint(1, 8), width=rng.randint(48, 160),
                     height=rng.randint(48, 160), gaussians=_log(rng, 20_000, 5_000_000), sh=rng.randint(0, 1),
                     layout=rng.choice(("room", "normal")), tile=rng.choice((1, 1, 2, 4)),
                     deterministic=rng.random() < 0.3)
    if kind == "ray":
        return _case(None, "service", cameras=_log(rng, 1, 16), width=_log(rng, 96, 640), height=_log(rng, 64, 480),
                     gaussians=_log(rng, 20_000, 1_000_000), sh=rng.randint(0, 3), ray=True, deterministic=True,
                     tile=rng.choice((8, 16)))
    if kind == "batched":
        if rng.random() < 0.3:
            return _case(None, "batched", cameras=_log(rng, 16, 256), gaussians=_log(rng, 200_000, 2_000_000),
                         scenes=rng.randint(1, 4), sh=rng.randint(0, 3), uneven=True)
        return _case(None, "batched", cameras=_log(rng, 16, 1024), width=rng.randint(96, 200),
                     height=rng.randint(64, 120), gaussians=_log(rng, 100_000, 2_500_000), sh=rng.randint(0, 2),
                     layout="room")
    if kind == "pose":
        return _case(None, "pose", cameras=_log(rng, 8, 256), width=rng.randint(64, 160), height=rng.randint(48, 120),
                     gaussians=_log(rng, 50_000, 2_000_000), sh=rng.randint(0, 2), layout="room")
    return _case(None, "train", cameras=rng.randint(1, 16), width=_log(rng, 64, 512), height=_log(rng, 64, 512),
                 gaussians=_log(rng, 2_000, 500_000), sh=rng.randint(0, 3), tile=rng.choice((8, 16, 16)),
                 antialiased=rng.random() < 0.3)


# ------------------------------------------------------------------------------------- inputs
def _scene(count: int, seed: int, sh: int, layout: str) -> dict[str, torch.Tensor]:
    """The package's synthetic scene distributions, generated on the GPU."""
    g = torch.Generator(device=DEVICE).manual_seed(seed)

    def normal(*shape):
        return torch.randn(shape, generator=g, device=DEVICE)

    def uniform(*shape):
        return torch.rand(shape, generator=g, device=DEVICE)

    if layout == "room":
        # 70 % inside [-10,10]^2 x [0,4], 30 % on the walls with 2 cm of jitter.
        interior = int(round(0.7 * count))
        walls = count - interior
        low = torch.tensor([-10.0, -10.0, 0.0], device=DEVICE)
        span = torch.tensor([20.0, 20.0, 4.0], device=DEVICE)
        inside = low + span * uniform(interior, 3)
        side = torch.randint(0, 4, (walls,), generator=g, device=DEVICE)
        along, height = 20.0 * uniform(walls) - 10.0, 4.0 * uniform(walls)
        plane = torch.where(side % 2 == 0, 10.0, -10.0) + 0.02 * normal(walls)
        on_x = side < 2
        means = torch.cat((inside, torch.stack((torch.where(on_x, plane, along), torch.where(on_x, along, plane),
                                                height), dim=1)))
    else:
        means = 3.0 * normal(count, 3)
    quats = torch.nn.functional.normalize(normal(count, 4), dim=-1)
    features = 0.1 * normal(count, 3 * (sh + 1) ** 2)
    features[:, :3] = uniform(count, 3)
    return {"means": means.contiguous(), "scales": torch.exp(-4.0 + 0.5 * normal(count, 3)),
            "rotations": torch.where(quats[:, :1] < 0, -quats, quats).contiguous(),
            "opacities": torch.sigmoid(1.5 * normal(count)), "features": features.contiguous(),
            "semantic_ids": torch.randint(0, 64, (count,), generator=g, device=DEVICE)}


def _resolutions(case: dict[str, Any]) -> list[tuple[int, int]]:
    if not case["uneven"]:
        return [(case["width"], case["height"])] * case["cameras"]
    choice = random.Random(case["cameras"])
    return [choice.choice(((128, 128), (320, 240), (640, 480), (1280, 720))) for _ in range(case["cameras"])]


def _cameras(case: dict[str, Any], seed: int) -> tuple[torch.Tensor, torch.Tensor]:
    """World->camera matrices and intrinsics; about 60 degrees of horizontal field of view."""
    count = case["cameras"]
    resolutions = _resolutions(case)
    intrinsics = torch.cat([synthetic.pinhole(1, w, h, 0.866 * w) for w, h in resolutions])
    if case["layout"] == "room":
        samples = min(count, 32)
        rig = synthetic.trajectory_rig(-(-count // samples), samples, 1, 1, 1.0, seed=seed)
    else:
        rig = synthetic.orbit_rig(count, 1, 1, 1.0, seed=seed, radius=(10.0, 15.0))
    return rig.viewmats[:count].contiguous().to(DEVICE), intrinsics.to(DEVICE)


def _scene_sizes(case: dict[str, Any]) -> list[int]:
    if case["uneven"]:
        return [max(1, case["gaussians"] * (k + 1) // case["scenes"]) for k in range(case["scenes"])]
    return [case["gaussians"]] * case["scenes"]


def _inputs(case: dict[str, Any], seed: int):
    scenes = [_scene(count, seed * 1009 + k, case["sh"], case["layout"]) for k, count in enumerate(_scene_sizes(case))]
    viewmats, intrinsics = _cameras(case, seed)
    ids = torch.arange(case["cameras"], device=DEVICE) % case["scenes"]
    return scenes, viewmats, intrinsics, ids


def _training_inputs(case: dict[str, Any], seed: int):
    scenes, viewmats, intrinsics, _ = _inputs(case, seed)
    scene = scenes[0]
    leaves = {"means": scene["means"], "log_scales": torch.log(scene["scales"]), "quats": scene["rotations"],
              "opacity_logits": torch.logit(scene["opacities"], eps=1e-6), "features": scene["features"]}
    g = torch.Generator(device=DEVICE).manual_seed(seed + 1)
    shape = (case["cameras"], case["height"], case["width"])
    photo = torch.rand((*shape, 3), generator=g, device=DEVICE)
    distance = 8.0 + 8.0 * torch.rand((*shape, 1), generator=g, device=DEVICE)
    return leaves, viewmats, intrinsics, photo, distance


def _training_loss(rgb, depth, photo, distance):
    """L1 colour plus L1 depth where something was hit."""
    hit = torch.isfinite(depth)
    return (rgb - photo).abs().mean() + 0.05 * (torch.where(hit, depth, distance) - distance).abs().mean()


def _pose_loss(rgb, alpha, photo):
    return (rgb - photo).abs().mean() + alpha.mean()


def _pose_photo(case: dict[str, Any], seed: int) -> torch.Tensor:
    g = torch.Generator(device=DEVICE).manual_seed(seed + 1)
    return torch.rand((case["cameras"] * case["width"] * case["height"], 3), generator=g, device=DEVICE)


# ---------------------------------------------------------------------------- prepare and run
def prepare(case: dict[str, Any], seed: int) -> dict[str, Any]:
    state: dict[str, Any] = {"kind": case["kind"]}
    if case["kind"] == "train":
        leaves, viewmats, intrinsics, photo, distance = _training_inputs(case, seed)
        renderer = DifferentiableRenderer(height=case["height"], width=case["width"], device=DEVICE,
                                          tile_size=case["tile"],
                                          rasterize_mode="antialiased" if case["antialiased"] else "classic")
        with torch.no_grad():  # sizes the buffers
            renderer.render(*leaves.values(), viewmats, intrinsics)
        state.update(renderer=renderer, viewmats=viewmats, intrinsics=intrinsics, photo=photo, distance=distance,
                     leaves={name: value.requires_grad_(True) for name, value in leaves.items()},
                     twist=torch.zeros((case["cameras"], 6), device=DEVICE, requires_grad=True))
        return state
    scenes, viewmats, intrinsics, ids = _inputs(case, seed)
    state.update(viewmats=viewmats, intrinsics=intrinsics)
    if case["kind"] in ("batched", "pose"):
        renderer = BatchedRenderer(device=DEVICE, pose_gradients=case["kind"] == "pose")
        for k, scene in enumerate(scenes):
            renderer.register_scene(k, **scene)
        renderer.plan([CameraSpec(i % case["scenes"], w, h) for i, (w, h) in enumerate(_resolutions(case))])
        renderer.calibrate(viewmats, intrinsics)
        renderer.capture()
        state["renderer"] = renderer
        if case["kind"] == "pose":
            state.update(photo=_pose_photo(case, seed),
                         twist=torch.zeros((case["cameras"], 6), device=DEVICE, requires_grad=True))
        return state
    knobs: dict[str, Any] = {}
    if case["physical"]:
        knobs.update(max_physical_views=case["physical"], fixed_capacity_sort=True, adaptive_capacity=False,
                     visible_capacity_per_view=400_000, intersections_per_visible=4.0)
    backend = CustomHipBackend(tile_size=case["tile"], output_srgb=case["srgb"], deterministic=case["deterministic"],
                               rasterize_mode="antialiased" if case["antialiased"] else "classic",
                               ray_gaussian_evaluation=case["ray"], **knobs)
    outputs = ("rgb", "depth", "alpha", "semantic_id") if case["full"] else ("rgb",)
    service = RendererService(backend, height=case["height"], width=case["width"], outputs=outputs,
                              max_views=case["cameras"])
    service.initialize(stage=None, device=DEVICE)
    for k, scene in enumerate(scenes):
        service.load_scene(k, **scene)
    # The simulator writes each frame's poses into one camera tensor.
    state.update(service=service, ids=ids, camera=viewmats.clone())
    service.render(state["camera"], intrinsics, ids)  # sizes the buffers
    if case["physical"]:
        backend.check_capacity()
    return state


def run(state: dict[str, Any]) -> dict[str, Any]:
    if state["kind"] == "service":
        state["camera"].copy_(state["viewmats"])  # this frame's poses
        return state["service"].render(state["camera"], state["intrinsics"], state["ids"])
    if state["kind"] == "batched":
        return state["renderer"].render(state["viewmats"], state["intrinsics"])
    twist = state["twist"]
    twist.grad = None
    views = compose_pose(twist, state["viewmats"])
    if state["kind"] == "pose":
        renderer = state["renderer"]
        renderer.set_cameras(state["viewmats"], state["intrinsics"])
        rgb, depth, alpha = renderer.render_pose(views)
        _pose_loss(rgb, alpha, state["photo"]).backward()
        return {"rgb": rgb.detach(), "depth": depth.detach(), "alpha": alpha.detach(), "twist": twist.grad}
    leaves = state["leaves"]
    for leaf in leaves.values():
        leaf.grad = None
    out = state["renderer"].render(*leaves.values(), views, state["intrinsics"])
    loss = _training_loss(out["rgb"], out["depth"], state["photo"], state["distance"])
    loss.backward()
    return {"loss": loss.detach(), "rgb": out["rgb"].detach(), "depth": out["depth"].detach(),
            "alpha": out["alpha"].detach(), "semantic_id": out["semantic_id"], "twist": twist.grad,
            **{name: leaf.grad for name, leaf in leaves.items()}}


def work(case: dict[str, Any]) -> dict[str, float]:
    """Scene and cameras read once, outputs written once; about 60 operations per (camera, Gaussian)
    pair and 20 per (pixel, Gaussian) evaluation, of which a pixel needs a few hundred at most."""
    channels = 3 * (case["sh"] + 1) ** 2
    sizes = _scene_sizes(case)
    pixels = sum(w * h for w, h in _resolutions(case))
    # A row: mean 3, scales 3, quaternion 4, opacity 1, channels and an int64 label.
    scene_bytes = sum(sizes) * (4 * (11 + channels) + 8)
    out_bytes = 12 if not case["full"] else 28
    pairs = case["cameras"] * sum(sizes) / len(sizes)
    evaluations = pixels * min(300.0, 20.0 + sum(sizes) / len(sizes) / 4000.0)
    total = {"bytes": scene_bytes + case["cameras"] * 100 + pixels * out_bytes,
             "flops": 60.0 * pairs + 20.0 * evaluations}
    if case["kind"] in ("train", "pose"):
        total["bytes"] += pixels * 24 + (scene_bytes if case["kind"] == "train" else 0)
        total["flops"] *= 3.0
    return total


# --------------------------------------------------------------------- the same in 64 bits
_THRESHOLD, _STOP, _SIGMA, _DILATION, _NEAR, _FAR = 1.0 / 255.0, 1.0e-4, 3.33, 0.3, 0.01, 100.0
_BLOCK = 32


def _basis64(d: torch.Tensor, degree: int) -> torch.Tensor:
    """Real spherical harmonics of bands 1..degree at unit directions (Condon-Shortley signs)."""
    x, y, z = d.unbind(-1)
    rows = []
    if degree >= 1:
        c = math.sqrt(3.0 / (4.0 * math.pi))
        rows += [-c * y, c * z, -c * x]
    if degree >= 2:
        c, c0 = math.sqrt(15.0 / (4.0 * math.pi)), math.sqrt(5.0 / (16.0 * math.pi))
        rows += [c * x * y, -c * y * z, c0 * (2 * z * z - x * x - y * y), -c * x * z, 0.5 * c * (x * x - y * y)]
    if degree >= 3:
        c3, c2 = math.sqrt(35.0 / (32.0 * math.pi)), math.sqrt(105.0 / (4.0 * math.pi))
        c1, c0 = math.sqrt(21.0 / (32.0 * math.pi)), math.sqrt(7.0 / (16.0 * math.pi))
        rows += [-c3 * y * (3 * x * x - y * y), c2 * x * y * z, -c1 * y * (4 * z * z - x * x - y * y),
                 c0 * z * (2 * z * z - 3 * x * x - 3 * y * y), -c1 * x * (4 * z * z - x * x - y * y),
                 0.5 * c2 * z * (x * x - y * y), -c3 * x * (x * x - 3 * y * y)]
    return torch.stack(rows, dim=-1)


def _splats64(scene: dict[str, torch.Tensor], view, k, w: int, h: int, case: dict[str, Any]):
    """One camera's visible splats in depth order (differentiable) and their pixel boxes."""
    fx, fy, cx, cy = k[0, 0], k[1, 1], k[0, 2], k[1, 2]
    rotation, shift = view[:3, :3], view[:3, 3]
    with torch.no_grad():
        z = scene["means"] @ rotation[2] + shift[2]
        keep = torch.nonzero((scene["opacities"] >= _THRESHOLD) & (z >= _NEAR) & (z <= _FAR)).squeeze(1)
    means, opacity = scene["means"][keep], scene["opacities"][keep]
    x, y, z = (means @ rotation.T + shift).unbind(-1)
    a, b, c, d = torch.nn.functional.normalize(scene["rotations"][keep], dim=-1).unbind(-1)
    axes = torch.stack((1 - 2 * (c * c + d * d), 2 * (b * c - a * d), 2 * (b * d + a * c),
                        2 * (b * c + a * d), 1 - 2 * (b * b + d * d), 2 * (c * d - a * b),
                        2 * (b * d - a * c), 2 * (c * d + a * b), 1 - 2 * (b * b + c * c)), -1).view(-1, 3, 3)
    half = (rotation @ axes) * scene["scales"][keep].unsqueeze(1)
    cov = half @ half.transpose(1, 2)
    tan_x, tan_y = 0.15 * w / fx, 0.15 * h / fy
    u = torch.minimum((w - cx) / fx + tan_x, torch.maximum(-cx / fx - tan_x, x / z))
    v = torch.minimum((h - cy) / fy + tan_y, torch.maximum(-cy / fy - tan_y, y / z))
    zero = torch.zeros_like(z)
    jacobian = torch.stack((fx / z, zero, -fx * u / z, zero, fy / z, -fy * v / z), -1).view(-1, 2, 3)
    flat = jacobian @ cov @ jacobian.transpose(1, 2)
    s00, s01, s11 = flat[:, 0, 0] + _DILATION, flat[:, 0, 1], flat[:, 1, 1] + _DILATION
    det = s00 * s11 - s01 * s01
    if case["antialiased"]:
        sharp = (flat[:, 0, 0] * flat[:, 1, 1] - s01 * s01) / det
        opacity = opacity * torch.sqrt(torch.clamp(sharp, min=0.005 ** 2))
    centre_x, centre_y = fx * x / z + cx, fy * y / z + cy
    with torch.no_grad():
        reach = torch.sqrt(torch.clamp(2 * torch.log(opacity / _THRESHOLD), min=0.0)).clamp(max=_SIGMA)
        box_x, box_y = torch.ceil(reach * torch.sqrt(s00)), torch.ceil(reach * torch.sqrt(s11))
        at_x, at_y = centre_x, centre_y
    extra = None
    if case["ray"]:
        inverse = torch.linalg.inv(cov)
        point = torch.stack((x, y, z), -1)
        toward = (inverse @ point.unsqueeze(-1)).squeeze(-1)
        reach2 = (point * toward).sum(-1)
        extra = torch.cat((inverse.reshape(-1, 9), toward, reach2.unsqueeze(-1)), dim=1)
        # Screen box of the rays that pass within the support.
        cone = (reach2 - _SIGMA ** 2)[:, None, None] * inverse - toward[:, :, None] * toward[:, None, :]
        area = cone[:, 0, 0] * cone[:, 1, 1] - cone[:, 0, 1] ** 2
        mid_x = (cone[:, 0, 1] * cone[:, 1, 2] - cone[:, 1, 1] * cone[:, 0, 2]) / area
        mid_y = (cone[:, 0, 1] * cone[:, 0, 2] - cone[:, 0, 0] * cone[:, 1, 2]) / area
        level = -(cone[:, 2, 2] + cone[:, 0, 2] * mid_x + cone[:, 1, 2] * mid_y)
        bounded = (cone[:, 0, 0] > 0) & (area > 0) & (level > 0)
        at_x = torch.where(bounded, fx * mid_x + cx, w / 2)
        at_y = torch.where(bounded, fy * mid_y + cy, h / 2)
        box_x = torch.where(bounded, torch.ceil(fx * torch.sqrt(level * cone[:, 1, 1] / area)), float(max(w, h)))
        box_y = torch.where(bounded, torch.ceil(fy * torch.sqrt(level * cone[:, 0, 0] / area)), float(max(w, h)))
    with torch.no_grad():
        seen = (opacity >= _THRESHOLD) & (at_x + box_x > 0) & (at_y + box_y > 0) & (at_x - box_x < w) & \
            (at_y - box_y < h)
        index = torch.nonzero(seen).squeeze(1)
        index = index[torch.sort(z[index].float(), stable=True).indices]
        boxes = torch.stack((at_x - box_x, at_x + box_x, at_y - box_y, at_y + box_y), -1)[index]
    origin = -torch.linalg.solve(rotation, shift)
    features = scene["features"][keep][index]
    bands = (case["sh"] + 1) ** 2
    colour = features[:, :3]
    if case["sh"] > 0:
        rest = features[:, 3:3 * bands].reshape(-1, bands - 1, 3)
        toward_splat = torch.nn.functional.normalize(means[index] - origin, dim=-1)
        colour = torch.clamp(colour + (_basis64(toward_splat, case["sh"]).unsqueeze(-1) * rest).sum(1), min=0.0)
    columns = torch.cat((torch.stack((centre_x, centre_y, s11 / det, -s01 / det, s00 / det, opacity.clamp(0, 1), z),
                                     -1)[index], colour), dim=1)
    return columns, None if extra is None else extra[index], boxes


def _block64(columns, extra, px, py, k, ray: bool):
    """rgb, depth sum and transmittance of one pixel block over its depth-ordered splats."""
    transmittance, alive = torch.ones_like(px), torch.ones_like(px)
    rgb, depth = px.new_zeros((px.numel(), 3)), torch.zeros_like(px)
    for start in range(0, columns.shape[0], 4096):
        part = columns[start:start + 4096]
        if ray:
            more = extra[start:start + 4096]
            rays = torch.stack(((px - k[0, 2]) / k[0, 0], (py - k[1, 2]) / k[1, 1], torch.ones_like(px)), -1)
            outer = (rays[:, :, None] * rays[:, None, :]).reshape(-1, 9)
            distance2 = torch.clamp(more[:, 12] - (rays @ more[:, 9:12].T) ** 2 / (outer @ more[:, :9].T), min=0.0)
            alpha = torch.clamp(part[:, 5] * torch.exp(-0.5 * distance2), max=1.0)
            alpha = torch.where(distance2 <= _SIGMA ** 2, alpha, 0.0) * alive[:, None]
            # A pixel takes the splat that ends it and nothing behind it.
            after = torch.cumprod(1 - alpha, dim=1) * transmittance[:, None]
            before = torch.cat((transmittance[:, None], after[:, :-1]), dim=1)
            alpha = torch.where(before > _STOP, alpha, 0.0)
        else:
            dx, dy = px[:, None] - part[:, 0], py[:, None] - part[:, 1]
            power = -0.5 * (part[:, 2] * dx * dx + 2 * part[:, 3] * dx * dy + part[:, 4] * dy * dy)
            alpha = torch.clamp(part[:, 5] * torch.exp(power), max=0.99)
            alpha = torch.where((power <= 0) & (alpha >= _THRESHOLD), alpha, 0.0) * alive[:, None]
            # A pixel leaves out the splat that would end it and everything behind it.
            with torch.no_grad():
                going = torch.cumprod(1 - alpha, dim=1) * transmittance[:, None] > _STOP
                alive = alive * going[:, -1]
            alpha = torch.where(going, alpha, 0.0)
        after = torch.cumprod(1 - alpha, dim=1) * transmittance[:, None]
        weight = alpha * torch.cat((transmittance[:, None], after[:, :-1]), dim=1)
        rgb = rgb + weight @ part[:, 7:10]
        depth = depth + weight @ part[:, 6]
        transmittance = after[:, -1]
        if ray:
            alive = alive * (transmittance.detach() > _STOP)
        if start + 4096 < columns.shape[0] and not bool(alive.any()):
            break
    return rgb, depth, transmittance


def _blocks64(columns, extra, boxes, k, w: int, h: int, ray: bool):
    """(pixel indices, rgb, depth sum, transmittance) of every block of one image."""
    for y0 in range(0, h, _BLOCK):
        row = torch.nonzero((boxes[:, 3] >= y0) & (boxes[:, 2] <= y0 + _BLOCK)).squeeze(1)
        for x0 in range(0, w, _BLOCK):
            ys = torch.arange(y0, min(h, y0 + _BLOCK), device=DEVICE)
            xs = torch.arange(x0, min(w, x0 + _BLOCK), device=DEVICE)
            py, px = torch.meshgrid(ys.double() + 0.5, xs.double() + 0.5, indexing="ij")
            hit = row[(boxes[row, 1] >= x0) & (boxes[row, 0] <= x0 + _BLOCK)]
            index = (ys[:, None] * w + xs[None, :]).reshape(-1)
            yield index, _block64(columns[hit], None if extra is None else extra[hit], px.reshape(-1), py.reshape(-1),
                                  k, ray)


def _image64(rgb, depth, transmittance, srgb: bool):
    alpha = 1 - transmittance
    depth = torch.where(alpha > 1e-8, depth / torch.clamp(alpha, min=1e-30), math.inf)
    if srgb:
        rgb = rgb.clamp(0, 1)
        rgb = torch.where(rgb <= 0.0031308, 12.92 * rgb, 1.055 * rgb ** (1 / 2.4) - 0.055)
    return rgb, depth.unsqueeze(-1), alpha.unsqueeze(-1)


def _render64(scenes, viewmats, intrinsics, ids, case):
    """Every camera's (rgb [P,3], depth [P,1], alpha [P,1])."""
    images = []
    for i, (w, h) in enumerate(_resolutions(case)):
        columns, extra, boxes = _splats64(scenes[ids[i]], viewmats[i], intrinsics[i], w, h, case)
        rgb = torch.zeros((w * h, 3), dtype=torch.float64, device=DEVICE)
        depth, transmittance = torch.zeros_like(rgb[:, 0]), torch.ones_like(rgb[:, 0])
        for index, (block_rgb, block_depth, block_t) in _blocks64(columns, extra, boxes, intrinsics[i], w, h,
                                                                  case["ray"]):
            rgb[index], depth[index], transmittance[index] = block_rgb, block_depth, block_t
        images.append(_image64(rgb, depth, transmittance, case["srgb"]))
    return images


def _gradients64(scene, viewmats, intrinsics, case, upstream):
    """Accumulates d(images)/d(scene, viewmats) against the images' upstream gradients, block by block."""
    w, h = case["width"], case["height"]
    for i in range(case["cameras"]):
        columns, _, boxes = _splats64(scene, viewmats[i], intrinsics[i], w, h, case)
        leaf = columns.detach().requires_grad_(True)
        grad_rgb, grad_depth, grad_alpha = upstream[i]
        for index, (rgb, depth, transmittance) in _blocks64(leaf, None, boxes, intrinsics[i], w, h, False):
            rgb, depth, alpha = _image64(rgb, depth, transmittance, False)
            total = (rgb * grad_rgb[index]).sum() + (alpha * grad_alpha[index]).sum()
            total = total + (torch.where(torch.isfinite(depth), depth, 0.0) * grad_depth[index]).sum()
            if total.requires_grad:
                total.backward()
        if leaf.grad is not None:
            columns.backward(leaf.grad)


def _twisted64(twist: torch.Tensor, base: torch.Tensor) -> torch.Tensor:
    """exp(twist^) @ base for twists (translation, rotation)."""
    rho, phi = twist[:, :3], twist[:, 3:]
    zero = torch.zeros_like(phi[:, 0])
    hat = torch.stack((zero, -phi[:, 2], phi[:, 1], rho[:, 0], phi[:, 2], zero, -phi[:, 0], rho[:, 1],
                       -phi[:, 1], phi[:, 0], zero, rho[:, 2], zero, zero, zero, zero), -1).view(-1, 4, 4)
    return torch.linalg.matrix_exp(hat) @ base


def exact(case: dict[str, Any], seed: int):
    blocks = sum(-(-w // _BLOCK) * -(-h // _BLOCK) for w, h in _resolutions(case))
    differentiable = case["kind"] in ("train", "pose")
    if blocks > (700 if differentiable else 5000):
        return None  # takes too long
    if case["kind"] == "train":
        leaves, viewmats, intrinsics, photo, distance = _training_inputs(case, seed)
        leaves = {name: value.double().requires_grad_(True) for name, value in leaves.items()}
        scene = {"means": leaves["means"], "scales": torch.exp(leaves["log_scales"]), "rotations": leaves["quats"],
                 "opacities": torch.sigmoid(leaves["opacity_logits"]), "features": leaves["features"]}
        scenes, ids = [scene], [0] * case["cameras"]
    else:
        scenes, viewmats, intrinsics, ids = _inputs(case, seed)
        scenes = [{name: value.double() for name, value in scene.items()} for scene in scenes]
        ids = ids.tolist()
    viewmats, intrinsics = viewmats.double(), intrinsics.double()
    twist = torch.zeros((case["cameras"], 6), dtype=torch.float64, device=DEVICE, requires_grad=differentiable)
    views = _twisted64(twist, viewmats) if differentiable else viewmats
    with torch.no_grad():
        images = _render64(scenes, views, intrinsics, ids, case)
    if case["kind"] == "batched":
        rgb, depth, alpha = (torch.cat([image[k] for image in images]) for k in range(3))
        return {"rgb": rgb, "depth": depth, "alpha": alpha, "semantic_id": None}
    w, h = case["width"], case["height"]
    rgb, depth, alpha = (torch.stack([image[k] for image in images]) for k in range(3))
    if case["kind"] == "service":
        rgb, depth, alpha = (v.view(-1, h, w, v.shape[-1]) for v in (rgb, depth, alpha))
        return {"rgb": rgb, "depth": depth, "alpha": alpha, "semantic_id": None} if case["full"] else {"rgb": rgb}
    out = [v.requires_grad_(True) for v in (rgb, depth, alpha)]
    if case["kind"] == "pose":
        loss = _pose_loss(rgb.view(-1, 3), alpha, _pose_photo(case, seed).double())
    else:
        loss = _training_loss(rgb, depth, photo.double().view(rgb.shape), distance.double().view(depth.shape))
    upstream = [torch.zeros_like(v) if g is None else g
                for v, g in zip(out, torch.autograd.grad(loss, out, allow_unused=True))]
    camera_views = views.detach().requires_grad_(True)
    if case["kind"] == "train":
        held = {name: value.detach().requires_grad_(True) for name, value in scenes[0].items()}
    else:
        held = scenes[0]
    _gradients64(held, camera_views, intrinsics, case, list(zip(*upstream)))
    views.backward(camera_views.grad)
    rgb, depth, alpha = (v.detach() for v in out)
    if case["kind"] == "pose":
        return {"rgb": rgb.reshape(-1, 3), "depth": depth.reshape(-1, 1), "alpha": alpha.reshape(-1, 1),
                "twist": twist.grad}
    for name, value in scenes[0].items():
        if value.requires_grad and value.grad_fn is not None:
            value.backward(held[name].grad)
        elif value.requires_grad:
            value.grad = held[name].grad
    shape = (case["cameras"], h, w, -1)
    return {"loss": loss.detach().reshape(()), "rgb": rgb.view(*shape[:3], 3), "depth": depth.view(*shape[:3], 1),
            "alpha": alpha.view(*shape[:3], 1), "semantic_id": None, "twist": twist.grad,
            **{name: leaf.grad for name, leaf in leaves.items()}}

"""What users of the renderer have it do, as timed cases.

A case is one frame: a scene, an image size, a compositing mode and either the forward pass alone ("view", as a
viewer draws) or forward and backward ("train", as an optimisation step runs, from the gradient of the loss with
respect to the image to the gradients of the vertices, colours and opacities).  Three kinds of scene:

  soup   independent triangles with vertices of their own, what an optimisation from scratch starts from: uniform
         centroids, Gaussian vertex offsets (mean edge `edge` pixels, log-normal with `spread`), uniform depths
  mesh   a closed shared-vertex surface (a jittered torus) before the camera, gradients meeting in shared vertices
  walk   the same surface around the camera: projection, near-plane splitting and rendering in every frame
"""
import math

import torch

import trigrad_amd
from trigrad_amd import camera

SCENE = dict(kind="soup", triangles=1000, width=256, height=256, edge=8.0, spread=0.0, tilted=False, low=0.2, high=0.95,
             task="train", pixel_order=True, layers=32, tile=16, depth_loss=False)


def _case(**kw):
    assert set(kw) <= set(SCENE) | {"name"}
    return dict(SCENE, **kw)


def listed():
    return [
        # a unit test's frame, or the first steps of a tutorial: nothing but launches and host work
        _case(name="fixture_train", triangles=20, width=50, height=50, edge=20.0),
        # a thumbnail that an interactive program fits, in tile order
        _case(name="thumbnail_train_tile", triangles=1000, width=256, height=256, edge=11.4, pixel_order=False, layers=-1),
        # an ordinary optimisation step with the defaults of the entry point
        _case(name="medium_train", triangles=100_000, width=1024, height=1024),
        # sizes that are no multiple of anything, small tiles, per-vertex depths, a loss on the depth map too
        _case(name="ragged_depth_train", triangles=33_331, width=1237, height=693, edge=13.0, spread=0.5, tilted=True, tile=8,
              depth_loss=True),
        # the headline frame: a million triangles with a heavy tail of large ones, in tile order and with the defaults
        _case(name="million_train_tile", triangles=1_000_000, width=1920, height=1080, edge=4.0, spread=1.0, pixel_order=False,
              layers=-1),
        _case(name="million_train", triangles=1_000_000, width=1920, height=1080, edge=4.0, spread=1.0),
        # the same frame shown, not trained
        _case(name="million_view", triangles=1_000_000, width=1920, height=1080, edge=4.0, spread=1.0, task="view"),
        # faint large triangles stacked hundreds deep, where early termination rarely helps
        _case(name="deep_train", triangles=200_000, width=512, height=512, edge=60.0, low=0.02, high=0.15),
        # exact compositing of a translucent volume: every fragment in depth order, no limit on the layers
        _case(name="unlimited_train", triangles=20_000, width=512, height=512, edge=60.0, low=0.02, high=0.15, layers=-1),
        # a large shared-vertex mesh being refined: up to four layers per pixel, six triangles at every vertex
        _case(name="mesh_train", kind="mesh", triangles=1_300_000, width=1920, height=1080, low=0.9, high=0.9),
        # a dense opaque mesh shown at the entry point's default image size
        _case(name="mesh_view_tile", kind="mesh", triangles=500_000, width=500, height=500, low=1.0, high=1.0, task="view",
              pixel_order=False),
        # a viewer's camera inside a scene: half of it behind the near plane, triangles across it
        _case(name="walk_view", kind="walk", triangles=200_000, width=1920, height=1080, low=0.5, high=0.95, task="view"),
    ]


def _log(rng, low, high):
    return math.exp(rng.uniform(math.log(low), math.log(high)))


def _area(case):
    """Mean area in pixels of a soup's triangle: three Gaussian points of deviation s span sqrt(3) / 2 s^2; the mean edge is s sqrt(pi)."""
    return math.sqrt(3.0) / 2.0 / math.pi * case["edge"] ** 2 * math.exp(2.0 * case["spread"] ** 2)


def _keys(case):
    """About how many (tile, triangle) pairs a soup has."""
    reach = 0.85 * case["edge"] * math.exp(0.5 * case["spread"] ** 2) / case["tile"]
    return case["triangles"] * (1.0 + 2.0 * reach + reach ** 2 * math.exp(case["spread"] ** 2))


def draw(rng):
    kind = rng.choice(["soup", "soup", "soup", "soup", "mesh", "walk"])
    pixels = _log(rng, 2_500, 2_073_600)
    aspect = rng.uniform(0.6, 1.8)
    width = max(33, min(1920, round(math.sqrt(pixels * aspect))))
    height = max(33, min(1080, round(pixels / width)))
    if kind != "soup":
        low = rng.choice([0.5, 0.9, 1.0])
        return _case(kind=kind, triangles=round(_log(rng, 2_000, 200_000 if kind == "walk" else 1_300_000)), width=width, height=height,
                     low=low, high=max(low, 0.95), task="view" if kind == "walk" else rng.choice(["view", "train"]),
                     pixel_order=rng.random() < 0.6)
    while True:
        order = rng.choice(["pixel", "pixel", "tile", "unlimited"])
        faint = rng.random() < 0.3
        case = _case(width=width, height=height, edge=round(_log(rng, 3.0, 64.0), 2), spread=rng.choice([0.0, 0.5, 1.0]),
                     tilted=rng.random() < 0.5, low=0.02 if faint else 0.2, high=0.15 if faint else 0.95,
                     task=rng.choice(["view", "train", "train"]), pixel_order=order != "tile",
                     layers=-1 if order != "pixel" else rng.choice([32, 32, 8]), tile=rng.choice([16, 16, 16, 8, 32]),
                     depth_loss=rng.random() < 0.25)
        depth = _log(rng, 0.5, 60.0 if order == "unlimited" else 700.0)
        case["triangles"] = round(depth * width * height / _area(case))
        # no larger than the largest listed cases: their pairs, and their (pixel, triangle) coverings
        covered = depth * width * height
        bound = 16e6 if order == "unlimited" else 150e6 if faint else 30e6
        if 10 <= case["triangles"] <= 1_000_000 and _keys(case) <= 3e6 and covered <= bound:
            return case


def _soup(case, g, device):
    n, w, h = case["triangles"], case["width"], case["height"]
    uniform = lambda *shape: torch.rand(shape, generator=g, device=device)  # noqa: E731
    normal = lambda *shape: torch.randn(shape, generator=g, device=device)  # noqa: E731
    sigma = case["edge"] / math.sqrt(math.pi) * torch.exp(case["spread"] * normal(n, 1, 1))
    xy = uniform(n, 1, 2) * 2.0 - 1.0 + normal(n, 3, 2) * sigma * torch.tensor([2.0 / w, 2.0 / h], device=device)
    z = (0.1 + 9.9 * uniform(n, 1, 1)).expand(n, 3, 1)
    if case["tilted"]:
        z = z * (0.9 + 0.2 * uniform(n, 3, 1))
    vertices = torch.cat([xy, z, 1.0 / z], dim=-1).reshape(3 * n, 4)
    return vertices, torch.arange(3 * n, dtype=torch.int32, device=device).reshape(n, 3)


def _torus(case, g, device):
    """Positions of a jittered torus of about `triangles` triangles (radii 1 and 0.4, spun about its axis) and its indices."""
    around = max(8, round(math.sqrt(case["triangles"])))
    across = max(4, case["triangles"] // (2 * around))
    u, v = torch.meshgrid(torch.arange(around, device=device), torch.arange(across, device=device), indexing="ij")
    spin, roll = (torch.rand(2, generator=g, device=device) * (2.0 * math.pi)).unbind()
    a, b = u * (2.0 * math.pi / around) + spin, v * (2.0 * math.pi / across) + roll
    ring = 1.0 + 0.4 * torch.cos(b)
    xyz = torch.stack([ring * torch.cos(a), ring * torch.sin(a), 0.4 * torch.sin(b)], dim=-1).reshape(-1, 3)
    xyz = xyz + 1e-3 * torch.randn(xyz.shape, generator=g, device=device)
    at = lambda i, j: (i % around) * across + j % across  # noqa: E731
    quads = torch.stack([at(u, v), at(u + 1, v), at(u, v + 1), at(u + 1, v), at(u + 1, v + 1), at(u, v + 1)], dim=-1)
    return xyz, quads.reshape(-1, 3).to(torch.int32).contiguous()


def _look(eye, forward, up, device):
    """World to eye coordinates of a camera at `eye` (it looks down -z)."""
    f = torch.tensor(forward, device=device) / math.dist(forward, (0.0, 0.0, 0.0))
    s = torch.linalg.cross(f, torch.tensor(up, device=device))
    s = s / s.norm()
    m = torch.eye(4, device=device)
    m[:3, :3] = torch.stack([s, torch.linalg.cross(s, f), -f])
    m[:3, 3] = -m[:3, :3] @ torch.tensor(eye, device=device)
    return m


def prepare(case, seed):
    device = torch.device("cuda")
    g = torch.Generator(device=device).manual_seed(seed)
    w, h, train = case["width"], case["height"], case["task"] == "train"
    state = {"walk": case["kind"] == "walk",
             "args": (w, h, case["tile"], case["tile"], 1 / 256, False, case["pixel_order"], case["layers"])}
    if case["kind"] == "soup":
        vertices, state["indices"] = _soup(case, g, device)
    else:
        xyz, state["indices"] = _torus(case, g, device)
        if case["kind"] == "mesh":
            view = _look((0.0, -2.6, 2.2), (0.0, 2.6, -2.2), (0.0, 0.0, 1.0), device)
            vertices = camera.project(xyz, camera.perspective(45.0, w, h, device=device) @ view).contiguous()
        else:
            view = _look((1.0, 0.0, 0.0), (-0.3, 1.0, 0.1), (0.0, 0.0, 1.0), device)
            state["matrix"] = camera.perspective(70.0, w, h, near=0.05, far=10.0, device=device) @ view
            vertices = xyz
    n = vertices.shape[0]
    colors = torch.rand((n, 3), generator=g, device=device)
    opacities = case["low"] + (case["high"] - case["low"]) * torch.rand((n,), generator=g, device=device)
    for name, t in (("vertices", vertices), ("colors", colors), ("opacities", opacities)):
        state[name] = t.requires_grad_() if train else t
    if train:
        # the gradient of a mean squared error against a random target
        state["upstream"] = [(torch.rand((h, w, 4), generator=g, device=device) * 2.0 - 1.0) / (2 * h * w)]
        if case["depth_loss"]:
            state["upstream"].append((torch.rand((h, w), generator=g, device=device) * 2.0 - 1.0) / (h * w))
    return state


def run(state):
    if "upstream" in state:
        leaves = (state["vertices"], state["colors"], state["opacities"])
        image, depthmap = trigrad_amd.render(leaves[0], state["indices"], leaves[1], leaves[2], *state["args"])
        upstream = state["upstream"]
        gradients = torch.autograd.grad((image, depthmap)[:len(upstream)], leaves, upstream)
        return (image.detach(), depthmap.detach(), *gradients)
    vertices, indices, colors, opacities = state["vertices"], state["indices"], state["colors"], state["opacities"]
    with torch.no_grad():
        if state["walk"]:
            clip = camera.to_clip(vertices, state["matrix"])
            clip, indices, colors, opacities = camera.split_clipped(clip, indices, colors, opacities)
            vertices = camera.clip_to_render(clip)
        return trigrad_amd.render(vertices, indices, colors, opacities, *state["args"])


def work(case):
    """Scene and upstream gradients read once, image, depth map and gradients written once; the arithmetic of the fragments that
    are blended (about 70 operations forward and 450 backward each), estimated from the triangles' mean area and opacity."""
    pixels, n = case["width"] * case["height"], case["triangles"]
    vertices = 3 * n if case["kind"] == "soup" else n // 2
    scene = 12.0 * n + 32.0 * vertices - (4.0 * vertices if case["kind"] == "walk" else 0.0)
    opacity = min(0.9999, 0.5 * (case["low"] + case["high"]))
    stop = math.log(256.0) / -math.log(1.0 - opacity)  # layers until the threshold is reached
    depth = n * _area(case) / pixels if case["kind"] == "soup" else 1.0 if case["kind"] == "mesh" else 3.0
    layers = case["layers"] if case["layers"] > 0 else math.inf
    fragments = pixels * min(depth, layers, math.ceil(stop))
    if case["task"] == "view":
        return {"bytes": scene + 20.0 * pixels, "flops": 70.0 * fragments}
    return {"bytes": scene + 32.0 * vertices + (36.0 + (4.0 if case["depth_loss"] else 0.0)) * pixels, "flops": 520.0 * fragments}


def tolerance(case):
    """float32 throughout; a gradient is a float32 sum of many terms that partly cancel, in no fixed order."""
    return {"rel": 1e-5, "max": 1e-3}

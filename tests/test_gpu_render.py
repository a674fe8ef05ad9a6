"""GPU parity of the forward blend and the backward pass against the CPU oracle.

Bars (the ones the task states): image within 1e-5 absolute; gradients within
1e-4 relative + 1e-6 absolute.  The forward kernels evaluate the oracle's
float32 expression tree operation for operation, so the image is in fact
expected to be bit-identical; the number of differing values is reported and
bounded.  The oracle accumulates gradients in float64, the GPU sums float32
terms with atomics in arbitrary order, hence the gradient tolerance.

Everything here calls the C ABI of libtrigrad_hip.so through trigrad_amd.
"""
import numpy as np
import pytest

from helpers import GRAD_ATOL, GRAD_RTOL, assert_gradients_close, assert_close, to_device, u64
from test_gpu_stages import SCENES

pytestmark = pytest.mark.gpu

IMAGE_ATOL = 1e-5

MODES = {
    "A_default": dict(per_pixel_sort=True, max_layers=32),
    "A_unlimited": dict(per_pixel_sort=True, max_layers=-1),
    "A_5_layers": dict(per_pixel_sort=True, max_layers=5),
    "A_40_layers": dict(per_pixel_sort=True, max_layers=40),
    "B_unlimited": dict(per_pixel_sort=False, max_layers=-1),
    "B_3_layers": dict(per_pixel_sort=False, max_layers=3),
}


def _nan_equal(a, b):
    return np.array_equal(a, b, equal_nan=True)


def _forward_both(scene, tw, th, mode, cuda, oracle, thr=1 / 256, frames=1):
    """frames: which frame of the scene it is; the first one's buffers are made for a guess of K, and what is a long tile, or
    sorted by one workgroup, goes by the buffers."""
    from trigrad_amd import _C
    W, H = scene["width"], scene["height"]
    d = to_device(scene, cuda)
    M = scene["indices"].shape[0]
    ml = mode["max_layers"] if mode["max_layers"] > 0 else M + 1
    want = oracle.render(scene["vertices"], scene["indices"], scene["colors"], scene["opacities"], W, H, tw, th, thr,
                         mode["per_pixel_sort"], ml)
    for _ in range(frames):
        got = _C._forward_full(d["vertices"], d["indices"], d["colors"], d["opacities"], W, H, tw, th, thr, True,
                               mode["per_pixel_sort"], ml)
    return d, want, got, ml


def _long_tile_limit(scene, tw, th, per_pixel_sort, n_keys):
    """How many list entries make a tile a long one, in a frame whose number of keys is known: 1024 and twice the mean, but in a
    frame of few workgroups and small triangles 1024."""
    from trigrad_amd import _C
    capacity, n = _C._round_capacity(int(n_keys)), scene["indices"].shape[0]
    tiles = -(-scene["width"] // tw) * -(-scene["height"] // th)
    few = tiles * -(-tw * th // 256) <= (128 if per_pixel_sort else 256) and capacity <= 4 * n
    return 1024 if few else max(1024, -(-2 * capacity // tiles))


def _shared_out(got, want, tw, th):
    """Of a frame in tile order: the tiles whose pixels were several workgroups', of which the saved hit masks do not say how far
    they got (the words in front of them, one for each workgroup of a tile)."""
    n_tiles, parts = want["offsets"].size - 1, -(-tw * th // 256)
    return (got[8][4][:n_tiles * parts].view(n_tiles, parts) == -1).all(1).cpu().numpy()


def _check_forward(name, want, got, tile_shape):
    from trigrad_amd import _C
    image, depthmap, weights, sorted_ids, offsets, bary, ends, timings, (last, last_depth, status, fragments, hit_masks) = got
    status.verify()
    np.testing.assert_array_equal(offsets.cpu().numpy(), want["offsets"])
    np.testing.assert_array_equal(sorted_ids.cpu().numpy(), want["sorted_ids"])
    img = image.cpu().numpy()
    finite = np.isfinite(want["image"])
    assert _nan_equal(np.isnan(img), np.isnan(want["image"])), f"{name}: NaN pattern differs"
    assert_close(f"{name}: image", np.where(finite, img, 0), np.where(finite, want["image"], 0), 0.0, IMAGE_ATOL)
    dm = depthmap.cpu().numpy()
    fin = np.isfinite(want["depthmap"])
    assert _nan_equal(np.isfinite(dm), fin)
    assert_close(f"{name}: depthmap", np.where(fin, dm, 0), np.where(fin, want["depthmap"], 0), 1e-5, 1e-5)
    np.testing.assert_array_equal(ends.cpu().numpy(), want["ends"])
    np.testing.assert_array_equal(last.cpu().numpy(), want["last"])
    if fragments is not None:
        # saved blend order: `ends` valid layers per pixel, no list position twice, and the last
        # layer is the entry `last` points at (the backward parity tests check the content)
        tile_h, tile_w = tile_shape
        fr = _C.saved_blend_order(fragments, offsets, tile_w, tile_h).cpu().numpy()
        en, la = want["ends"], want["last"]
        layer = np.arange(fr.shape[0])[:, None, None]
        valid = layer < en[None]
        assert (fr[valid] >= 0).all()
        ys, xs = np.nonzero(en > 0)
        np.testing.assert_array_equal(fr[en[ys, xs] - 1, ys, xs], la[ys, xs] - 1)
        srt = np.sort(np.where(valid, fr, -1 - layer), axis=0)
        assert (np.diff(srt, axis=0) != 0).all()
    # (NaN results carry different payload/sign bits on the two machines)
    differing = int(((img.view(np.uint32) != want["image"].view(np.uint32)) & ~np.isnan(img)).sum())
    assert differing == 0, f"{name}: {differing} image values are not bit-identical to the oracle"
    assert _nan_equal(weights.cpu().numpy(), want["weights"])


@pytest.mark.parametrize("mode", sorted(MODES))
@pytest.mark.parametrize("name", sorted(SCENES))
def test_forward_matches_oracle(name, mode, cuda, oracle):
    scene, tw, th = SCENES[name]()
    _, want, got, _ = _forward_both(scene, tw, th, MODES[mode], cuda, oracle)
    _check_forward(f"{name}/{mode}", want, got, (th, tw))


def _long_list_scene():
    """One 16x16 tile whose list is longer than 65535 entries next to tiles with short lists: the per-pixel-order
    forward pass keeps list positions in 16 bits where they fit and hands the other tiles to a second launch."""
    import scenes as S
    crowd = S.random_soup(70000, 32, 32, seed=3, sigma_px=1.5, opacity=(0.02, 0.2))
    v = crowd["vertices"].copy()
    v[:, :2] = v[:, :2] * 0.45 - 0.5  # into the first tile (with a fringe over its neighbours)
    rest = S.random_soup(1500, 32, 32, seed=4, sigma_px=5.0)
    vertices = np.concatenate([v, rest["vertices"]])
    indices = np.concatenate([crowd["indices"], rest["indices"] + v.shape[0]]).astype(np.int32)
    scene = dict(crowd)
    scene.update(vertices=vertices, indices=indices, colors=np.concatenate([crowd["colors"], rest["colors"]]),
                 opacities=np.concatenate([crowd["opacities"], rest["opacities"]]))
    return scene


@pytest.mark.parametrize("mode,tile", [("A_default", 16), ("A_40_layers", 16), ("B_3_layers", 16), ("A_default", 32)])
def test_tile_list_longer_than_16_bit_positions(mode, tile, cuda, oracle):
    import torch
    from trigrad_amd import _C
    scene = _long_list_scene()
    m = MODES[mode]
    d, want, got, ml = _forward_both(scene, tile, tile, m, cuda, oracle)
    lengths = np.diff(want["offsets"])
    # 16x16: one long list next to short ones; 32x32: the one tile is four workgroups on the long list
    assert lengths.max() > 65535 and (tile == 32 or lengths.min() < 65535)
    _check_forward(f"long list/{mode}", want, got, (tile, tile))
    gi, gd = _grad_inputs(scene, 9, True)
    wanted = oracle.render_backward(gi, gd, scene["vertices"], scene["indices"], scene["colors"], scene["opacities"], want,
                                    32, 32, tile, tile, m["per_pixel_sort"], ml, literal=False, magnitudes=True)
    image, depthmap, weights, sorted_ids, offsets, bary, ends, _, resume = got
    out = _C.render_backward(torch.from_numpy(gi).to(cuda), torch.from_numpy(gd).to(cuda), d["vertices"], d["indices"],
                             d["colors"], d["opacities"], sorted_ids, offsets, bary, image, depthmap, weights, ends, 32, 32,
                             tile, tile, 1 / 256, m["per_pixel_sort"], ml, resume=resume)
    for label, g, w, mag in zip(("grad_vertices", "grad_colors", "grad_opacities"), out, wanted[:3], wanted[3:]):
        assert_gradients_close(f"long list/{mode}: {label}", g.cpu().numpy(), w, mag)


def _crowded_scene(n, width, height):
    """Triangles of a pixel or two, most of them in one corner (a list far longer than the mean), a few large ones, and some
    whose vertices are infinite or NaN or whose 1/w is zero."""
    import scenes as S
    soup = S.random_soup(n, width, height, seed=21, sigma_px=0.8, opacity=(0.1, 0.9), varying_w=True)
    v = soup["vertices"].copy().reshape(n, 3, 4)
    corner = np.random.default_rng(5).random(n) < 0.7
    v[corner, :, :2] = (v[corner, :, :2] + 1.0) * 0.12 - 1.0
    big = np.arange(n) % 97 == 0
    centre = v[big, :, :2].mean(axis=1, keepdims=True)
    v[big, :, :2] = centre + (v[big, :, :2] - centre) * 15.0
    v[5::501, 1, 0], v[7::503, 2, 1], v[9::499, 0, 3] = np.inf, np.nan, 0.0
    return dict(soup, vertices=v.reshape(-1, 4))


@pytest.mark.parametrize("mode", ["A_default", "A_40_layers", "B_unlimited"])
@pytest.mark.parametrize("n,width,height,tw,th", [
    (12000, 70, 45, 16, 16),   # partial tiles on both sides
    (1500, 70, 45, 8, 8),      # one wave to a workgroup
    (12000, 70, 45, 24, 16),   # six squares of 8 x 8 pixels, two workgroups
    (12000, 64, 64, 32, 32),
    (6000, 70, 45, 12, 6),     # a wave's pixels are no square
    (40000, 640, 400, 16, 16),  # more tiles than run at once: the longest lists' first
])
def test_crowds_of_small_triangles_match_oracle(n, width, height, tw, th, mode, cuda, oracle):
    scene = _crowded_scene(n, width, height)
    _, want, got, _ = _forward_both(scene, tw, th, MODES[mode], cuda, oracle, frames=3)
    _check_forward(f"crowd {n}/{tw}x{th}/{mode}", want, got, (th, tw))
    lengths = np.diff(want["offsets"])
    long = lengths >= _long_tile_limit(scene, tw, th, MODES[mode]["per_pixel_sort"], lengths.sum())
    assert long.any() == (n > 1500)
    # with depth bounds where lists are of 512 entries on average and more, in per-pixel order
    assert (lengths.mean() >= 512) == (n == 12000)
    if not MODES[mode]["per_pixel_sort"]:
        assert np.array_equal(_shared_out(got, want, tw, th), long & (-(-tw * th // 64) >= 4))


@pytest.mark.parametrize("shape", ["tiny", "sliver", "on_centres", "far_corner", "flat"])
@pytest.mark.parametrize("width,height,tw,th", [(400, 304, 16, 16), (203, 101, 8, 8), (203, 101, 12, 10)])
def test_triangles_beside_a_waves_pixels(shape, width, height, tw, th, cuda, oracle):
    """Per-pixel order, batches of 64: a wave leaves out the entries whose vertices are all to one side of its pixels.  Triangles
    whose edges alone say little of that, or whose matrix is the inverse of their vertices in a few bits only: the images are the
    oracle's bit for bit."""
    import scenes as S
    n = 4000
    scene = S.random_soup(n, width, height, seed=3, sigma_px=1.0 if shape == "tiny" else 4.0, opacity=(0.05, 0.9), varying_w=True)
    rng = np.random.default_rng(len(shape))
    v = scene["vertices"].reshape(n, 3, 4)
    xy = v[:, :, :2].astype(np.float64)
    if shape == "sliver":  # the third vertex on the line through the others but for 1e-9 to 1e-2
        t = rng.uniform(0, 1, (n, 1))
        xy[:, 2] = xy[:, 0] * (1 - t) + xy[:, 1] * t + 10 ** rng.uniform(-9, -2, (n, 1)) * rng.standard_normal((n, 2))
    if shape == "on_centres":
        size = np.array([width, height])
        xy = (np.floor((xy + 1) / 2 * size) + 0.5) / size * 2 - 1
    if shape == "far_corner":
        xy[:, 0] *= 10 ** rng.uniform(0, 6, (n, 1))
    if shape == "flat":  # two vertices, or all three, with the same x or y up to a few roundings
        axis = rng.integers(0, 2, n)
        for k in (1, 2):
            xy[np.arange(n), k, axis] = xy[np.arange(n), 0, axis] + 1e-7 * rng.standard_normal(n) * (rng.random(n) < 0.8)
    v[:, :, :2] = xy.astype(np.float32)
    _, want, got, _ = _forward_both(scene, tw, th, MODES["A_default"], cuda, oracle, frames=2)
    assert np.diff(want["offsets"]).mean() < 512  # no depth bounds
    _check_forward(f"{shape}/{width}x{height}/{tw}x{th}", want, got, (th, tw))


@pytest.mark.parametrize("mode", ["A_default", "B_unlimited"])
@pytest.mark.parametrize("n,others,width,lane_by_lane", [(255, 0, 272, False), (256, 0, 272, True), (400, 28_000, 272, False),
                                                         (1023, 70_000, 272, False), (1024, 70_000, 272, True), (90, 0, 16, True),
                                                         (90, 15_000, 256, True)])
def test_small_triangles_around_the_edges_of_their_rule(n, others, width, lane_by_lane, mode, cuda, oracle):
    """Which lists have their small triangles tested lane by lane: of 1024 entries, or of 256 and four times the mean, in frames
    with more than 256 tiles (here 272), and every list in others.  One tile with a list of n, the rest spread evenly."""
    import scenes as S
    height = 16 if width == 16 else 256
    scene = S.random_soup(n + others, width, height, seed=n, sigma_px=0.7, opacity=(0.02, 0.2), varying_w=True)
    v = scene["vertices"].reshape(n + others, 3, 4)
    v[:n, :, 0] = (v[:n, :, 0] * 0.4 + 1.0) * 16 / width - 1.0
    v[:n, :, 1] = (v[:n, :, 1] * 0.4 + 1.0) * 16 / height - 1.0
    if others:  # none in the first column of tiles
        v[n:, :, 0] = np.where(v[n:, :, 0] < 33 / width * 2 - 1, v[n:, :, 0] * 0.5 + 0.4, v[n:, :, 0])
    _, want, got, _ = _forward_both(scene, 16, 16, MODES[mode], cuda, oracle)
    lengths = np.diff(want["offsets"])
    assert lengths[0] == n and lengths.size == (1 if width == 16 else width // 16 * 16)
    assert (lengths.size <= 256 or n >= 1024 or (n >= 256 and n >= 4 * lengths.mean())) == lane_by_lane
    _check_forward(f"{n} small of {others}/{mode}", want, got, (16, 16))


@pytest.mark.parametrize("mode", ["A_default", "A_40_layers", "B_unlimited"])
def test_more_long_tiles_than_slots(mode, cuda, monkeypatch):
    """Some 400 tiles with long lists, of which 128 are started first: the frame is that of the stage-by-stage route, which
    starts none first."""
    import torch
    import scenes as S
    from trigrad_amd import _C
    n, width, height, tile = 500_000, 320, 240, 8
    soup = S.random_soup(n, width, height, seed=8, sigma_px=0.6, opacity=(0.02, 0.3))
    v = soup["vertices"].reshape(n, 3, 4).copy()
    v[: n * 95 // 100, :, :2] = (v[: n * 95 // 100, :, :2] + 1.0) * 0.6 - 1.0
    d = to_device(dict(soup, vertices=v.reshape(-1, 4)), cuda)
    m = MODES[mode]
    ml = m["max_layers"] if m["max_layers"] > 0 else n + 1
    args = (d["vertices"], d["indices"], d["colors"], d["opacities"], width, height, tile, tile, 1 / 256, True, m["per_pixel_sort"], ml)
    for _ in range(3):  # the first frame's buffers are made for a guess of K, and what is long depends on them
        got = _C.render_forward(*args)
    lengths = got[4][1:] - got[4][:-1]
    assert int((lengths >= max(1024, -(-2 * _C._round_capacity(got[3].numel()) // lengths.numel()))).sum()) > 128
    monkeypatch.setattr(_C, "ONE_CALL_FRAME", False)
    want = _C.render_forward(*args)
    for i in (0, 1, 2, 3, 4, 5, 6):
        assert torch.equal(got[i].view(torch.int32), want[i].view(torch.int32)), i


def test_more_long_tiles_than_slots_in_tile_order(cuda, monkeypatch):
    """The same in tile order, where tiles are started out of turn in frames with more than 2048 of them: 4800 tiles, some 240
    of them with lists beyond 1024 entries."""
    import torch
    import scenes as S
    from trigrad_amd import _C
    n, width, height, tile = 500_000, 640, 480, 8
    soup = S.random_soup(n, width, height, seed=8, sigma_px=0.6, opacity=(0.02, 0.3))
    v = soup["vertices"].reshape(n, 3, 4).copy()
    v[: n * 95 // 100, :, :2] = (v[: n * 95 // 100, :, :2] + 1.0) * 0.225 - 1.0
    d = to_device(dict(soup, vertices=v.reshape(-1, 4)), cuda)
    args = (d["vertices"], d["indices"], d["colors"], d["opacities"], width, height, tile, tile, 1 / 256, True, False, n + 1)
    for _ in range(3):
        got = _C.render_forward(*args)
    lengths = got[4][1:] - got[4][:-1]
    assert lengths.numel() > 2048
    assert int((lengths >= max(1024, -(-2 * _C._round_capacity(got[3].numel()) // lengths.numel()))).sum()) > 128
    monkeypatch.setattr(_C, "ONE_CALL_FRAME", False)
    want = _C.render_forward(*args)
    for i in (0, 1, 2, 3, 4, 5, 6):
        assert torch.equal(got[i].view(torch.int32), want[i].view(torch.int32)), i


def _grad_inputs(scene, seed, with_depth):
    rng = np.random.default_rng(seed)
    H, W = scene["height"], scene["width"]
    gi = rng.standard_normal((H, W, 4)).astype(np.float32)
    gd = rng.standard_normal((H, W)).astype(np.float32) if with_depth else np.zeros((H, W), np.float32)
    return gi, gd


BACKWARD_SCENES = ["config0", "soup_varying_w", "soup_shared", "soup_big_tris", "soup_tile4", "soup_tile32", "soup_tile_8x4",
                   "squares", "large_triangles", "depth_overlap", "overlapping_triangles", "unit_square_negative_z", "overlap_mesh_inf_w",
                   "grid_mesh", "degenerate", "center_island", "soup_tile8", "soup_tile_24x16"]


@pytest.mark.parametrize("with_depth", [False, True])
@pytest.mark.parametrize("mode", sorted(MODES))
@pytest.mark.parametrize("name", BACKWARD_SCENES)
def test_backward_matches_oracle(name, mode, with_depth, cuda, oracle):
    import torch
    from trigrad_amd import _C
    scene, tw, th = SCENES[name]()
    m = MODES[mode]
    d, want, got, ml = _forward_both(scene, tw, th, m, cuda, oracle)
    W, H = scene["width"], scene["height"]
    gi, gd = _grad_inputs(scene, 5, with_depth)
    wanted = oracle.render_backward(gi, gd, scene["vertices"], scene["indices"], scene["colors"], scene["opacities"], want,
                                    W, H, tw, th, m["per_pixel_sort"], ml, literal=False, magnitudes=True)
    image, depthmap, weights, sorted_ids, offsets, bary, ends, _, resume = got
    # the blend order is saved exactly when per-pixel order meets max_layers <= 32;
    # then the route that selects the fragments again is checked as well
    saved_order = resume[3] is not None
    assert saved_order == (bool(m["per_pixel_sort"]) and ml <= _C.MAX_SAVED_LAYERS)
    assert (resume[4] is not None) == (not m["per_pixel_sort"])  # tile order saves its hit masks
    routes = [("", resume)]
    if saved_order:
        routes.append((" (re-selected)", resume[:3] + (None, None)))
    if resume[4] is not None:
        routes.append((" (inside tests repeated)", resume[:4] + (None,)))
    for route, res in routes:
        out = _C.render_backward(torch.from_numpy(gi).to(cuda), torch.from_numpy(gd).to(cuda), d["vertices"], d["indices"],
                                 d["colors"], d["opacities"], sorted_ids, offsets, bary, image, depthmap, weights, ends, W, H,
                                 tw, th, 1 / 256, m["per_pixel_sort"], ml, resume=res)
        for label, g, w, mag in zip(("grad_vertices", "grad_colors", "grad_opacities"), out, wanted[:3], wanted[3:]):
            assert_gradients_close(f"{name}/{mode}{route}: {label}", g.cpu().numpy(), w, mag)  # NaN where the oracle has NaN
        assert float(out[0][:, 2].abs().max()) == 0.0  # z never receives a gradient (render.cu:531-533)
    if name == "soup_shared" and with_depth:
        # the three layouts of the gradient arrays the kernels know: dense, one (V,8) block, run-time strides
        for strides in ((4, 3, 1), (8, 8, 8), (6, 5, 2)):
            alt = _C.render_backward(torch.from_numpy(gi).to(cuda), torch.from_numpy(gd).to(cuda), d["vertices"], d["indices"],
                                     d["colors"], d["opacities"], sorted_ids, offsets, bary, image, depthmap, weights, ends, W,
                                     H, tw, th, 1 / 256, m["per_pixel_sort"], ml, resume=resume, grad_strides=strides)
            for a, b in zip(alt, out):
                assert a.is_contiguous() and a.shape == b.shape
                assert float((a - b).abs().max()) <= 1e-5 * float(b.abs().max()) + 1e-6


def test_default_mode_literal_and_policy_agree(oracle):
    """With per_pixel_sort on and at most 32 blended fragments the literal
    reference traversal and the reverse-order policy are the same computation."""
    import scenes as S
    scene = S.random_soup(300, 64, 64, seed=9, sigma_px=14.0, varying_w=True)
    W = H = 64
    fwd = oracle.render(scene["vertices"], scene["indices"], scene["colors"], scene["opacities"], W, H)
    gi, gd = _grad_inputs(scene, 1, True)
    a = oracle.render_backward(gi, gd, scene["vertices"], scene["indices"], scene["colors"], scene["opacities"], fwd, W, H, literal=True)
    b = oracle.render_backward(gi, gd, scene["vertices"], scene["indices"], scene["colors"], scene["opacities"], fwd, W, H, literal=False)
    for x, y in zip(a, b):
        np.testing.assert_array_equal(x, y)


def test_render_autograd_end_to_end(cuda, oracle):
    """trigrad_amd.render + loss.backward() on configuration 0 (both modes)."""
    import torch
    import trigrad_amd
    import scenes as S
    scene = S.config(0)
    W, H = scene["width"], scene["height"]
    d = to_device(scene, cuda)
    for kw in (dict(), dict(per_pixel_sort=False, max_layers=-1)):
        v = d["vertices"].clone().requires_grad_()
        c = d["colors"].clone().requires_grad_()
        o = d["opacities"].clone().requires_grad_()
        image, depthmap = trigrad_amd.render(v, d["indices"], c, o, W, H, **kw)
        loss = ((image - d["target"]) ** 2).sum()
        loss.backward()
        pps = kw.get("per_pixel_sort", True)
        ml = kw.get("max_layers", 32)
        fwd = oracle.render(scene["vertices"], scene["indices"], scene["colors"], scene["opacities"], W, H, per_pixel_sort=pps,
                            max_layers=ml)
        assert_close("image", image.detach().cpu().numpy(), fwd["image"], 0.0, IMAGE_ATOL)
        gi = 2.0 * (fwd["image"] - scene["target"])
        wanted = oracle.render_backward(gi, np.zeros((H, W), np.float32), scene["vertices"], scene["indices"], scene["colors"],
                                        scene["opacities"], fwd, W, H, per_pixel_sort=pps, max_layers=ml, magnitudes=True)
        for label, g, w, mag in zip(("grad_vertices", "grad_colors", "grad_opacities"), (v.grad, c.grad, o.grad), wanted[:3], wanted[3:]):
            assert_gradients_close(label, g.cpu().numpy(), w, mag)


def test_forward_mode_is_refused_for_known_frames_too(cuda):
    """The first frame of a kind goes through the Python function, later ones do not: a tangent is refused either way."""
    import scenes as S
    import torch
    import trigrad_amd
    from torch.autograd import forward_ad
    d = to_device(S.random_soup(40, 48, 48, seed=2), cuda)
    args = (d["indices"], d["colors"], d["opacities"], 48, 48)
    for _ in range(3):
        trigrad_amd.render(d["vertices"], *args)
    with forward_ad.dual_level():
        dual = forward_ad.make_dual(d["vertices"], torch.ones_like(d["vertices"]))
        with pytest.raises(RuntimeError):
            trigrad_amd.render(dual, *args)
    with pytest.raises(RuntimeError):
        torch.func.vmap(lambda v: trigrad_amd.render(v, *args)[0])(d["vertices"][None])


def test_loss_on_depth_only(cuda, oracle):
    """Only the depth map takes part in the loss: the image's gradient arrives as None."""
    import torch
    import trigrad_amd
    import scenes as S
    scene = S.random_soup(400, 96, 80, seed=21, sigma_px=9.0, varying_w=True)
    W, H = scene["width"], scene["height"]
    d = to_device(scene, cuda)
    v = d["vertices"].clone().requires_grad_()
    c = d["colors"].clone().requires_grad_()
    o = d["opacities"].clone().requires_grad_()
    image, depthmap = trigrad_amd.render(v, d["indices"], c, o, W, H)
    hit = torch.isfinite(depthmap)
    weight = torch.linspace(0.5, 1.5, W * H, device=cuda).reshape(H, W)
    (torch.where(hit, depthmap, torch.zeros_like(depthmap)) * weight).sum().backward()
    fwd = oracle.render(scene["vertices"], scene["indices"], scene["colors"], scene["opacities"], W, H)
    gd = np.where(np.isfinite(fwd["depthmap"]), weight.cpu().numpy(), 0.0).astype(np.float32)
    wanted = oracle.render_backward(np.zeros((H, W, 4), np.float32), gd, scene["vertices"], scene["indices"], scene["colors"],
                                    scene["opacities"], fwd, W, H, magnitudes=True)
    for label, g, w, mag in zip(("grad_vertices", "grad_colors", "grad_opacities"), (v.grad, c.grad, o.grad), wanted[:3], wanted[3:]):
        assert_gradients_close(label, g.cpu().numpy(), w, mag)
    assert float(v.grad.abs().max()) > 0


@pytest.mark.parametrize("mode", ["A_default", "B_unlimited"])
def test_repeatable_and_stream_ordered(mode, cuda):
    """Two calls give bit-identical images and lists (only the gradient sums depend on the order of atomics), and a
    call on a side stream, ordered after the inputs' producer, gives the same result as on the default stream."""
    import torch
    import trigrad_amd
    import scenes as S
    if mode not in MODES:
        pytest.skip("mode table changed")
    kw = dict(per_pixel_sort=MODES[mode]["per_pixel_sort"], max_layers=MODES[mode]["max_layers"])
    scene = S.random_soup(2500, 200, 160, seed=31, sigma_px=10.0, varying_w=True)
    W, H = scene["width"], scene["height"]
    d = to_device(scene, cuda)

    def run():
        v = d["vertices"].clone().requires_grad_()
        c = d["colors"].clone().requires_grad_()
        o = d["opacities"].clone().requires_grad_()
        image, depthmap = trigrad_amd.render(v, d["indices"], c, o, W, H, **kw)
        (image.square().sum() + torch.where(torch.isfinite(depthmap), depthmap, torch.zeros_like(depthmap)).sum()).backward()
        return image.detach(), depthmap.detach(), v.grad, c.grad, o.grad

    first = run()
    second = run()
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        third = run()
    side.synchronize()
    for other in (second, third):
        assert torch.equal(first[0], other[0]) and torch.equal(first[1], other[1])
        for a, b in zip(first[2:], other[2:]):
            scale = float(a.abs().max())
            assert float((a - b).abs().max()) <= 1e-5 * scale + 1e-6


@pytest.mark.parametrize("mode", ["A_default", "A_5_layers", "A_40_layers", "A_unlimited"])
@pytest.mark.parametrize("name", ["soup_big_tris", "squares", "config0", "overlap_mesh_inf_w", "unit_square_negative_z"])
def test_selection_early_stop_changes_nothing(name, mode, cuda, monkeypatch):
    """With depth bounds of the lists the per-pixel selection may leave a list early; every output stays bit-identical."""
    import torch
    from trigrad_amd import _C
    scene, tw, th = SCENES[name]()
    m = MODES[mode]
    W, H = scene["width"], scene["height"]
    d = to_device(scene, cuda)
    ml = m["max_layers"] if m["max_layers"] > 0 else scene["indices"].shape[0] + 1
    outs = []
    for threshold in (1 << 30, 0):  # never / always
        monkeypatch.setattr(_C, "EARLY_STOP_MIN_AVG_LIST", threshold)
        outs.append(_C._forward_full(d["vertices"], d["indices"], d["colors"], d["opacities"], W, H, tw, th, 1 / 256, True, True, ml))
    for a, b in zip(outs[0][:7], outs[1][:7]):
        assert torch.equal(a.view(torch.int32) if a.is_floating_point() else a, b.view(torch.int32) if b.is_floating_point() else b)
    ra, rb = outs[0][8], outs[1][8]
    assert torch.equal(ra[0], rb[0]) and torch.equal(ra[1].view(torch.int32), rb[1].view(torch.int32))
    if ra[3] is not None:
        layer = torch.arange(ra[3].shape[0], device=cuda)[:, None, None]
        valid = layer < outs[0][6][None]
        assert torch.equal(torch.where(valid, ra[3], 0), torch.where(valid, rb[3], 0))


def test_list_bounds_values(cuda):
    """tg_list_bounds: per tile and 256 entries, min over the rest of the list of (min z - 32 ulp max|z|); -inf where a
    weight is not positive and finite."""
    import torch
    from trigrad_amd import _C, _lib
    import scenes as S
    scene = S.random_soup(3000, 64, 48, seed=13, sigma_px=30.0, varying_w=True)
    v = scene["vertices"].copy()
    v[5, 3] = -1.0          # a negative weight
    v[40, 3] = np.inf       # an infinite one
    scene = dict(scene, vertices=v)
    W, H = scene["width"], scene["height"]
    d = to_device(scene, cuda)
    ids, offsets, keys, status = _C.per_tile_lists(d["vertices"], d["indices"], W, H, 16, 16)
    T = _C.num_tiles(W, H, 16, 16)
    K = ids.numel()
    lib = _lib.load(32)
    bounds = torch.full((int(lib.tg_list_bound_words(K, T)),), float("nan"), dtype=torch.float32, device=cuda)
    far_start = torch.full((T,), -1, dtype=torch.int32, device=cuda)
    low = torch.empty((scene["indices"].shape[0],), dtype=torch.float32, device=cuda)
    _lib.check(lib.tg_list_bounds(_C._ptr(d["vertices"]), v.shape[0], _C._ptr(d["indices"]), scene["indices"].shape[0],
                                  _C._ptr(keys), _C._ptr(ids), _C._ptr(offsets), T, _C._ptr(low), _C._ptr(bounds),
                                  _C._ptr(far_start), _C._stream(ids)), "tg_list_bounds")
    got, far_got = bounds.cpu().numpy(), far_start.cpu().numpy()
    ids_h, off = ids.cpu().numpy(), offsets.cpu().numpy()
    far = (u64(keys) & np.uint64(0xFFFFFFFF)) == np.uint64(np.array([1e30], np.float32).view(np.uint32)[0] ^ 0x80000000)
    tri = v[scene["indices"][ids_h]]                       # (K,3,4)
    z, w = tri[:, :, 2], tri[:, :, 3]
    ok = ((w > 0) & np.isfinite(w) & np.isfinite(z)).all(axis=1)
    lb = np.where(ok, z.min(axis=1) - np.float32(32) * np.finfo(np.float32).eps * np.abs(z).max(axis=1), -np.inf).astype(np.float32)
    lb = np.where(far, np.float32(np.inf), lb)
    assert far.any() and not far.all()
    checked = 0
    for t in range(T):
        seg_far = far[off[t]:off[t + 1]]
        assert far_got[t] == (int(np.argmax(seg_far)) if seg_far.any() else off[t + 1] - off[t])
        for p in range(0, off[t + 1] - off[t], 256):
            want = lb[off[t] + p:off[t + 1]].min()
            assert got[off[t] // 256 + t + p // 256] == want
            checked += 1
    assert checked > T and (lb == -np.inf).any() and max(off[1:] - off[:-1]) > 256


def test_record_timing_and_empty_scene(cuda):
    import torch
    import trigrad_amd
    import scenes as S
    d = to_device(S.config(0), cuda)
    image, depthmap, timings = trigrad_amd.render(d["vertices"], d["indices"], d["colors"], d["opacities"], 256, 256, record_timing=True)
    assert set(timings) == {"init", "per_tile_lists", "sorting", "bary_transforms", "rasterization"}
    assert all(t >= 0 for t in timings.values())
    v = d["vertices"].clone().requires_grad_()
    empty = torch.empty((0, 3), dtype=torch.int32, device=cuda)
    image, depthmap = trigrad_amd.render(v, empty, d["colors"], d["opacities"], 64, 48)
    assert image.shape == (48, 64, 4) and float(image[..., 3].min()) == 1.0 and float(image[..., :3].abs().max()) == 0.0
    assert torch.isinf(depthmap).all()
    image.sum().backward()
    assert float(v.grad.abs().max()) == 0.0
    image, depthmap, timings = trigrad_amd.render(v, empty, d["colors"], d["opacities"], 64, 48, record_timing=True)
    assert timings is None


def test_argument_errors(cuda):
    import torch
    import trigrad_amd
    import scenes as S
    d = to_device(S.config(0), cuda)
    v, i, c, o = d["vertices"], d["indices"], d["colors"], d["opacities"]
    with pytest.raises(ValueError, match="tile_width \\* tile_height must be <= 1024"):
        trigrad_amd.render(v, i, c, o, 64, 64, 64, 32)
    with pytest.raises(TypeError, match="vertices must be on cuda"):
        trigrad_amd.render(v.cpu(), i, c, o)
    with pytest.raises(TypeError, match="indices must be of type torch.int32"):
        trigrad_amd.render(v, i.long(), c, o)
    with pytest.raises(ValueError, match="colors must be of shape"):
        trigrad_amd.render(v, i, c[:-1], o)
    with pytest.raises(TypeError, match="opacities must be of type torch.float32"):
        trigrad_amd.render(v, i, c, o.double())


class _ReferenceShapedRenderer:
    """The call pattern of the reference's autograd Function (src/trigrad/wrapper.py:56-70, 87-98): twelve arguments
    into render_forward, eight results out, exactly eleven tensors saved, twenty arguments into render_backward."""

    @staticmethod
    def make(drop_private_state):
        import torch
        from trigrad_amd import _C

        class Fn(torch.autograd.Function):
            @staticmethod
            def forward(ctx, vertices, indices, colors, opacities, width, height, tw, th, thr, record_timing, pps, max_layers):
                ctx.args = (width, height, tw, th, thr, pps, max_layers)
                image, depthmap, final_weights, sorted_ids, offsets, bary_transforms, ends, timings = _C.render_forward(
                    vertices, indices, colors, opacities, width, height, tw, th, thr, not record_timing, pps, max_layers)
                if drop_private_state:
                    del ends._tg_resume
                ctx.save_for_backward(vertices, indices, colors, opacities, sorted_ids, offsets, bary_transforms, image, depthmap,
                                      final_weights, ends)
                return image, depthmap

            @staticmethod
            def backward(ctx, grad_image, grad_depthmap):
                saved = ctx.saved_tensors
                # which route render_backward takes: with the private state it walks what the forward pass saved,
                # without it the forward kernel runs once more
                Fn.resume_seen.append(getattr(saved[-1], "_tg_resume", None) is not None)
                gv, gc, go = _C.render_backward(grad_image, grad_depthmap, *saved, *ctx.args)
                return (gv, None, gc, go) + (None,) * 8

        Fn.resume_seen = []
        return Fn


@pytest.mark.parametrize("drop_private_state", [False, True])
@pytest.mark.parametrize("mode", ["A_default", "B_unlimited", "B_3_layers", "A_40_layers"])
def test_native_surface_as_the_reference_wrapper_calls_it(mode, drop_private_state, cuda, oracle):
    """_C.render_forward / _C.render_backward with the reference's argument lists and nothing else carried over:
    with the private state that travels on `ends`, and after a caller lost it (it is then computed again)."""
    import torch
    import scenes as S
    scene = S.random_soup(700, 150, 110, seed=21, sigma_px=11.0, varying_w=True)
    m = MODES[mode]
    W, H = scene["width"], scene["height"]
    d = to_device(scene, cuda)
    ml = m["max_layers"] if m["max_layers"] > 0 else scene["indices"].shape[0] + 1
    v = d["vertices"].clone().requires_grad_()
    c = d["colors"].clone().requires_grad_()
    o = d["opacities"].clone().requires_grad_()
    Fn = _ReferenceShapedRenderer.make(drop_private_state)
    image, depthmap = Fn.apply(v, d["indices"], c, o, W, H, 16, 16, 1 / 256, False, m["per_pixel_sort"], ml)
    rng = np.random.default_rng(5)
    gi = rng.standard_normal((H, W, 4)).astype(np.float32)
    gd = rng.standard_normal((H, W)).astype(np.float32)
    want = oracle.render(scene["vertices"], scene["indices"], scene["colors"], scene["opacities"], W, H, 16, 16, 1 / 256,
                         m["per_pixel_sort"], ml)
    assert int((image.detach().cpu().numpy().view(np.uint32) != want["image"].view(np.uint32)).sum()) == 0
    finite = np.isfinite(want["depthmap"])
    gd = np.where(finite, gd, 0).astype(np.float32)
    torch.autograd.backward([image, depthmap], [torch.from_numpy(gi).to(cuda), torch.from_numpy(gd).to(cuda)])
    wanted = oracle.render_backward(gi, gd, scene["vertices"], scene["indices"], scene["colors"], scene["opacities"], want,
                                    W, H, 16, 16, m["per_pixel_sort"], ml, magnitudes=True)
    for label, got, w, mag in zip(("grad_vertices", "grad_colors", "grad_opacities"), (v.grad, c.grad, o.grad), wanted[:3], wanted[3:]):
        assert_gradients_close(f"{mode}: {label}", got.cpu().numpy(), w, mag)
    # the attribute on `ends` must survive save_for_backward, or every backward pass pays for a second forward kernel
    assert Fn.resume_seen == [not drop_private_state]


def test_expired_wait_is_reported_on_every_path(cuda):
    """A non-zero status word of the list kernels (a bounded look-back wait expired: the lists are invalid) raises in
    the backward pass, at the start of the next frame and in verify_frames, not only when timings are recorded, and
    switches the kernels to ticketed tile numbers.  No wait is provoked: the status word is forged."""
    import torch
    import trigrad_amd
    from trigrad_amd import _C
    import scenes as S
    d = to_device(S.config(0), cuda)
    args = (d["vertices"], d["indices"], d["colors"], d["opacities"], 256, 256, 16, 16, 1 / 256)
    *results, resume = _C._forward_full(*args, True, False, 2000)
    image, depthmap, weights, sorted_ids, offsets, bary, ends = results[:7]
    try:
        bad = _C.StatusCheck(torch.ones((1,), dtype=torch.int32, device=cuda), frame=7)
        gi = torch.ones_like(image)
        with pytest.raises(RuntimeError, match="look-back wait timed out.*frame 7"):
            _C.render_backward(gi, None, *args[:4], sorted_ids, offsets, bary, image, depthmap, weights, ends, *args[4:], False, 2000,
                               resume=(resume[0], resume[1], bad, resume[3], resume[4]))
        assert _C._tickets_forced
        # the same through the public entry point: the next frame refuses to start
        _C._pending_checks.append(_C.StatusCheck(torch.ones((1,), dtype=torch.int32, device=cuda)))
        torch.cuda.synchronize()
        with pytest.raises(RuntimeError, match="look-back wait timed out"):
            trigrad_amd.render(*args[:6])
        assert not _C._pending_checks or all(not c.checked for c in _C._pending_checks)
        trigrad_amd.render(*args[:6])  # reported once; later frames run (their tiles numbered by ticket)
        # a caller that only renders forward asks before it trusts its frames
        _C._pending_checks.append(_C.StatusCheck(torch.ones((1,), dtype=torch.int32, device=cuda)))
        with pytest.raises(RuntimeError, match="look-back wait timed out"):
            trigrad_amd.verify_frames()
        trigrad_amd.verify_frames()
        # and a healthy frame's word is zero
        resume[2].verify()
    finally:
        _C.force_tickets(False)


def test_invalid_lists_show_in_the_frame(cuda):
    """The forward kernels look at the status word of the list kernels: with a word that reports an expired wait they
    read no list and fill image and depth map with NaN, in both compositing orders.  The word is forged."""
    import ctypes as C
    import torch
    from trigrad_amd import _C, _lib
    import scenes as S
    d = to_device(S.config(0), cuda)
    W = H = 256
    v, idx, col, op = d["vertices"], d["indices"], d["colors"], d["opacities"]
    *results, resume = _C._forward_full(v, idx, col, op, W, H, 16, 16, 1 / 256, True, False, 2000)
    want_image, _, _, sorted_ids, offsets, bary = results[:6]
    lib = _lib.load(32)
    for word, pps in ((0, False), (1, False), (1, True)):
        status = torch.full((1,), word, dtype=torch.int32, device=cuda)
        image = torch.zeros((H, W, 4), device=cuda)
        planes = [torch.zeros((H, W), device=cuda) for _ in range(3)]
        ends = torch.zeros((H, W), dtype=torch.int32, device=cuda)
        last = torch.zeros((H, W), dtype=torch.int32, device=cuda)
        p = lambda t: C.c_void_p(t.data_ptr())
        _lib.check(lib.tg_render_forward(p(v), p(idx), p(col), p(op), p(sorted_ids), p(offsets), p(bary), W, H, 16, 16, 1 / 256, int(pps),
                                         2000, p(image), p(planes[0]), p(planes[1]), p(ends), p(last), p(planes[2]) if pps else None,
                                         None, None, None, None, p(status), C.c_void_p(torch.cuda.current_stream().cuda_stream)),
                   "tg_render_forward")
        if word == 0:
            assert torch.equal(image, want_image)
        else:
            assert torch.isnan(image).all() and torch.isnan(planes[0]).all() and int(ends.abs().max()) == 0


def test_ticketed_tile_numbers_change_nothing(cuda, oracle):
    """force_tickets: the kernels that wait on other workgroups take their tile numbers from an atomic ticket whatever
    the size of the grid.  Lists and image are, bit for bit, what they are without."""
    import torch
    import trigrad_amd
    from trigrad_amd import _C
    import scenes as S
    scene = S.config(1)
    d = to_device(scene, cuda)
    W, H = scene["width"], scene["height"]

    def frame():
        image, _ = trigrad_amd.render(d["vertices"], d["indices"], d["colors"], d["opacities"], W, H, 16, 16, 1 / 256, False, False, -1)
        b = _C.bin_frame(d["vertices"], d["indices"], W, H, 16, 16)
        K = int(b["total_and_status"][0].item())
        keys, ids, status, offsets = _C.build_frame_lists(b, K)
        assert int(status.item()) == 0
        return image, keys.clone(), ids.clone(), offsets.clone()

    plain = frame()
    try:
        _C.force_tickets(True)
        ticketed = frame()
    finally:
        _C.force_tickets(False)
    for a, b in zip(plain, ticketed):
        assert torch.equal(a, b)


def test_frames_on_two_streams_keep_their_own_state(cuda):
    """Two streams render different frames at the same time (tickets on: the device is shared between them).  The
    binning's state between calls -- epoch-stamped look-back words, alternating digit totals -- is kept per stream,
    so every frame is what its stream gives alone."""
    import torch
    import trigrad_amd
    from trigrad_amd import _C
    import scenes as S
    frames = []
    for config in (1, 0):
        scene = S.config(config)
        d = to_device(scene, cuda)
        frames.append((d, scene["width"], scene["height"]))

    def render(k):
        d, W, H = frames[k]
        return trigrad_amd.render(d["vertices"], d["indices"], d["colors"], d["opacities"], W, H, 16, 16, 1 / 256, False, False, -1)[0]

    alone = [render(0), render(1)]
    torch.cuda.synchronize()
    streams = [torch.cuda.Stream(device=cuda), torch.cuda.Stream(device=cuda)]
    got = [[], []]
    try:
        _C.force_tickets(True)
        for _ in range(6):
            for k in (0, 1):
                with torch.cuda.stream(streams[k]):
                    got[k].append(render(k))
        torch.cuda.synchronize()
        trigrad_amd.verify_frames()
    finally:
        _C.force_tickets(False)
    states = {key for key in _C._frame_states if key[0] == cuda.index}
    assert len({key[1] for key in states}) >= 3  # the default stream's and the two streams' own
    for k in (0, 1):
        for image in got[k]:
            assert torch.equal(image, alone[k])


@pytest.mark.parametrize("mode", ["A_default", "B_unlimited"])
def test_scene_without_a_single_key(mode, cuda):
    """M >= 1 but K = 0 (every triangle degenerate): transparent image, infinite depth, zero gradients."""
    import torch
    import trigrad_amd
    m = MODES[mode]
    v = torch.tensor([[0.1, 0.1, 0.5, 2.0]] * 3 + [[float("nan"), 0.0, 0.5, 1.0], [0.2, 0.3, 0.5, 1.0], [0.4, 0.1, 0.5, 1.0]],
                     dtype=torch.float32, device=cuda).requires_grad_()
    idx = torch.tensor([[0, 1, 2], [3, 4, 5], [0, 0, 4]], dtype=torch.int32, device=cuda)
    c = torch.rand((6, 3), device=cuda).requires_grad_()
    o = torch.rand((6,), device=cuda).requires_grad_()
    image, depthmap = trigrad_amd.render(v, idx, c, o, 70, 50, 16, 16, 1 / 256, False, m["per_pixel_sort"], m["max_layers"])
    assert float(image[..., :3].abs().max()) == 0.0 and float(image[..., 3].min()) == 1.0 and torch.isinf(depthmap).all()
    (image.sum() + torch.where(torch.isinf(depthmap), torch.zeros_like(depthmap), depthmap).sum()).backward()
    for g in (v.grad, c.grad, o.grad):
        assert float(g.abs().max()) == 0.0


@pytest.mark.parametrize("mode", ["A_default", "A_40_layers", "B_unlimited"])
@pytest.mark.parametrize("n_triangles,size,tile", [(1, 16, 16), (2048, 16, 16), (2049, 16, 16), (4097, 40, 16), (900, 256, 1), (900, 257, 1)])
def test_frame_in_one_call_is_the_frame_stage_by_stage(n_triangles, size, tile, mode, cuda, monkeypatch):
    """The one-call route against the stages with K on the host, at the edges of its rules: one triangle, one list of 2048 and
    2049 entries (what the small segment sort takes), more than one sort tile, 256 and 257 tile columns (the staged route's).
    The second run is the torch module's, the third has key buffers that are far too small: empty lists first, then the frame
    again."""
    import torch
    import trigrad_amd
    from trigrad_amd import _C
    import scenes as S
    scene = S.random_soup(n_triangles, size, size, seed=n_triangles, sigma_px=6.0, varying_w=True)
    d = to_device(scene, cuda)
    m = MODES[mode]
    key = (cuda.index, n_triangles, size, size, tile, tile)
    gi = torch.from_numpy(np.random.default_rng(1).standard_normal((size, size, 4)).astype(np.float32)).to(cuda)

    def run():
        leaves = [d[k].clone().requires_grad_() for k in ("vertices", "colors", "opacities")]
        image, depth = trigrad_amd.render(leaves[0], d["indices"], *leaves[1:], size, size, tile, tile, 1 / 256, False,
                                          m["per_pixel_sort"], m["max_layers"])
        return [image.detach(), depth.detach(), *torch.autograd.grad((image,), leaves, (gi,))]

    _C._frame_key_hints.pop(key, None)
    got = [run()]
    supported = _C.frame_supported(d["vertices"], size, size, tile, tile)
    assert supported == (size // tile <= 256) and (key in _C._frame_key_hints) == supported
    if supported:
        K = _C._frame_key_hints[key]
        got.append(run())  # by the torch module
        _C._frame_key_hints[key] = 0
        _C._module().forget()
        monkeypatch.setattr(_C, "_round_capacity", lambda n: max(n, 1))
        got.append(run())
        assert _C._frame_key_hints[key] == K
    monkeypatch.setattr(_C, "ONE_CALL_FRAME", False)
    want = run()
    for one in got:
        assert torch.equal(one[0], want[0]) and torch.equal(one[1], want[1])
        for a, b in zip(one[2:], want[2:]):
            # sums of float32 terms in another order: two rounding steps of the largest sum
            assert float((a - b).abs().max()) <= 1e-5 * float(b.abs().max()) + 1e-6


def _stacks_with_a_nan_depth(with_nan):
    """Three 16 x 16 tiles with a stack of 40 half-tile triangles each, all of one shape (a pixel is covered by
    a whole stack or by none of it); the last one of the middle stack has a NaN depth."""
    W, H, n = 48, 16, 40
    vertices, tile_of = [], []
    for tile in range(3):
        for k in range(n - (tile == 1 and not with_nan)):
            x = 16 * tile + np.array([1.0, 15.0, 1.0])
            y = np.array([1.0, 1.0, 15.0])
            z = np.full(3, np.nan if tile == 1 and k == n - 1 else 0.1 + 0.2 * k)
            vertices.append(np.stack([2 * x / W - 1, 2 * y / H - 1, z, np.full(3, 1 / (0.1 + 0.2 * k))], axis=-1))
            tile_of.append(tile)
    m = len(vertices)
    v = np.concatenate(vertices).astype(np.float32)
    colors = np.random.default_rng(18).uniform(0, 1, (3 * 3 * n, 3)).astype(np.float32)
    opacities = np.full(3 * 3 * n, 0.004, np.float32)
    keep = np.arange(3 * 3 * n).reshape(-1, 3)
    if not with_nan:
        keep = np.delete(keep, 2 * n - 1, axis=0)
    scene = dict(vertices=v, indices=np.arange(3 * m, dtype=np.int32).reshape(m, 3), colors=colors[keep.ravel()],
                 opacities=opacities[keep.ravel()], width=W, height=H)
    return scene, np.repeat(tile_of, 3)


@pytest.mark.parametrize("max_layers", [41, 500])
@pytest.mark.parametrize("one_call", [True, False])
def test_nan_depth_stays_inside_its_rows_of_the_order_pool(one_call, max_layers, cuda, oracle, monkeypatch):
    """A NaN depth has a pixel's list blended again and again: the image is the oracle's, but the order pool has one row per
    list entry.  Nothing is written behind the pool, and the gradients of the other tiles' triangles are those of the same
    frame without the NaN triangle."""
    import torch
    import trigrad_amd
    from trigrad_amd import _C
    monkeypatch.setattr(_C, "ONE_CALL_FRAME", one_call)
    behind = []

    def pool_and_sentinels(n_keys, n_triangles, tile_width, tile_height, device):
        words = int(trigrad_amd._lib.load(32).tg_order_pool_words(n_keys, n_triangles, tile_width, tile_height))
        rows = torch.full((words + (max_layers + 1) * tile_width * tile_height,), 0x5a5a, dtype=torch.int16, device=device)
        behind.append(rows[words:])
        return rows[:words]

    monkeypatch.setattr(_C, "_order_pool", pool_and_sentinels)
    mode = dict(per_pixel_sort=True, max_layers=max_layers)
    scene, tile_of = _stacks_with_a_nan_depth(True)
    _, want, got, _ = _forward_both(scene, 16, 16, mode, cuda, oracle, thr=0.0)
    assert np.diff(want["offsets"]).tolist() == [40, 40, 40] and want["ends"].max() == max_layers > 40
    _check_forward("NaN depth", want, got, (16, 16))
    for sentinels in behind:
        assert int((sentinels != 0x5a5a).sum()) == 0
    assert bool(behind) != one_call

    clean, clean_tile = _stacks_with_a_nan_depth(False)
    W, H = scene["width"], scene["height"]
    gi = np.random.default_rng(3).standard_normal((H, W, 4)).astype(np.float32)
    reference = oracle.render(clean["vertices"], clean["indices"], clean["colors"], clean["opacities"], W, H, 16, 16, 0.0, True, max_layers)
    wanted = oracle.render_backward(gi, np.zeros((H, W), np.float32), clean["vertices"], clean["indices"], clean["colors"],
                                    clean["opacities"], reference, W, H, 16, 16, True, max_layers, magnitudes=True)
    d = to_device(scene, cuda)
    leaves = [d[k].clone().requires_grad_() for k in ("vertices", "colors", "opacities")]
    for _ in range(2):  # the second one is the torch module's
        image, _ = trigrad_amd.render(leaves[0], d["indices"], *leaves[1:], W, H, 16, 16, 0.0, False, True, max_layers)
        grads = torch.autograd.grad((image,), leaves, (torch.from_numpy(gi).to(cuda),))
        for label, g, w, mag in zip(("grad_vertices", "grad_colors", "grad_opacities"), grads, wanted[:3], wanted[3:]):
            g = g.cpu().numpy()
            assert np.isfinite(g).all()
            assert_gradients_close(f"beside a NaN depth: {label}", g[tile_of != 1], w[clean_tile != 1], mag[clean_tile != 1])


def test_pairs_of_an_expired_scan_are_not_sorted(cuda, monkeypatch):
    """A wait of the scan that expired leaves a K that does not belong to the digit totals: the lists are empty, nothing is
    moved, and the image is NaN.  No wait is provoked: the state word is set between the binning and the lists."""
    import struct
    import torch
    from trigrad_amd import _C, _lib
    import scenes as S
    d = to_device(S.config(0), cuda)
    args = (d["vertices"], d["indices"], d["colors"], d["opacities"], 256, 256, 16, 16, 1 / 256, True, 32)
    lib = _lib.load(32)
    in_phases, forged = lib.tg_frame_forward, []

    def forward(call):
        words = struct.unpack_from("<11Q3q", call)
        state, (epoch, state_bytes, phases) = words[8], words[11:]
        code = in_phases(call)
        if phases == _C._FRAME_BIN:
            memory = next(st["frame"] for st in _C._frame_states.values() if st["frame"].data_ptr() == state)
            forged.append(memory[state_bytes + 4:state_bytes + 8].view(torch.int32).fill_(epoch))
        return code

    monkeypatch.setattr(lib, "tg_frame_forward", forward)
    monkeypatch.setattr(_C, "_FRAME_UNTIMED", ((_C._FRAME_BIN, None), (_C._FRAME_LISTS | _C._FRAME_RASTER | _C._FRAME_WAIT, None)))
    try:
        image, depthmap, kept, frame = _C.frame_forward(*args)
        with pytest.raises(RuntimeError, match="look-back wait timed out"):
            frame.status.verify()
    finally:
        _C.force_tickets(False)
        _C._module().forget()
        for word in forged:
            word.zero_()
    assert len(forged) == 1 and frame.n_keys > 0
    assert torch.isnan(image).all() and torch.isnan(depthmap).all()
    *_, offsets, _, _, _ = _C._frame_results(image, depthmap, kept, frame, 256, 256, 16, 16, True, 32, d["indices"].shape[0])
    assert int(offsets.abs().max()) == 0
    ids = kept[frame.plan.at["ids"]:frame.plan.at["ids"] + 4 * frame.n_keys].view(torch.int32)
    binned = _C.bin_frame(d["vertices"], d["indices"], 256, 256, 16, 16)
    assert torch.equal(ids, binned["values"][:frame.n_keys])  # in emission order still


def test_exceptions_of_a_known_frame_keep_their_type(cuda):
    """What fails inside a frame that the torch module renders arrives as it does from the Python function: an allocation as
    OutOfMemoryError, a saved-tensor hook's own exception as itself.  The frame after it is rendered as ever."""
    import torch
    import trigrad_amd
    import scenes as S
    d = to_device(S.random_soup(50, 700, 600, seed=2), cuda)
    leaf = d["vertices"].clone().requires_grad_()

    def frame():
        return trigrad_amd.render(leaf, d["indices"], d["colors"], d["opacities"], 700, 600)

    want = [frame()[0].detach() for _ in range(2)][-1]  # the module knows the kind now
    torch.cuda.synchronize()
    torch.cuda.empty_cache()
    allowed = (torch.cuda.memory_reserved() + (1 << 20)) / torch.cuda.get_device_properties(cuda).total_memory
    try:
        torch.cuda.set_per_process_memory_fraction(allowed)
        with pytest.raises(torch.OutOfMemoryError):
            frame()
    finally:
        torch.cuda.set_per_process_memory_fraction(1.0)
    assert torch.equal(frame()[0].detach(), want)

    class Refused(Exception):
        pass

    def pack(t):
        raise Refused("not this one")

    with torch.autograd.graph.saved_tensors_hooks(pack, lambda t: t):
        with pytest.raises(Refused, match="not this one"):
            frame()
    assert torch.equal(frame()[0].detach(), want)


@pytest.mark.parametrize("by_module", [True, False])
def test_status_words_of_a_failed_call_outlive_its_kernels(by_module, cuda):
    """A call that fails when its kernels are launched already: the words they write in pinned memory are given back only
    when the stream is done with them.  The failure is the test's: the library's call is made, then its code replaced."""
    import ctypes as C
    import torch
    from trigrad_amd import _C, _lib
    import trigrad_amd
    import scenes as S
    d = to_device(S.random_soup(60, 80, 64, seed=2), cuda)
    args = (d["vertices"], d["indices"], d["colors"], d["opacities"], 80, 64)
    want = [trigrad_amd.render(*args)[0] for _ in range(2)][-1]
    lib = _lib.load(32)
    real, stream, busy = lib.tg_frame_forward, torch.cuda.current_stream(), []
    address = lambda f: C.cast(f, C.c_void_p).value

    def bind(forward):
        _C._module().bind(address(forward), *[address(getattr(lib, name)) for name in (
            "tg_frame_backward", "tg_frame_wait", "tg_force_tickets", "tg_last_error")], _C._key_count_hint)

    @C.CFUNCTYPE(C.c_int, C.c_void_p)
    def failing(call):
        phases = C.c_int64.from_address(call + 104)
        phases.value &= ~_C._FRAME_WAIT
        torch.cuda._sleep(200_000_000)  # about a tenth of a second in front of the kernels
        real(call)
        busy.append(not stream.query())
        return -1

    try:
        if by_module:
            bind(failing)
        else:
            _C._module().forget()
            lib.tg_frame_forward = lambda call: failing(C.addressof(call))
        with pytest.raises(RuntimeError, match="tg_frame_forward failed with code -1"):
            trigrad_amd.render(*args)
        assert busy == [True] and stream.query()
    finally:
        lib.tg_frame_forward = real
        bind(real)
        torch.cuda.synchronize()
    for _ in range(2):
        assert torch.equal(trigrad_amd.render(*args)[0], want)


@pytest.mark.parametrize("route", ["module", "one call", "staged"])
def test_frames_after_a_refused_one(route, cuda, monkeypatch):
    """Vertices off a 16-byte boundary are refused before the binning's scan runs; the state it keeps from call to call is
    in step again for the frames that follow."""
    import torch
    import trigrad_amd
    from trigrad_amd import _C
    import scenes as S
    monkeypatch.setattr(_C, "ONE_CALL_FRAME", route != "staged")
    scene = S.random_soup(900, 200, 150, seed=2)
    d = to_device(scene, cuda)
    n = d["vertices"].shape[0]
    shifted = torch.empty((4 * n + 1,), device=cuda)[1:].view(n, 4).copy_(d["vertices"])

    def frame(vertices):
        if route == "one call":
            _C._module().forget()
        return trigrad_amd.render(vertices, d["indices"], d["colors"], d["opacities"], 200, 150)[0]

    want = [frame(d["vertices"]) for _ in range(3)][-1]
    for _ in range(2):  # either parity of the calls so far
        frame(d["vertices"])
        with pytest.raises(RuntimeError, match="16-byte aligned"):
            frame(shifted)
        state = [st["frame"] for st in _C._frame_states.values()]
        if route != "module":
            assert any(int(memory.abs().max()) == 0 for memory in state)
        for _ in range(3):
            assert torch.equal(frame(d["vertices"]), want)
    trigrad_amd.verify_frames()


@pytest.mark.parametrize("mode", ["A_default", "A_unlimited", "B_unlimited"])
@pytest.mark.parametrize("around", [29, 2030, 65530])
def test_frames_whose_number_of_triangles_changes_share_plans(around, mode, cuda, monkeypatch):
    """A camera that moves through a split scene has another number of triangles in every frame: such frames share plans (up
    to a sixteenth more triangles), so all but the first of a bucket are the torch module's; every frame is the staged
    route's.  The counts pass the edges of buckets, of 32 triangles and of 16-bit list positions."""
    import torch
    import trigrad_amd
    from trigrad_amd import _C
    import scenes as S
    W, H, m = 150, 100, MODES[mode]
    d = to_device(S.random_soup(around + 40, W, H, seed=3, sigma_px=3.0), cuda)
    gi = torch.from_numpy(np.random.default_rng(1).standard_normal((H, W, 4)).astype(np.float32)).to(cuda)
    counts = [around + k for k in (7, 0, 3, 20, 6, 11, 1, 9, 5, 33, 4, 2)]

    def run(n):
        leaves = [d[k][:3 * n].clone().requires_grad_() for k in ("vertices", "colors", "opacities")]
        image, depth = trigrad_amd.render(leaves[0], d["indices"][:n], *leaves[1:], W, H, 16, 16, 1 / 256, False, m["per_pixel_sort"],
                                          m["max_layers"])
        return [image.detach(), depth.detach(), *torch.autograd.grad((image,), leaves, (gi,))]

    _C._module().forget()
    by_python, in_python = [], _C.frame_forward
    monkeypatch.setattr(_C, "frame_forward", lambda *a, **k: by_python.append(a[1].shape[0]) or in_python(*a, **k))
    got = [run(n) for n in counts]
    buckets = {_C._round_count(n) for n in counts}
    assert len(by_python) == len(buckets) and {_C._round_count(n) for n in by_python} == buckets
    assert len(buckets) < len(counts) or around < 32
    monkeypatch.setattr(_C, "ONE_CALL_FRAME", False)
    for n, one in zip(counts, got):
        want = run(n)
        assert torch.equal(one[0], want[0]) and torch.equal(one[1], want[1])
        for a, b in zip(one[2:], want[2:]):
            # sums of float32 terms in another order: two rounding steps of the largest sum
            assert float((a - b).abs().max()) <= 1e-5 * float(b.abs().max()) + 1e-6


def test_key_buffers_of_a_size_seen_before(cuda):
    """A number of triangles not seen before takes its key buffers from the last frame of the image and tile size, not from a
    guess, and the tables of such numbers stay bounded."""
    import trigrad_amd
    from trigrad_amd import _C
    import scenes as S
    W, H = 410, 300
    d = to_device(S.random_soup(5000, W, H, seed=3, sigma_px=1.0), cuda)
    made = []
    for n in range(4000, 5000, 3):
        image, depth, kept, frame = _C.frame_forward(d["vertices"], d["indices"][:n], d["colors"], d["opacities"], W, H, 16, 16, 1 / 256,
                                                     True, 32)
        made.append((frame.n_keys, frame.plan.capacity))
    assert made[0][1] == 3 * 4000 + 65536
    few = _C.frame_forward(d["vertices"], d["indices"][:1200], d["colors"], d["opacities"], W, H, 16, 16, 1 / 256, True, 32)[3]
    assert few.plan.capacity == 3 * 1200 + 65536  # another scene: its keys per triangle say nothing
    assert all(keys <= capacity <= 1.3 * keys + 2048 for keys, capacity in made[1:])
    for table in (_C._frame_key_hints, _C._frame_size_hints, _C._frame_plans):
        assert len(table) <= _C._MAX_REMEMBERED
    trigrad_amd.verify_frames()


@pytest.mark.parametrize("keep", [True, False])
@pytest.mark.parametrize("n_triangles", [40, 3000])
def test_order_pool_of_a_first_frame_is_made_for_its_keys(n_triangles, keep, cuda, oracle, monkeypatch):
    """A frame without a layer limit keeps a row of a tile's pixels per key.  The first one of its kind and size counts its
    keys before it takes the memory; ORDER_POOL_MAX_BYTES = 0 keeps nothing and gives the same gradients."""
    import torch
    import trigrad_amd
    from trigrad_amd import _C
    import scenes as S
    W, H = 223, 117 + n_triangles % 7  # of no other test
    scene = S.random_soup(n_triangles, W, H, seed=4, sigma_px=7.0, opacity=(0.02, 0.2))
    d = to_device(scene, cuda)
    if not keep:
        monkeypatch.setattr(_C, "ORDER_POOL_MAX_BYTES", 0)
    for table in (_C._frame_key_hints, _C._frame_size_hints):
        for key in [k for k in table if k[-4:-2] == (W, H)]:
            del table[key]
    args = (d["vertices"], d["indices"], d["colors"], d["opacities"], W, H, 16, 16, 1 / 256, True, n_triangles + 1)
    image, depthmap, kept, frame = _C.frame_forward(*args)
    pool = _C._round_capacity(frame.n_keys) * 256 * 2
    assert frame.plan.capacity == (_C._round_capacity(frame.n_keys) if keep else 3 * n_triangles + 65536)
    assert pool < kept.numel() < pool + 400_000 + 44 * n_triangles + 28 * W * H if keep else kept.numel() < pool + 700_000
    want = oracle.render(*(scene[k] for k in ("vertices", "indices", "colors", "opacities")), W, H, 16, 16, 1 / 256, True, n_triangles + 1)
    assert np.array_equal(image.cpu().numpy(), want["image"])
    gi, gd = _grad_inputs(scene, 5, False)
    wanted = oracle.render_backward(gi, gd, *(scene[k] for k in ("vertices", "indices", "colors", "opacities")), want, W, H, 16, 16, True,
                                    n_triangles + 1, magnitudes=True)
    leaves = [d[k].clone().requires_grad_() for k in ("vertices", "colors", "opacities")]
    for _ in range(2):
        image, _ = trigrad_amd.render(leaves[0], d["indices"], *leaves[1:], W, H, max_layers=-1)
        grads = torch.autograd.grad((image,), leaves, (torch.from_numpy(gi).to(cuda),))
        for label, g, w, mag in zip(("grad_vertices", "grad_colors", "grad_opacities"), grads, wanted[:3], wanted[3:]):
            assert_gradients_close(f"pool of a first frame: {label}", g.cpu().numpy(), w, mag)


@pytest.mark.parametrize("mode", ["A_default", "A_40_layers", "A_unlimited", "B_3_layers", "B_unlimited"])
@pytest.mark.parametrize("n,sigma,tw,th", [
    (1023, 0.7, 16, 16), (1024, 0.7, 16, 16),  # at the rule's edge
    (1025, 0.7, 16, 16), (1281, 5.0, 16, 16),  # a block of one entry; triangles that cover most of the tile
    (2500, 2.0, 32, 32), (1500, 2.0, 24, 16),  # the tile's squares are several workgroups'
    (1100, 3.0, 20, 13),  # a wave's pixels are no square
])
def test_long_tiles_shared_out(n, sigma, tw, th, mode, cuda, oracle):
    """Tiles whose lists of 1024 entries and more are four waves' work: one list of n next to short ones, forward and backward,
    with lists that are longer than the layers a selection takes and partial tiles on both sides."""
    import torch
    import scenes as S
    from trigrad_amd import _C
    width, height = 3 * tw - 5, 2 * th - 3
    scene = S.random_soup(n + 60, tw, th, seed=n, sigma_px=sigma, opacity=(0.02, 0.2), varying_w=True)
    v = scene["vertices"].reshape(n + 60, 3, 4)
    rng = np.random.default_rng(n)
    xy = rng.uniform(-0.7, 0.7, (2 * n, 1, 2)) + rng.standard_normal((2 * n, 3, 2)) * sigma * 2.0 / np.array([tw, th])
    xy = np.clip(xy, -0.98, 0.98)
    edges = xy[:, 1:] - xy[:, :1]
    xy = xy[np.abs(np.linalg.det(edges)) > 1e-3][:n]  # a triangle without an area is in no list
    v[:n, :, :2] = (xy + 1.0) * np.array([tw / width, th / height]) - 1.0  # into the first tile
    v[n:, :, 0] = v[n:, :, 0] * 0.3 + 0.6  # the others beside it
    scene.update(width=width, height=height)
    m = MODES[mode]
    d, want, got, ml = _forward_both(scene, tw, th, m, cuda, oracle, frames=3)
    lengths = np.diff(want["offsets"])
    assert lengths[0] == n and lengths[1:].max() < 100
    assert _long_tile_limit(scene, tw, th, m["per_pixel_sort"], lengths.sum()) == 1024
    if not m["per_pixel_sort"]:
        assert np.array_equal(_shared_out(got, want, tw, th), lengths >= 1024)
    _check_forward(f"long tile {n}/{tw}x{th}/{mode}", want, got, (th, tw))
    gi, gd = _grad_inputs(scene, 9, True)
    wanted = oracle.render_backward(gi, gd, scene["vertices"], scene["indices"], scene["colors"], scene["opacities"], want, width, height,
                                    tw, th, m["per_pixel_sort"], ml, literal=False, magnitudes=True)
    image, depthmap, weights, sorted_ids, offsets, bary, ends, _, resume = got
    out = _C.render_backward(torch.from_numpy(gi).to(cuda), torch.from_numpy(gd).to(cuda), d["vertices"], d["indices"], d["colors"],
                             d["opacities"], sorted_ids, offsets, bary, image, depthmap, weights, ends, width, height, tw, th, 1 / 256,
                             m["per_pixel_sort"], ml, resume=resume)
    for label, g, w, mag in zip(("grad_vertices", "grad_colors", "grad_opacities"), out, wanted[:3], wanted[3:]):
        assert_gradients_close(f"long tile {n}/{mode}: {label}", g.cpu().numpy(), w, mag)


@pytest.mark.parametrize("width,per_pixel_sort", [(1024, True), (1024, False), (512, False)])
def test_long_tiles_match_the_other_route(width, per_pixel_sort, cuda, monkeypatch):
    """Some 1200 tiles (of 4096) with lists of 1024 entries and more, shared out in per-pixel order; in tile order the first of
    them are started first, and with 1024 tiles the long ones are shared out there too.  Some depths are NaN: in per-pixel order such a candidate ends a selection, so
    what is kept depends on the order of looking.  The frame is that of the stage-by-stage route, which knows no long tile."""
    import torch
    import scenes as S
    from trigrad_amd import _C
    side = 36 if width == 1024 else 10  # tiles to a side of the crowded corner
    n = side * side * 1250
    soup = S.random_soup(n, width, width, seed=8, sigma_px=0.6, opacity=(0.1, 0.6))
    v = soup["vertices"].reshape(n, 3, 4).copy()
    v[: n * 97 // 100, :, :2] = (v[: n * 97 // 100, :, :2] + 1.0) * (side * 16 / width) - 1.0
    v[::5003, 1, 2] = np.nan
    d = to_device(dict(soup, vertices=v.reshape(-1, 4)), cuda)
    args = (d["vertices"], d["indices"], d["colors"], d["opacities"], width, width, 16, 16, 1 / 256, True, per_pixel_sort, 32)
    for _ in range(3):  # the first frame's buffers are made for a guess of K, and what is long depends on them
        got = _C.render_forward(*args)
    lengths = got[4][1:] - got[4][:-1]
    assert int((lengths >= 1024).sum()) > (1024 if width == 1024 else 64)
    monkeypatch.setattr(_C, "ONE_CALL_FRAME", False)
    want = _C.render_forward(*args)
    for i in (0, 1, 2, 3, 4, 5, 6):
        assert torch.equal(got[i].view(torch.int32), want[i].view(torch.int32)), i


@pytest.mark.parametrize("tw,width,entries,layers,crowded,per_tile", [
    *[(16, 512, 4, 32, crowded, 1100) for crowded in (1, 31, 33, 150)],  # with 23 places a candidate list
    *[(16, 320, 4, 32, crowded, 1100) for crowded in (1, 40, 150)],  # with all of them
    *[(16, 320, 700, 40, crowded, 4000) for crowded in (1, 40)],  # with depth bounds, where they do not help
    *[(24, 384, 4, -1, crowded, 1100) for crowded in (1, 40, 150)],  # a tile is two workgroups
])
def test_tiles_that_are_done_help_with_the_long_ones(tw, width, entries, layers, crowded, per_tile, cuda, monkeypatch):
    """Up to 1024 workgroups, of which those of short lists draw the long tiles' work by a counter that ends at zero: the raster
    phase is run twice on the same lists, into another image each time, and both are the stage-by-stage route's.  From fewer long
    tiles than there are workgroups in front of the others (one item for four of them) to several items for each."""
    import ctypes as C
    import struct
    import torch
    import scenes as S
    from trigrad_amd import _C, _lib
    columns, rows = width // tw, width // 16
    tiles, rng = columns * rows, np.random.default_rng(crowded)
    soup = S.random_soup(entries * tiles + crowded * per_tile, width, width, seed=crowded, sigma_px=1.5, opacity=(0.02, 0.3))
    v = soup["vertices"].reshape(-1, 3, 4).copy()
    at = rng.choice(tiles, crowded, replace=False)[np.arange(crowded * per_tile) % crowded]
    corner = np.stack([at % columns * tw, at // columns * 16], axis=-1)[:, None]
    pixels = corner + rng.uniform(0.3, 15.7, (crowded * per_tile, 3, 2))
    v[: crowded * per_tile, :, :2] = pixels / width * 2.0 - 1.0
    d = to_device(dict(soup, vertices=v.astype(np.float32).reshape(-1, 4)), cuda)
    n = d["indices"].shape[0]
    args = (d["vertices"], d["indices"], d["colors"], d["opacities"], width, width, tw, 16, 1 / 256, True, layers if layers > 0 else n + 1)
    for _ in range(2):  # the first frame's buffers are made for a guess of K, and what is long depends on them
        frame = _C.frame_forward(*args)[3]
    lib = _lib.load(32)
    real, others = lib.tg_frame_forward, []

    def forward(call):
        other = torch.zeros((width, width, 4), device=cuda)
        words = list(struct.unpack_from("<14Q", call))
        struct.pack_into("<Q", call, 4 * 8, other.data_ptr())
        struct.pack_into("<Q", call, 13 * 8, _C._FRAME_BIN | _C._FRAME_LISTS | _C._FRAME_RASTER)
        assert real(call) == 0
        struct.pack_into("<Q", call, 4 * 8, words[4])
        struct.pack_into("<Q", call, 13 * 8, _C._FRAME_RASTER | _C._FRAME_WAIT)
        others.append(other)
        return real(call)

    monkeypatch.setattr(lib, "tg_frame_forward", forward)
    image, depthmap, kept, frame = _C.frame_forward(*args)
    monkeypatch.setattr(lib, "tg_frame_forward", real)
    frame.status.verify()
    *_, offsets, _, _, _ = _C._frame_results(image, depthmap, kept, frame, width, width, tw, 16, True, args[-1], n)
    lengths = (offsets[1:] - offsets[:-1]).cpu().numpy()
    scene = dict(width=width, height=width, indices=d["indices"])
    assert (lengths >= _long_tile_limit(scene, tw, 16, True, frame.n_keys)).sum() == crowded
    assert tiles * -(-tw // 16) <= 1024 and (lengths.mean() >= 512) == (entries == 700)
    monkeypatch.setattr(_C, "ONE_CALL_FRAME", False)
    want = _C.render_forward(*args[:9], True, True, args[-1])
    assert len(others) == 1
    for got in (image, others[0]):
        assert torch.equal(got.view(torch.int32), want[0].view(torch.int32))


@pytest.mark.parametrize("layers", [5, 23, 24, 27, 32, 40, -1])
@pytest.mark.parametrize("n", [22, 23, 24, 25, 31, 32, 33, 60])
@pytest.mark.parametrize("size,tiles,places", [
    (24, [(16, 16), (8, 8), (8, 16)], 32),
    (400, [(8, 8)], 23),  # one wave to a workgroup
    (460, [(16, 16), (8, 16), (12, 16)], 23),  # four waves, two and three
])
def test_candidate_lists_around_their_places_in_lds(size, tiles, places, n, layers, cuda, oracle):
    """A pixel's first 23 candidates are kept in LDS, the others up to 32 in registers -- or all in LDS, where that takes no more
    generations of workgroups: n triangles over every pixel, tilted, so that their order at a pixel is not the list's, a third of
    them at equal depths, and layers that end inside either part."""
    import scenes as S
    from trigrad_amd import _lib
    rng = np.random.default_rng(100 * n + layers)
    z = rng.uniform(1.0, 5.0, (n, 1)) * rng.uniform(0.5, 1.5, (n, 3))
    z[::3] = rng.choice([2.0, 3.0], (z[::3].shape[0], 1))
    xy = np.array([[-9.0, -9.0], [9.0, -9.0], [0.0, 16.0]]) * rng.uniform(0.9, 1.1, (n, 1, 1))
    vertices = np.concatenate([xy, z[:, :, None], 1.0 / z[:, :, None]], axis=-1).astype(np.float32).reshape(-1, 4)
    scene = dict(S.random_soup(n, size, size, seed=n, opacity=(0.02, 0.3)), vertices=vertices)
    mode = dict(per_pixel_sort=True, max_layers=layers)
    for tw, th in tiles:
        assert _lib.load(32).tg_candidate_places(size, size, tw, th) == places
        _, want, got, _ = _forward_both(scene, tw, th, mode, cuda, oracle)
        assert int(want["ends"].max()) == min(n, layers if layers > 0 else n)
        _check_forward(f"{n} candidates, {layers} layers, tiles of {tw} x {th}", want, got, (th, tw))


@pytest.mark.parametrize("width,height", [(16, 16), (70, 45), (1024, 1024), (1040, 1024)])
@pytest.mark.parametrize("n", [1, 40, 700, 1020, 1030, 2040, 2060, 4090, 4100, 6200, 8200])
def test_frames_with_few_keys_have_the_other_routes_lists(n, width, height, cuda, monkeypatch):
    """Frames whose buffers are for up to 8192 keys (6372 of the frame) and 4096 tiles are sorted by one workgroup, by tile, and by
    depth as well up to 2048 (911): around the numbers of keys a thread takes, with equal depths (the order is then the triangles'),
    tiles without a key, and a tile whose list is a long one.  Lists and image are those of the stage-by-stage route."""
    import torch
    import scenes as S
    from trigrad_amd import _C
    soup = S.random_soup(n, width, height, seed=n, sigma_px=1.0, opacity=(0.1, 0.6))
    v = soup["vertices"].reshape(n, 3, 4).copy()
    v[::3, :, 2:] = (2.0, 0.5)
    if n > 2000:
        v[: n // 2, :, :2] = v[: n // 2, :, :2] * (4.0 / max(width, height)) + 0.13  # half of them in a tile or two
    d = to_device(dict(soup, vertices=v.reshape(-1, 4)), cuda)
    args = (d["vertices"], d["indices"], d["colors"], d["opacities"], width, height, 16, 16, 1 / 256, True, True, 32)
    for _ in range(3):  # the first frame's buffers are made for a guess of K, and the route goes by them
        got = _C.render_forward(*args)
    monkeypatch.setattr(_C, "ONE_CALL_FRAME", False)
    want = _C.render_forward(*args)
    for i in (0, 1, 2, 3, 4, 5, 6):
        assert torch.equal(got[i].view(torch.int32), want[i].view(torch.int32)), i


@pytest.mark.parametrize("width,height", [(16, 16), (1024, 1024), (1040, 1024)])
@pytest.mark.parametrize("n_keys,capacity", [(911, 2048), (912, 3072), (6372, 8192), (6373, 9216)])
def test_frames_with_few_keys_at_the_edges_of_their_rule(n_keys, capacity, width, height, cuda, monkeypatch):
    """Every triangle is in one tile, so the number of keys is theirs: the last and the first one on either side of a buffer of
    2048 keys (sorted by depth by the one workgroup) and of 8192 (by tile), with 1, 4096 and 4160 tiles."""
    import torch
    import scenes as S
    from trigrad_amd import _C
    soup = S.random_soup(n_keys, 16, 16, seed=n_keys, sigma_px=2.0, opacity=(0.02, 0.3))
    rng = np.random.default_rng(n_keys)
    v = soup["vertices"].reshape(n_keys, 3, 4).copy()
    v[:, :, :2] = rng.uniform(-0.9, 0.9, (n_keys, 3, 2))  # of a tile
    size, tiles = np.array([width, height]), np.array([width, height]) // 16
    at = rng.integers(0, tiles, (n_keys, 1, 2)) if width > 16 else np.zeros((n_keys, 1, 2))
    at[: n_keys // 2] = tiles // 2  # half of them in one
    v[:, :, :2] = ((v[:, :, :2] + 1.0) * 8.0 + 16.0 * at) / size * 2.0 - 1.0
    v[::3, :, 2:] = (2.0, 0.5)  # equal depths
    d = to_device(dict(soup, vertices=v.astype(np.float32).reshape(-1, 4)), cuda)
    args = (d["vertices"], d["indices"], d["colors"], d["opacities"], width, height, 16, 16, 1 / 256, True, True, 32)
    for _ in range(3):  # the first frame's buffers are made for a guess of K, and the route goes by them
        got = _C.render_forward(*args)
    assert int(got[4][-1]) == n_keys and _C._round_capacity(n_keys) == capacity
    monkeypatch.setattr(_C, "ONE_CALL_FRAME", False)
    want = _C.render_forward(*args)
    for i in (0, 1, 2, 3, 4, 5, 6):
        assert torch.equal(got[i].view(torch.int32), want[i].view(torch.int32)), i


@pytest.mark.parametrize("layers,tile_entries", [(15, 100), (16, 100), (16, 40)])
@pytest.mark.parametrize("columns,rows", [(1, 1), (15, 1), (16, 1), (17, 1), (43, 3), (19, 27)])
def test_gradients_whichever_tiles_an_xcd_takes(columns, rows, layers, tile_entries, cuda, oracle):
    """The saved-order backward kernel deals the tiles out to the XCDs in eighths of them, or in sixteenths from either end where
    there are 16 layers and 96 keys a tile: numbers of tiles around sixteen and with a remainder, every tile with triangles of its
    own and shared ones."""
    import torch
    import scenes as S
    import trigrad_amd
    width, height = 16 * columns - 3, 16 * rows - 5
    n = tile_entries * columns * rows
    scene = S.random_soup(n, width, height, seed=n + layers, sigma_px=3.0, opacity=(0.1, 0.5), varying_w=True)
    want = oracle.render(scene["vertices"], scene["indices"], scene["colors"], scene["opacities"], width, height, 16, 16, 1 / 256, True, layers)
    assert (want["offsets"][-1] >= 96 * columns * rows) == (tile_entries == 100)
    gi, gd = _grad_inputs(scene, 4, True)
    wanted = oracle.render_backward(gi, gd, scene["vertices"], scene["indices"], scene["colors"], scene["opacities"], want, width, height,
                                    16, 16, True, layers, literal=False, magnitudes=True)
    d = to_device(scene, cuda)
    leaves = [d[k].clone().requires_grad_() for k in ("vertices", "colors", "opacities")]
    for _ in range(2):  # a first frame, and one whose number of keys is known
        outputs = trigrad_amd.render(leaves[0], d["indices"], *leaves[1:], width, height, max_layers=layers)
        out = torch.autograd.grad(outputs, leaves, (torch.from_numpy(gi).to(cuda), torch.from_numpy(gd).to(cuda)))
        for label, g, w, mag in zip(("grad_vertices", "grad_colors", "grad_opacities"), out, wanted[:3], wanted[3:]):
            assert_gradients_close(f"{columns}x{rows} tiles, {layers} layers: {label}", g.cpu().numpy(), w, mag)


@pytest.mark.parametrize("mode", ["A_default", "A_40_layers", "B_unlimited"])
def test_gradients_of_a_scene_far_away(mode, cuda, oracle):
    """w around 2e-19 (depths around 5e18): the square of an interpolation's denominator is just above the smallest normal number and its
    reciprocal times a gradient of some hundreds is not in float32, but the w gradient is: it has the reciprocal times differences
    of the size of w."""
    import torch
    import scenes as S
    from trigrad_amd import _C
    scene = S.random_soup(300, 70, 45, seed=12, sigma_px=7.0, opacity=(0.2, 0.9))
    v = scene["vertices"].copy()
    rng = np.random.default_rng(12)
    v[:, 2] = rng.uniform(4e18, 6e18, v.shape[0])
    v[:, 3] = 1.0 / v[:, 2]
    scene.update(vertices=v)
    m = MODES[mode]
    d, want, got, ml = _forward_both(scene, 16, 16, m, cuda, oracle)
    _check_forward(f"far away/{mode}", want, got, (16, 16))
    gi, gd = _grad_inputs(scene, 12, False)
    gi = (gi * 300.0).astype(np.float32)
    gd = np.zeros((45, 70), np.float32)
    wanted = oracle.render_backward(gi, gd, scene["vertices"], scene["indices"], scene["colors"], scene["opacities"], want, 70, 45, 16, 16,
                                    m["per_pixel_sort"], ml, literal=False, magnitudes=True)
    assert all(np.isfinite(w).all() for w in wanted) and np.abs(wanted[0][:, 3]).max() > 1e19
    image, depthmap, weights, sorted_ids, offsets, bary, ends, _, resume = got
    out = _C.render_backward(torch.from_numpy(gi).to(cuda), torch.from_numpy(gd).to(cuda), d["vertices"], d["indices"], d["colors"],
                             d["opacities"], sorted_ids, offsets, bary, image, depthmap, weights, ends, 70, 45, 16, 16, 1 / 256,
                             m["per_pixel_sort"], ml, resume=resume)
    for label, g, w, mag in zip(("grad_vertices", "grad_colors", "grad_opacities"), out, wanted[:3], wanted[3:]):
        assert_gradients_close(f"far away/{mode}: {label}", g.cpu().numpy(), w, mag)


@pytest.mark.parametrize("per_pixel_sort", [True, False])
def test_transmittance_is_put_together_by_correctly_rounded_division(per_pixel_sort, cuda):
    """Bit for bit, down to 2^-124 (a threshold of 0): every pixel of 32 x 32 has 52 triangles of its own, whose barycentric coordinates
    at the pixel are 1/4, 1/4 and 1/2 exactly, so a colour gradient is a power of two times (transmittance in front of the fragment
    * opacity), the transmittance being the image's, divided by (1 - opacity) fragment by fragment from the far end."""
    import torch
    from trigrad_amd import _C
    size, layers, scale = 32, 52, np.float32(2.0 ** 60)
    rng = np.random.default_rng(7)
    centre = ((2 * np.arange(size) + 1) / size - 1.0).astype(np.float32)
    h = np.float32(1.0 / 64.0)
    corners = np.array([[-h, -h], [h, -h], [0.0, h]], np.float32)
    v = np.zeros((layers, size, size, 3, 4), np.float32)
    v[..., 0] = centre[None, None, :, None] + corners[:, 0]
    v[..., 1] = centre[None, :, None, None] + corners[:, 1]
    v[..., 2] = (1.0 + np.arange(layers))[:, None, None, None]
    v[..., 3] = 1.0
    opacity = rng.uniform(0.5, 0.97, (layers, size, size)).astype(np.float32)
    n = layers * size * size
    d = [torch.from_numpy(a).to(cuda) for a in (v.reshape(-1, 4), np.arange(3 * n, dtype=np.int32).reshape(n, 3), np.full((3 * n, 3), 0.5, np.float32),
                                                np.repeat(opacity.reshape(-1), 3))]
    got = _C._forward_full(*d, size, size, 16, 16, 0.0, True, per_pixel_sort, n + 1)
    image, depthmap, weights, sorted_ids, offsets, bary, ends, _, resume = got
    assert bool((ends == layers).all())
    gi = torch.zeros((size, size, 4), device=cuda)
    gi[..., :3] = float(scale)
    out = _C.render_backward(gi, torch.zeros((size, size), device=cuda), *d, sorted_ids, offsets, bary, image, depthmap, weights, ends, size,
                             size, 16, 16, 0.0, per_pixel_sort, n + 1, resume=resume)
    grad = out[1].cpu().numpy().reshape(layers, size, size, 3, 3)[..., 0]
    alpha = image.cpu().numpy()[..., 3]
    assert 2.0 ** -124 > alpha.min() and (alpha < 2.0 ** -104).mean() > 0.5
    compared = 0
    for layer in range(layers - 1, -1, -1):
        o = opacity[layer]
        alpha = (alpha / (np.float32(1.0) - o)).astype(np.float32)
        want = (alpha * o).astype(np.float32) * scale
        whole = alpha > 2.0 ** -124  # below, alpha * o and the quotient itself may be denormal
        compared += int(whole.sum())
        differ = (grad[layer].max(-1) != (want * np.float32(0.5))) & whole
        assert not differ.any(), f"layer {layer}: {differ.sum()} of {whole.sum()} pixels, transmittances from {alpha[differ].min():.3g}"
    assert compared > 0.95 * n


@pytest.mark.parametrize("layers", [32, 40])
@pytest.mark.parametrize("n", [1500, 66_000])
def test_selection_of_a_shared_out_tile_is_made_again_by_one_wave(n, layers, cuda, monkeypatch):
    """Every fourth triangle of a tile's list is near and the others are far, so all of a pixel's nearest are candidates of one of
    the four waves that take the list's entries in turn: more than the 23 it has places for (17 where positions take 32 bits), so
    the merge comes to the end of its list and the selection is one wave's.  A triangle's key is its depth in one corner of the
    tile, and its number is its place in the list.  Frame and saved order are those of the stage-by-stage route."""
    import torch
    import scenes as S
    from trigrad_amd import _C, _lib
    size = 512  # 1024 tiles, which run at once with 23 places a candidate list and would not with all of them
    assert _lib.load(32).tg_candidate_places(size, size, 16, 16) == 23
    rng = np.random.default_rng(n)
    corner = np.float32(2.0 ** -9)  # of the tile in row 16 and column 16
    crowd = np.ones((n, 3, 4), np.float32)
    crowd[:, :, :2] = corner
    crowd[:, 1, 0] = crowd[:, 2, 1] = corner + np.float32(2.0 ** -4)
    key = 2.0 + np.arange(n) * 2.0 ** (-10 if n < 2048 else -15)
    crowd[:, 0, 2] = key
    crowd[:, 1:, 2] = (key + rng.integers(0, 64, n) / 64.0 + np.where(np.arange(n) % 4 == 0, 0.0, 64.0))[:, None]
    others = S.random_soup(800, size, size, seed=n, sigma_px=4.0)
    others["vertices"][:, 0] = others["vertices"][:, 0] * 0.4 - 0.55  # not in that tile
    vertices = np.concatenate([crowd.reshape(-1, 4), others["vertices"]])
    scene = dict(vertices=vertices, indices=np.arange(vertices.shape[0], dtype=np.int32).reshape(-1, 3),
                 colors=rng.uniform(0, 1, (vertices.shape[0], 3)).astype(np.float32),
                 opacities=rng.uniform(0.02, 0.08, vertices.shape[0]).astype(np.float32))
    d = to_device(scene, cuda)
    args = (d["vertices"], d["indices"], d["colors"], d["opacities"], size, size, 16, 16, 1 / 256, True, True, layers)
    for _ in range(3):  # the first frame's buffers are made for a guess of K, and what is long depends on them
        got = _C._forward_full(*args)
    capacity = _C._round_capacity(int(got[4][-1]))
    assert n >= max(1024, -(-2 * capacity // 1024))  # the tile is a long one
    tile = 16 * 32 + 16
    assert torch.equal(got[3][int(got[4][tile]):int(got[4][tile + 1])], torch.arange(n, dtype=torch.int32, device=cuda))
    assert int(got[6][256:272, 256:272].max()) == layers
    monkeypatch.setattr(_C, "ONE_CALL_FRAME", False)
    want = _C._forward_full(*args)
    for i in (0, 1, 2, 3, 4, 5, 6):
        assert torch.equal(got[i].view(torch.int32), want[i].view(torch.int32)), i
    if layers == 32:  # in planes
        order = [_C.saved_blend_order(frame[8][3], frame[4], 16, 16) for frame in (got, want)]
        taken = torch.arange(layers, device=cuda)[:, None, None] < got[6]
        assert torch.equal(order[0][taken], order[1][taken])
        near = order[0][:, 258, 258]
        assert bool((near % 4 == 0).all()) and near.unique().numel() == layers


def _with_w(scene, w):
    v = scene["vertices"].copy()
    v[:, 3] = w
    v[:, 2] = 1.0 / np.where(v[:, 3] == 0.0, 1.0, v[:, 3])
    return dict(scene, vertices=v)


def _assert_same_terms(name, got, want):
    """Gradients of the same terms, added in another order: NaNs and infinities in the same places, the others within the rounding of a sum
    of some hundreds of the column's largest (the derivatives of w are 1 / w times those of x and y)."""
    not_finite = ~np.isfinite(want)
    np.testing.assert_array_equal(np.where(not_finite, got, 0), np.where(not_finite, want, 0), err_msg=name)
    for column, (g, w, skip) in enumerate(zip(*(a.reshape(len(a), -1).T for a in (got, want, not_finite)))):
        largest = float(np.abs(w[~skip]).max(initial=0.0))
        assert_close(f"{name}, column {column}", np.where(skip, 0, g), np.where(skip, 0, w), 1e-4, 300 * 2.0 ** -24 * largest + 2.0 ** -126)


@pytest.mark.parametrize("mode", ["A_default", "A_40_layers", "B_unlimited"])
@pytest.mark.parametrize("w", ["soup_varying_w", "degenerate", "overlap_mesh_inf_w", "unit_square_negative_z", 0.9e-6, 1.1e-6, 0.9e6, 1.1e6,
                               1e-8, 1e-20, 1e-30, 1e-38, 1e30, 0.0, "around zero", "inf"])
def test_gradients_where_the_depth_map_has_none(w, mode, cuda):
    """A frame whose depth map took no part in the loss has kernels of its own, which leave out what is 0 times the depth's derivatives
    but keep the NaNs it makes where those are not finite: against the general ones with a gradient of zeros."""
    import torch
    import scenes as S
    from trigrad_amd import _C
    from trigrad_amd._C import _forward_full
    if w in SCENES:
        scene, tw, th = SCENES[w]()
    else:
        rng = np.random.default_rng(3)
        scene, tw, th = S.random_soup(400, 70, 45, seed=3, sigma_px=7.0, opacity=(0.2, 0.9)), 16, 16
        n = scene["vertices"].shape[0]
        with np.errstate(all="ignore"):
            if w == "around zero":
                scene = _with_w(scene, (rng.standard_normal(n) * 1e-3).astype(np.float32))
            elif w == "inf":  # some vertices
                scene = _with_w(scene, np.where(rng.random(n) < 0.05, np.inf, rng.uniform(0.1, 2.0, n)).astype(np.float32))
            else:
                scene = _with_w(scene, (w * rng.uniform(1.0, 1.0001, n)).astype(np.float32))
    m = MODES[mode]
    W, H = scene["width"], scene["height"]
    d = to_device(scene, cuda)
    ml = m["max_layers"] if m["max_layers"] > 0 else scene["indices"].shape[0] + 1
    image, depthmap, weights, sorted_ids, offsets, bary, ends, _, resume = _forward_full(
        d["vertices"], d["indices"], d["colors"], d["opacities"], W, H, tw, th, 1 / 256, True, m["per_pixel_sort"], ml)
    gi, gd = _grad_inputs(scene, 3, False)
    outs = [_C.render_backward(torch.from_numpy(gi).to(cuda), g, d["vertices"], d["indices"], d["colors"], d["opacities"], sorted_ids,
                               offsets, bary, image, depthmap, weights, ends, W, H, tw, th, 1 / 256, m["per_pixel_sort"], ml, resume=resume)
            for g in (None, torch.from_numpy(gd).to(cuda))]
    for label, got, want in zip(("grad_vertices", "grad_colors", "grad_opacities"), *(tuple(g.cpu().numpy() for g in out) for out in outs)):
        _assert_same_terms(f"{w}/{mode}: {label}", got, want)


@pytest.mark.parametrize("width,height,tw,th", [(513, 512, 16, 16), (512, 512, 16, 16), (478, 480, 16, 16), (500, 452, 16, 16), (448, 512, 16, 16),
                                                (509, 511, 32, 8), (505, 497, 8, 8), (411, 403, 12, 20), (256, 192, 16, 16), (257, 190, 16, 16)])
@pytest.mark.parametrize("layers", [32, 40, None])
def test_gradients_by_waves_alone_and_in_fours(width, height, tw, th, layers, cuda, oracle):
    """The backward kernels run a wave to a workgroup, or four where the frame's waves (ceil(tile / 64) a tile) fill the chip's SIMDs up to
    four times, the last time to more than three quarters (769 to 1024, 1793 to 2048, ... 4096 waves): numbers of waves on both sides,
    tiles of one, two and four waves, numbers of tiles that are no multiple of eight; tile order where layers is None."""
    import torch
    import scenes as S
    import trigrad_amd
    scene = S.random_soup(1500, width, height, seed=width + (layers or 0), sigma_px=14.0, opacity=(0.1, 0.6), varying_w=True)
    order, limit = layers is not None, layers or 1501
    want = oracle.render(scene["vertices"], scene["indices"], scene["colors"], scene["opacities"], width, height, tw, th, 1 / 256, order, limit)
    gi, gd = _grad_inputs(scene, 4, False)
    wanted = oracle.render_backward(gi, gd, scene["vertices"], scene["indices"], scene["colors"], scene["opacities"], want, width, height,
                                    tw, th, order, limit, literal=False, magnitudes=True)
    d = to_device(scene, cuda)
    leaves = [d[k].clone().requires_grad_() for k in ("vertices", "colors", "opacities")]
    image, _ = trigrad_amd.render(leaves[0], d["indices"], *leaves[1:], width, height, tw, th, per_pixel_sort=order, max_layers=limit)
    out = torch.autograd.grad(image, leaves, torch.from_numpy(gi).to(cuda))
    for label, g, w, mag in zip(("grad_vertices", "grad_colors", "grad_opacities"), out, wanted[:3], wanted[3:]):
        assert_gradients_close(f"{width}x{height}, tiles of {tw}x{th}, {layers} layers: {label}", g.cpu().numpy(), w, mag)


@pytest.mark.parametrize("n", [1, 63, 64, 65, 128, 129, 300])
@pytest.mark.parametrize("width,height,tw,th", [(16, 16, 16, 16), (21, 13, 16, 16), (40, 24, 8, 8), (50, 26, 24, 24), (9, 7, 3, 5)])
def test_tile_order_gradients_around_blocks_of_a_list(width, height, tw, th, n, cuda, oracle):
    """In tile order a wave walks its tile's list backwards in blocks of 64 entries and takes the (pixel, entry) hits of a block in
    rounds of 64: lists around multiples of 64, every pixel with one fragment of a block or with all of them, pixels that stop
    inside a block, waves without a pixel; with the forward pass's hit masks and without."""
    import torch
    import scenes as S
    from trigrad_amd import _C
    scene = S.random_soup(n, width, height, seed=n + width, sigma_px=9.0, opacity=(0.02, 0.4), varying_w=True)
    mode = dict(per_pixel_sort=False, max_layers=n + 1)
    d, want, got, ml = _forward_both(scene, tw, th, mode, cuda, oracle)
    _check_forward(f"{n} in {width}x{height}", want, got, (th, tw))
    gi, gd = _grad_inputs(scene, 6, False)
    wanted = oracle.render_backward(gi, gd, scene["vertices"], scene["indices"], scene["colors"], scene["opacities"], want, width, height,
                                    tw, th, False, ml, literal=False, magnitudes=True)
    image, depthmap, weights, sorted_ids, offsets, bary, ends, _, resume = got
    for masks in (resume, resume[:4] + (None,)):
        for depth_gradient in (None, torch.from_numpy(gd).to(cuda)):
            out = _C.render_backward(torch.from_numpy(gi).to(cuda), depth_gradient, d["vertices"], d["indices"], d["colors"], d["opacities"],
                                     sorted_ids, offsets, bary, image, depthmap, weights, ends, width, height, tw, th, 1 / 256, False, ml, resume=masks)
            for label, g, w, mag in zip(("grad_vertices", "grad_colors", "grad_opacities"), out, wanted[:3], wanted[3:]):
                assert_gradients_close(f"{n} in {width}x{height}, tiles of {tw}x{th}: {label}", g.cpu().numpy(), w, mag)


@pytest.mark.parametrize("mode", ["A_default", "A_40_layers", "B_unlimited"])
@pytest.mark.parametrize("width,height,tw,th", [(1, 1, 16, 16), (2, 1, 16, 16), (5, 3, 16, 16), (8, 8, 8, 8), (64, 1, 64, 1), (9, 9, 8, 8)])
@pytest.mark.parametrize("n", [1, 2, 5, 63, 65, 130])
def test_gradients_of_pixels_with_many_slots_of_a_round(n, width, height, tw, th, mode, cuda, oracle):
    """A round of the backward pass hands the state from one of a pixel's slots to the next in as many turns as a pixel has slots: waves
    of one pixel, whose fragments fill every slot, of a few, and of 64 with one or many each; with a gradient of the depth map and
    without one."""
    import torch
    import scenes as S
    import trigrad_amd
    m = MODES[mode]
    ml = m["max_layers"] if m["max_layers"] > 0 else n + 1
    scene = S.random_soup(n, width, height, seed=n + width, sigma_px=40.0, opacity=(0.01, 0.2), varying_w=True)
    want = oracle.render(scene["vertices"], scene["indices"], scene["colors"], scene["opacities"], width, height, tw, th, 1 / 256,
                         m["per_pixel_sort"], ml)
    gi, gd = _grad_inputs(scene, 5, True)
    d = to_device(scene, cuda)
    for depth_gradient in (None, gd):
        wanted = oracle.render_backward(gi, np.zeros_like(gd) if depth_gradient is None else gd, scene["vertices"], scene["indices"], scene["colors"],
                                        scene["opacities"], want, width, height, tw, th, m["per_pixel_sort"], ml, literal=False, magnitudes=True)
        leaves = [d[k].clone().requires_grad_() for k in ("vertices", "colors", "opacities")]
        outputs = trigrad_amd.render(leaves[0], d["indices"], *leaves[1:], width, height, tw, th, per_pixel_sort=m["per_pixel_sort"], max_layers=m["max_layers"])
        upstream = [torch.from_numpy(x).to(cuda) for x in ((gi,) if depth_gradient is None else (gi, gd))]
        out = torch.autograd.grad(outputs[:len(upstream)], leaves, upstream)
        for label, g, w, mag in zip(("grad_vertices", "grad_colors", "grad_opacities"), out, wanted[:3], wanted[3:]):
            assert_gradients_close(f"{n} in {width}x{height}/{mode}: {label}", g.cpu().numpy(), w, mag)


@pytest.mark.parametrize("mode", ["A_default", "A_5_layers", "A_40_layers", "A_unlimited"])
@pytest.mark.parametrize("tw,th", [(16, 16), (8, 8), (6, 5)])
@pytest.mark.parametrize("n", [1, 22, 23, 24, 31, 32, 33, 64, 65, 140])
def test_candidates_behind_and_in_front_of_the_last(n, tw, th, mode, cuda, oracle):
    """A pixel's candidates come in the order of the list, which is not the pixel's where triangles are steep: behind the last candidate,
    in front of it, and at its depth, in lists with room, at the edge of what is kept in LDS (23 places), and full (32); with one, two
    and more selections."""
    import scenes as S
    rng = np.random.default_rng(n)
    width, height = 24, 20
    scene = S.random_soup(n, width, height, seed=n, sigma_px=60.0, opacity=(0.01, 0.2))
    v = scene["vertices"].reshape(n, 3, 4)
    v[::3, :, 2] = rng.uniform(0.1, 10.0, (len(v[::3]), 3))  # steep ones, flat ones, and pairs at one depth
    v[1::3, :, 2] = np.round(v[1::3, :1, 2] * 0.5) + 1.0
    v[..., 3] = 1.0 / v[..., 2]
    scene["vertices"] = np.ascontiguousarray(v.reshape(3 * n, 4), np.float32)
    _, want, got, _ = _forward_both(scene, tw, th, MODES[mode], cuda, oracle)
    _check_forward(f"{n} candidates/{tw}x{th}/{mode}", want, got, (th, tw))


@pytest.mark.parametrize("mode", ["A_default", "A_unlimited", "B_unlimited"])
@pytest.mark.parametrize("width,height,tw,th", [(1, 1, 16, 16), (1, 9, 8, 8), (9, 7, 16, 16), (17, 33, 16, 16), (40, 25, 32, 32), (23, 19, 24, 8),
                                                (50, 47, 40, 24), (129, 9, 128, 8), (20, 21, 10, 6), (33, 5, 7, 8)])
def test_waves_at_the_edges_of_an_image(width, height, tw, th, mode, cuda, oracle):
    """The rectangle of a wave's pixels decides which list entries it looks at: whole squares of 8 x 8, those the image cuts, waves
    without a pixel, and waves that are no squares; tiles of a power of two of squares a row, and of 3 and 5."""
    import scenes as S
    scene = S.random_soup(500, width, height, seed=width + height, sigma_px=3.0, opacity=(0.05, 0.4), varying_w=True)
    _, want, got, _ = _forward_both(scene, tw, th, MODES[mode], cuda, oracle)
    _check_forward(f"{width}x{height}/{tw}x{th}/{mode}", want, got, (th, tw))


@pytest.mark.parametrize("mode", ["A_default", "A_40_layers", "A_unlimited", "B_unlimited"])
@pytest.mark.parametrize("width,height,tw,th,big", [(520, 410, 16, 16, 0), (301, 203, 8, 8, 0), (300, 200, 32, 32, 3000), (160, 120, 16, 16, 900), (1920, 400, 16, 16, 0)])
@pytest.mark.parametrize("saved", [True, False])
def test_frames_with_records_of_their_triangles(saved, width, height, tw, th, big, mode, cuda, monkeypatch):
    """Many triangles with vertices of their own are rendered from records (TG_FRAME_RECORDS), others from the arrays: the same image, depth
    map and lists, and gradients the same up to the order of the atomics; tiles of one and several workgroups, frames of few and
    many, and lists of thousands, which depth bounds and the long tiles' kernels are for; in tile order without the saved hit masks too (in per-pixel order a backward pass
    without a saved order reads the matrices, so there are no records).  Some triangles name a vertex that is
    none, some are degenerate or far off the screen, and some attributes are zero or infinite."""
    import torch
    import scenes as S
    from trigrad_amd import _C
    m = MODES[mode]
    monkeypatch.setattr(_C, "SAVE_HIT_MASKS", saved)
    monkeypatch.setattr(_C, "SAVE_BLEND_ORDER", saved)
    n = 160_000 if m["per_pixel_sort"] else 510_000
    ml = m["max_layers"] if m["max_layers"] > 0 else n + 1
    rng = np.random.default_rng(width)
    scene = S.random_soup(n, width, height, seed=width, sigma_px=0.6, opacity=(0.2, 0.9), varying_w=True)
    v = scene["vertices"].reshape(n, 3, 4)
    if big:
        v[:big, :, :2] = rng.standard_normal((big, 3, 2)) * (6.0 / width)
    v[5000] = v[5000, :1]
    v[5001, :, :2] += 1.0e6
    idx = scene["indices"].copy()
    idx[5002, 1], idx[5003, 2] = 3 * n, -1
    scene["colors"][15012:15030] = 0.0
    scene["colors"][15033:15036] = np.inf
    d = to_device(dict(scene, indices=idx), cuda)
    args = (d["vertices"], d["indices"], d["colors"], d["opacities"], width, height, tw, th, 1 / 256, m["per_pixel_sort"], ml)
    for _ in range(2):  # the second frame's buffers go by the first one's keys
        packed, plain = _C.frame_forward(*args), _C.frame_forward(*args, records=False)
    short = packed[3].plan.capacity <= 800 * (-(-width // tw) * -(-height // th))  # in tile order long lists are left early
    assert packed[3].records == (saved if m["per_pixel_sort"] else short) and not plain[3].records
    for a, b in zip(packed[:2], plain[:2]):
        assert torch.equal(torch.nan_to_num(a, 7.0), torch.nan_to_num(b, 7.0)) and torch.equal(torch.isnan(a), torch.isnan(b))
    results = [_C._frame_results(*f, width, height, tw, th, m["per_pixel_sort"], ml, n) for f in (packed, plain)]
    for k in (2, 3, 4, 5, 6):  # weights, sorted ids, offsets, bary matrices, ends
        a, b = results[0][k], results[1][k]
        assert a.shape == b.shape and torch.equal(torch.nan_to_num(a.double(), 7.0), torch.nan_to_num(b.double(), 7.0))
    gi, gd = (torch.from_numpy(x).to(cuda) for x in _grad_inputs(scene, 3, True))
    for depth_gradient in (None, gd):
        got, want = (_C.frame_backward(f[3], gi, depth_gradient, *args[:4], f[0], f[1], f[2]) for f in (packed, plain))
        again = _C.frame_backward(plain[3], gi, depth_gradient, *args[:4], plain[0], plain[1], plain[2])
        for g, w, w2 in zip(got, want, again):
            assert torch.equal(torch.isfinite(g), torch.isfinite(w))
            g, w, w2 = (torch.nan_to_num(x, 0.0, 0.0, 0.0).double() for x in (g, w, w2))
            # two runs of one route differ by the order of their atomics; the two routes by no more than four times that
            assert (g - w).norm() <= 4 * (w2 - w).norm() + 1e-6 * w.norm()


# two triangles a thread of the scan, and four; a wave's last triangles are fewer than its lanes
@pytest.mark.parametrize("width,height,tile,n,mode", [(*size, mode) for size in ((520, 410, 16, 160_037), (301, 203, 8, 270_011), (300, 200, 32, 160_037), (1920, 400, 16, 270_011))
                                                      for mode in ("A_default", "A_40_layers", "A_unlimited", "B_unlimited")
                                                      if mode != "B_unlimited" or size[2] < 32])  # in tile order frames of long lists have no records
def test_gradients_by_element_of_frames_with_records(width, height, tile, n, mode, cuda, oracle):
    """Each gradient of a frame with triangles' records is as near the oracle's as sums in another order are, and its image, depth map and lists are
    those without; the last triangles are those of a wave with lanes to spare, some name a vertex that is none, and an infinite colour is
    in the sums of few."""
    import torch
    import scenes as S
    from trigrad_amd import _C
    m = MODES[mode]
    n = n if m["per_pixel_sort"] else 510_001
    ml = m["max_layers"] if m["max_layers"] > 0 else n + 1
    scene = S.random_soup(n, width, height, seed=width, sigma_px=0.6, opacity=(0.2, 0.9), varying_w=True)
    scene["vertices"].reshape(n, 3, 4)[-64:, :, :2] *= 0.3  # on the image
    scene["colors"][15033:15036] = np.inf
    idx = scene["indices"].copy()
    idx[5002, 1], idx[5003, 2] = 3 * n, -1
    d = to_device(dict(scene, indices=idx), cuda)
    args = (d["vertices"], d["indices"], d["colors"], d["opacities"], width, height, tile, tile, 1 / 256, m["per_pixel_sort"], ml)
    for _ in range(2):  # the second frame's buffers go by the first one's keys
        packed, plain = _C.frame_forward(*args), _C.frame_forward(*args, records=False)
    assert packed[3].records and not plain[3].records
    for a, b in zip(packed[:2], plain[:2]):
        assert torch.equal(torch.nan_to_num(a, 7.0), torch.nan_to_num(b, 7.0)) and torch.equal(torch.isnan(a), torch.isnan(b))
    results = [_C._frame_results(*f, width, height, tile, tile, m["per_pixel_sort"], ml, n) for f in (packed, plain)]
    for k in (2, 3, 4, 5, 6):  # weights, sorted ids, offsets, bary matrices, ends
        a, b = results[0][k], results[1][k]
        assert a.shape == b.shape and torch.equal(torch.nan_to_num(a.double(), 7.0), torch.nan_to_num(b.double(), 7.0))
    known = dict(scene, indices=scene["indices"].copy())
    known["indices"][5002:5004] = 0  # in no list either
    known = [known[k] for k in ("vertices", "indices", "colors", "opacities")]
    known += [oracle.render(*known, width, height, tile, tile, 1 / 256, m["per_pixel_sort"], ml), width, height, tile, tile, m["per_pixel_sort"], ml]
    gi, gd = _grad_inputs(scene, 3, True)
    for depth_gradient in (None, gd):
        wanted = oracle.render_backward(gi, np.zeros_like(gd) if depth_gradient is None else gd, *known, literal=False, magnitudes=True)
        got = _C.frame_backward(packed[3], torch.from_numpy(gi).to(cuda), None if depth_gradient is None else torch.from_numpy(gd).to(cuda),
                                *args[:4], packed[0], packed[1], packed[2])
        for label, g, w, mag in zip(("grad_vertices", "grad_colors", "grad_opacities"), got, wanted[:3], wanted[3:]):
            finite = np.isfinite(w) & np.isfinite(mag)  # an infinite colour is not in the sums of all
            assert finite.mean() > 0.99
            assert_gradients_close(f"{n} in {width}x{height}/{mode}: {label}", g.cpu().numpy()[finite], w[finite], mag[finite])


@pytest.mark.parametrize("mode,n", [("A_default", 160_037), ("A_40_layers", 270_011), ("B_unlimited", 510_001), ("A_default", 140_000)])
def test_timed_frames_run_the_kernels_of_untimed_ones(n, mode, cuda, oracle, monkeypatch):
    """The stages that record_timing=True times are those of the frame that a user gets without asking: from triangles' records where that
    one is; the same image and, by the route by stages with the matrices out of the records, the gradients."""
    import torch
    import scenes as S
    import trigrad_amd
    from trigrad_amd import _C
    m, width, height = MODES[mode], 520, 410
    ml = m["max_layers"] if m["max_layers"] > 0 else n + 1
    scene = S.random_soup(n, width, height, seed=n, sigma_px=0.6, opacity=(0.2, 0.9), varying_w=True)
    want = oracle.render(scene["vertices"], scene["indices"], scene["colors"], scene["opacities"], width, height, 16, 16, 1 / 256, m["per_pixel_sort"], ml)
    gi, gd = _grad_inputs(scene, 6, True)
    wanted = oracle.render_backward(gi, gd, scene["vertices"], scene["indices"], scene["colors"], scene["opacities"], want, width, height, 16, 16,
                                    m["per_pixel_sort"], ml, literal=False, magnitudes=True)
    rendered, frame_forward = [], _C.frame_forward

    def seen(*args, **kwargs):
        rendered.append(frame_forward(*args, **kwargs))
        return rendered[-1]

    monkeypatch.setattr(_C, "frame_forward", seen)
    _C._module().forget()  # an untimed frame by the Python route too
    d = to_device(scene, cuda)
    leaves = [d[k].clone().requires_grad_() for k in ("vertices", "colors", "opacities")]
    frames = [trigrad_amd.render(leaves[0], d["indices"], *leaves[1:], width, height, record_timing=timed, per_pixel_sort=m["per_pixel_sort"],
                                 max_layers=m["max_layers"]) for timed in (False, True)]
    assert [f[3].records for f in rendered] == [n != 140_000] * 2 and "rasterization" in frames[1][2]
    for outputs in frames:
        assert torch.equal(outputs[0], frames[0][0]) and torch.equal(outputs[1], frames[0][1])
        out = torch.autograd.grad(outputs[:2], leaves, (torch.from_numpy(gi).to(cuda), torch.from_numpy(gd).to(cuda)))
        for label, g, w, mag in zip(("grad_vertices", "grad_colors", "grad_opacities"), out, wanted[:3], wanted[3:]):
            assert_gradients_close(f"{n}/{mode}: {label}", g.cpu().numpy(), w, mag)


@pytest.mark.parametrize("n,mode", [(160_037, "A_default"), (510_001, "B_unlimited"), (140_000, "A_default")])
@pytest.mark.parametrize("disable_timing", [True, False])
def test_matrices_of_render_forward_are_a_dense_array(disable_timing, n, mode, cuda):
    """render_forward hands out the bary matrices as an array of their own, of frames with timing too, and so a kernel or a view takes them
    as they are."""
    import torch
    import scenes as S
    from trigrad_amd import _C
    m, width, height = MODES[mode], 520, 410
    d = to_device(S.random_soup(n, width, height, seed=n, sigma_px=0.6), cuda)
    bary = _C.render_forward(d["vertices"], d["indices"], d["colors"], d["opacities"], width, height, 16, 16, 1 / 256, disable_timing,
                             m["per_pixel_sort"], 32)[5]
    assert bary.shape == (n, 3, 3) and bary.is_contiguous()
    want = _C.cartesian_to_bary(d["vertices"], d["indices"])
    assert torch.equal(bary.view(-1), want.view(-1))


def test_reaches_in_records_are_outside_of_their_triangles_and_not_far(cuda):
    """A record's bounds are steps of 2^-14 rounded to the outside, held in [-2, 2): no triangle's corner is beyond them, those of triangles of
    some pixels are no further out than two steps and a tenth of a pixel wherever on the screen, and NaN and infinity leave nothing out."""
    import scenes as S
    from trigrad_amd import _C
    n, width, height = 160_037, 1920, 1080
    scene = S.random_soup(n, width, height, seed=3, sigma_px=3.0, varying_w=True)
    v = scene["vertices"].reshape(n, 3, 4)
    v[:1000, :, :2] *= 3.0  # partly and wholly beside the image
    v[1000, 0, 0], v[1001, 1, 1] = np.nan, np.inf
    d = to_device(scene, cuda)
    args = (d["vertices"], d["indices"], d["colors"], d["opacities"], width, height, 16, 16, 1 / 256, True, 32)
    _, _, kept, frame = _C.frame_forward(*args)
    assert frame.records
    at = frame.plan.at["bary"]
    words = kept[at:at + 128 * n].cpu().numpy().view(np.int32).reshape(n, 32)[:, 15:17]
    lo, hi = ((words << 16) >> 16) / 2.0 ** 14, (words >> 16) / 2.0 ** 14  # (n, 2): x and y
    xy = v[..., :2].astype(np.float64)
    least, most = xy.min(axis=1), xy.max(axis=1)
    fine = np.isfinite(xy).all(axis=(1, 2))
    top = 2.0 - 2.0 ** -14
    assert (lo[fine] <= np.maximum(least[fine], -2.0)).all() and (hi[fine] >= np.minimum(most[fine], top)).all()
    assert (lo[1000:1002] == -2.0).all() and (hi[1000:1002] == top).all()  # in both directions: the matrix is of NaN
    e = (xy[:, 1:] - xy[:, :1]) * [width / 2, height / 2]
    longest = np.sqrt(np.maximum(np.maximum((e ** 2).sum(axis=2).max(axis=1), ((e[:, 1] - e[:, 0]) ** 2).sum(axis=1)), 1e-30))
    round_ones = fine & (np.abs(e[:, 0, 0] * e[:, 1, 1] - e[:, 0, 1] * e[:, 1, 0]) > 3.0 * longest) & (np.abs(xy).max(axis=(1, 2)) < 1.5)
    assert round_ones.sum() > n // 8
    slack = 2 * 2.0 ** -14 + 0.1 * np.array([2 / width, 2 / height])
    assert (least - lo <= slack)[round_ones].all() and (hi - most <= slack)[round_ones].all()


@pytest.mark.parametrize("mode,n", [("A_default", 149_999), ("A_default", 150_000), ("A_default", 150_001), ("A_40_layers", 150_037), ("B_unlimited", 499_999),
                                    ("B_unlimited", 500_000), ("B_unlimited", 500_001)])
def test_plans_of_frames_around_the_numbers_that_have_records(n, mode, cuda, oracle):
    """Frames share the plan of a rounded number of triangles: with records and without them, and a mesh behind a soup of as many triangles;
    the first frame of a kind by the Python route, later ones by the module's."""
    import torch
    import scenes as S
    import trigrad_amd
    from trigrad_amd import _C
    m, width, height = MODES[mode], 520, 410
    ml = m["max_layers"] if m["max_layers"] > 0 else n + 1
    soup = S.random_soup(n, width, height, seed=n, sigma_px=0.6, opacity=(0.2, 0.9), varying_w=True)
    mesh, k = S.random_soup(-(-n // 3), width, height, seed=n + 1, sigma_px=1.0, opacity=(0.2, 0.9), varying_w=True), -(-n // 3)
    # each of its triangles is cut in three at its middle: four vertices for three
    a, b, c, middle = *mesh["indices"].T, np.arange(3 * k, 4 * k)
    mesh["indices"] = np.ascontiguousarray(np.stack([a, b, middle, b, c, middle, c, a, middle], axis=1).reshape(-1, 3)[:n], dtype=np.int32)
    for name in ("vertices", "colors", "opacities"):
        x = mesh[name].reshape(k, 3, -1)
        mesh[name] = np.ascontiguousarray(np.concatenate([x.reshape(3 * k, -1), x.mean(axis=1)]).reshape(4 * k, *mesh[name].shape[1:]), dtype=np.float32)
    mesh["vertices"][3 * k:, 3] = 1.0 / mesh["vertices"][3 * k:, 2]
    expected = []
    for scene in (soup, mesh):
        want = oracle.render(scene["vertices"], scene["indices"], scene["colors"], scene["opacities"], width, height, 16, 16, 1 / 256, m["per_pixel_sort"], ml)
        gi, gd = _grad_inputs(scene, 4, True)
        wanted = oracle.render_backward(gi, gd, scene["vertices"], scene["indices"], scene["colors"], scene["opacities"], want, width, height, 16, 16,
                                        m["per_pixel_sort"], ml, literal=False, magnitudes=True)
        d = to_device(scene, cuda)
        plain = _C.frame_forward(d["vertices"], d["indices"], d["colors"], d["opacities"], width, height, 16, 16, 1 / 256, m["per_pixel_sort"], ml, records=False)
        expected.append((d, plain[:2], [torch.from_numpy(x).to(cuda) for x in (gi, gd)], wanted))
    _C._module().forget()
    for kind, routes in ((0, ("Python", "module")), (1, ("Python", "module")), (0, ("module",))):
        d, plain, upstream, wanted = expected[kind]
        leaves = [d[k].clone().requires_grad_() for k in ("vertices", "colors", "opacities")]
        for route in routes:
            outputs = trigrad_amd.render(leaves[0], d["indices"], *leaves[1:], width, height, per_pixel_sort=m["per_pixel_sort"], max_layers=m["max_layers"])
            assert ("RendererBackward" in type(outputs[0].grad_fn).__name__) == (route == "Python")
            for a, b in zip(outputs, plain):
                assert torch.equal(a, b)
            out = torch.autograd.grad(outputs, leaves, upstream)
            for label, g, w, mag in zip(("grad_vertices", "grad_colors", "grad_opacities"), out, wanted[:3], wanted[3:]):
                assert_gradients_close(f"{n}/{mode}/{kind}/{route}: {label}", g.cpu().numpy(), w, mag)


@pytest.mark.parametrize("n,width,height,tw,sigma", [(1, 64, 64, 16, 9.0), (511, 64, 64, 16, 2.0), (512, 300, 200, 16, 2.0), (513, 300, 200, 8, 6.0), (9000, 500, 400, 8, 6.0),
                                                     (131071, 640, 480, 16, 1.0), (131072, 640, 480, 16, 0.3), (131073, 640, 480, 16, 1.0),
                                                     (262144, 1000, 700, 16, 0.5), (262145, 1000, 700, 16, 2.0), (600000, 1000, 700, 16, 3.0)])
def test_lists_of_frames_around_the_sizes_that_split_the_work_otherwise(n, width, height, tw, sigma, cuda, monkeypatch):
    """The scan takes 1, 2 or 4 triangles a thread, the emission 1 or 2 keys and the sweeps 2, 4 or 8 pairs: frames on both sides of every line have the lists
    of the route by stages, which knows none of them."""
    import torch
    import scenes as S
    from trigrad_amd import _C
    d = to_device(S.random_soup(n, width, height, seed=n, sigma_px=sigma), cuda)
    args = (d["vertices"], d["indices"], d["colors"], d["opacities"], width, height, tw, 16, 1 / 256, True, True, 8)
    for _ in range(2):  # the second frame's buffers go by the first one's keys
        got = _C._forward_full(*args)
    got[8][2].verify()
    monkeypatch.setattr(_C, "ONE_CALL_FRAME", False)
    want = _C._forward_full(*args)
    want[8][2].verify()
    for k in (0, 1, 3, 4, 6):  # image, depth map, sorted ids, offsets, ends
        assert torch.equal(got[k], want[k])


def _blocks_of_a_backward_pass(backward, n_vertices):
    """Its results, and how many (V,8) blocks it summed the gradients in, by the memory it asked for: 32 bytes a vertex for the gradients
    and as many for each block."""
    import torch
    torch.cuda.reset_peak_memory_stats()
    before = torch.cuda.memory_stats()["requested_bytes.all.current"]
    results = backward()
    blocks, rest = divmod(torch.cuda.memory_stats()["requested_bytes.all.peak"] - before, 32 * n_vertices)
    assert rest == 0
    return results, blocks - 1


@pytest.mark.parametrize("mode", ["A_default", "A_40_layers", "B_unlimited"])
@pytest.mark.parametrize("vertices,shared,width,height", [
    (32767, False, 128, 128), (32768, False, 128, 128), (32770, False, 130, 97), (3000, False, 129, 128), (3000, True, 256, 256),
    (3000, True, 257, 256), (32768, False, 1024, 511), (32768, False, 1024, 512), (32767, False, 1024, 512)])
def test_gradients_summed_in_a_block_or_in_place(vertices, shared, width, height, mode, cuda, oracle):
    """In per-pixel order from 32768 vertices on or in images of more than 16384 pixels, and in tile order where triangles share vertices
    in images of more than 65536 or 32768 vertices are in one of 2^19, the gradients are summed in a (V,8) block, else in the
    dense arrays: on both sides of the lines, by the frame's call (a first frame, and ones whose plan is there) and by the
    stage-by-stage route."""
    import torch
    import scenes as S
    import trigrad_amd
    from trigrad_amd import _C, _lib
    m = MODES[mode]
    scene = S.random_soup(-(-vertices // 3), width, height, seed=8, sigma_px=3.0, opacity=(0.1, 0.6), varying_w=True)
    indices = np.minimum(scene["indices"], vertices - 1)
    if shared:  # every vertex is three triangles', none of them larger than the others
        indices = np.concatenate([indices, indices[:, [1, 2, 0]], indices[:, [2, 0, 1]]])
    scene.update(vertices=scene["vertices"][:vertices], colors=scene["colors"][:vertices], opacities=scene["opacities"][:vertices],
                 indices=np.ascontiguousarray(indices, dtype=np.int32))
    by_block = (vertices >= 32768 or width > 128) if m["per_pixel_sort"] else (shared and width == 257) or (vertices == 32768 and height == 512)
    kind = _C._FRAME_KIND.pack(vertices, scene["indices"].shape[0], width, height, 16, 16, m["per_pixel_sort"], 32, 0, 0, 0, 0, 0.0)
    assert _C._gradient_copies(_lib.load(32), kind) == by_block
    d, want, got, ml = _forward_both(scene, 16, 16, m, cuda, oracle)
    gi, gd = _grad_inputs(scene, 2, False)
    wanted = oracle.render_backward(gi, gd, scene["vertices"], scene["indices"], scene["colors"], scene["opacities"], want, width, height, 16, 16,
                                    m["per_pixel_sort"], ml, literal=False, magnitudes=True)
    gi = torch.from_numpy(gi).to(cuda)
    image, depthmap, weights, sorted_ids, offsets, bary, ends, _, resume = got
    outs = [_C.render_backward(gi, None, d["vertices"], d["indices"], d["colors"], d["opacities"], sorted_ids, offsets, bary, image, depthmap,
                               weights, ends, width, height, 16, 16, 1 / 256, m["per_pixel_sort"], ml, resume=resume)]
    leaves = [d[k].clone().requires_grad_() for k in ("vertices", "colors", "opacities")]
    for _ in range(3):
        image, _ = trigrad_amd.render(leaves[0], d["indices"], *leaves[1:], width, height, per_pixel_sort=m["per_pixel_sort"], max_layers=m["max_layers"])
        out, blocks = _blocks_of_a_backward_pass(lambda: torch.autograd.grad(image, leaves, gi), vertices)
        assert blocks == by_block
        outs.append(out)
    for out in outs:
        for label, g, w, mag in zip(("grad_vertices", "grad_colors", "grad_opacities"), out, wanted[:3], wanted[3:]):
            assert g.is_contiguous()
            assert_gradients_close(f"{vertices} vertices/{mode}: {label}", g.cpu().numpy(), w, mag)


@pytest.mark.parametrize("mode", ["A_default", "A_40_layers", "A_unlimited", "B_unlimited"])
@pytest.mark.parametrize("n,sigma,width,height,tw,th,per_waves", [
    (150, 20.0, 150, 121, 16, 16, True), (150, 20.0, 128, 128, 16, 16, False), (1512, 20.0, 150, 121, 16, 16, True), (1513, 20.0, 150, 121, 16, 16, False), (400, 30.0, 200, 131, 8, 8, True), (400, 4.0, 200, 131, 8, 8, False),
    (60, 50.0, 160, 160, 32, 32, True), (20, 2.0, 256, 256, 16, 16, False), (341, 2.0, 256, 256, 16, 16, False), (3000, 2.0, 400, 300, 16, 16, False)])
def test_gradients_summed_by_xcds(n, sigma, width, height, tw, th, per_waves, mode, cuda, oracle):
    """Where triangles are in 20 waves on average each XCD sums the gradients in a block of its own: on both sides of the lines, by a
    first frame (the Python route, whose buffers have room for 65536 keys more) and by ones whose plan is there (the module's)."""
    import torch
    import scenes as S
    import trigrad_amd
    from trigrad_amd import _C
    m = MODES[mode]
    scene = S.random_soup(n, width, height, seed=n, sigma_px=sigma, opacity=(0.05, 0.5), varying_w=True)
    ml = m["max_layers"] if m["max_layers"] > 0 else n + 1
    want = oracle.render(scene["vertices"], scene["indices"], scene["colors"], scene["opacities"], width, height, tw, th, 1 / 256,
                         m["per_pixel_sort"], ml)
    gi, gd = _grad_inputs(scene, 9, True)
    wanted = oracle.render_backward(gi, gd, scene["vertices"], scene["indices"], scene["colors"], scene["opacities"], want, width, height, tw, th,
                                    m["per_pixel_sort"], ml, literal=False, magnitudes=True)
    d = to_device(scene, cuda)
    leaves = [d[k].clone().requires_grad_() for k in ("vertices", "colors", "opacities")]
    upstream = (torch.from_numpy(gi).to(cuda), torch.from_numpy(gd).to(cuda))
    _C._frame_key_hints.clear()
    _C._frame_size_hints.clear()
    _C._module().forget()
    for frame in range(4):
        outputs = trigrad_amd.render(leaves[0], d["indices"], *leaves[1:], width, height, tw, th, per_pixel_sort=m["per_pixel_sort"], max_layers=m["max_layers"])
        assert ("RendererBackward" in type(outputs[0].grad_fn).__name__) == (frame == 0)
        out, blocks = _blocks_of_a_backward_pass(lambda: torch.autograd.grad(outputs, leaves, upstream), 3 * n)
        assert blocks == (8 if per_waves else int(m["per_pixel_sort"] and width * height > 16384))
        for label, g, w, mag in zip(("grad_vertices", "grad_colors", "grad_opacities"), out, wanted[:3], wanted[3:]):
            assert_gradients_close(f"{n} triangles/{mode}: {label}", g.cpu().numpy(), w, mag)

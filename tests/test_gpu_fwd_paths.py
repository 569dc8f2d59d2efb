"""The forward rasterizer's routes: frames of up to 256 tiles (one workgroup per
quadrant), up to 512 (the same where a few tiles are crowded, by the lists'
lengths beside the order) and larger ones, whole and partial tiles and blocks of channels, plain and other batches.  One scene drawn
into canvases of every size must have the same bits; frames of odd sizes, their
edges covered, must have the oracle's."""

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _frame(W, H, C, depth, plain, n=900):
    """(outputs cropped to the scene's 96 x 80 pixels, tile bounds) of a W x H canvas."""
    import torch

    from mlx3d_amd.splatting.rasterize import raster_forward, tile_order_buffer
    from mlx3d_amd.splatting.tiles import bin_gaussians

    rng = np.random.default_rng(17 + C)
    cu = lambda a: torch.from_numpy(np.ascontiguousarray(a, np.float32)).cuda()  # noqa: E731
    xy = rng.uniform([-4, -4], [100, 84], (n, 2))
    a = rng.uniform(0.02, 0.5, n)
    c = rng.uniform(0.02, 0.5, n)
    b = rng.uniform(-0.7, 0.7, n) * np.sqrt(a * c)
    op = rng.uniform(0.0, 1.2, n)
    op[::40] = 0.0
    if not plain:  # a singular conic, a huge opacity and an infinite channel
        b[5] = np.sqrt(a[5] * c[5])
        op[9] = 1e31
    feats = rng.standard_normal((n, C))
    if not plain:
        feats[11, 0] = np.inf
    co = cu(np.stack([a, b, c, op], 1))
    z = cu(rng.uniform(1, 9, n))
    ids, ranges, _, _ = bin_gaussians(cu(xy), cu(np.full(n, 24.0)), z, W, H)
    order = tile_order_buffer(W, H, co.device)
    order.fill_(0)
    bg = cu(rng.standard_normal(C))
    out = raster_forward(cu(xy), co, cu(feats), ids, ranges, bg, W, H,
                         depths=z if depth else None, tile_order=order)
    tx, ty = (W + 15) // 16, (H + 15) // 16
    bounds = order[:tx * ty].view(ty, tx)[:5, :6].cpu().numpy()
    crop = [None if t is None else t[:80, :96].contiguous().cpu().numpy() for t in out]
    return crop, bounds


@pytest.mark.parametrize("C,depth,plain", [(1, False, True), (2, True, True), (3, False, True),
                                           (3, True, True), (4, True, True), (3, True, False),
                                           (5, False, True), (16, True, True)])
def test_frame_sizes_agree(C, depth, plain):
    # 30, 192 | 208, 256 | 272, 396 | 525, 3600, 6500 tiles
    base, bounds = _frame(96, 80, C, depth, plain)
    n_contrib = base[2]
    tiles = n_contrib.reshape(5, 16, 6, 16).max(axis=(1, 3))
    np.testing.assert_array_equal(bounds, tiles)
    assert int(n_contrib.max()) > 48  # several chunks of a workgroup's list
    for W, H in ((192, 256), (208, 256), (256, 256), (272, 256), (352, 288), (400, 336),
                 (1280, 720), (1600, 1040)):
        got, b = _frame(W, H, C, depth, plain)
        np.testing.assert_array_equal(b, bounds)
        for name, x, y in zip(("out", "final_T", "n_contrib", "depth", "alpha"), base, got):
            if x is not None:
                np.testing.assert_array_equal(x, y, err_msg=f"{name} {W}x{H}")


@pytest.mark.parametrize("n", [1, 2, 3, 4, 5, 6, 255, 256, 257, 515])
def test_needle_lists_match_oracle(n):
    """Batches with an ill-conditioned conic, an opacity past the exp's range and
    an infinite channel, in lists of every remainder of a round: the oracle's bits."""
    from gpu_util import assert_bits, cu, host
    from mlx3d_amd.splatting.rasterize import pack_conic_opacity, raster_forward
    from mlx3d_amd.splatting.tiles import bin_gaussians
    from oracle import oracle as O

    W, H, C = 561, 369, 3  # a corner tile of 1 x 1 pixels
    rng = np.random.default_rng(n)
    xy = rng.uniform([W - 12, H - 12], [W + 2, H + 2], (n, 2)).astype(np.float32)
    a, c = rng.uniform(0.01, 0.3, n), rng.uniform(0.01, 0.3, n)
    con = np.stack([a, rng.uniform(-0.7, 0.7, n) * np.sqrt(a * c), c], 1).astype(np.float32)
    op = rng.uniform(0.004, 0.1, n).astype(np.float32)
    feats = rng.standard_normal((n, C)).astype(np.float32)
    z = rng.uniform(1, 9, n).astype(np.float32)
    k = n // 2
    con[k], xy[k] = (1e3, 0.0, 1e-4), (W - 7.5, H - 40.0)
    if n > 3:
        op[0], feats[3, 1] = 1e31, np.inf
    ids, ranges, _, _ = bin_gaussians(cu(xy), cu(np.full(n, 24.0, np.float32)), cu(z), W, H)
    bg = rng.random(C, dtype=np.float32)
    ref = O.raster_fwd(xy, con, op, feats, host(ids), host(ranges), W, H, bg=bg, depths=z)
    out, fT, nc, depth, _ = raster_forward(cu(xy), pack_conic_opacity(cu(con), cu(op)), cu(feats),
                                           ids, ranges, cu(bg), W, H, depths=cu(z))
    assert ref["n_contrib"].max() >= min(n, 3) - 1
    np.testing.assert_array_equal(host(nc), ref["n_contrib"])
    for name, got in (("image", out), ("final_T", fT), ("depth", depth)):
        assert_bits(host(got), ref[name], name)


@pytest.mark.parametrize("C", [5, 6, 7, 9, 10, 11, 13, 14, 15, 16, 38, 41, 47])
def test_channel_blocks_match_oracle(C):
    """Every remainder of a block's groups of four channels (the last ones overlap),
    the block's last channel infinite for one Gaussian: the oracle's bits."""
    from gpu_util import assert_features, cu, host
    from mlx3d_amd.splatting.rasterize import pack_conic_opacity, raster_forward
    from mlx3d_amd.splatting.tiles import bin_gaussians
    from oracle import oracle as O

    W, H, n = 57, 41, 300
    rng = np.random.default_rng(C)
    xy = rng.uniform([-2, -2], [W + 2, H + 2], (n, 2)).astype(np.float32)
    a, c = rng.uniform(0.02, 0.5, n), rng.uniform(0.02, 0.5, n)
    con = np.stack([a, rng.uniform(-0.7, 0.7, n) * np.sqrt(a * c), c], 1).astype(np.float32)
    op = rng.uniform(0.01, 0.6, n).astype(np.float32)
    feats = rng.standard_normal((n, C)).astype(np.float32)
    feats[17, C - 1] = np.inf
    ids, ranges, _, _ = bin_gaussians(cu(xy), cu(np.full(n, 16.0, np.float32)),
                                      cu(rng.uniform(1, 9, n).astype(np.float32)), W, H)
    bg = rng.random(C, dtype=np.float32)
    ref = O.raster_fwd(xy, con, op, feats, host(ids), host(ranges), W, H, bg=bg)
    out, _, nc, _, _ = raster_forward(cu(xy), pack_conic_opacity(cu(con), cu(op)), cu(feats),
                                      ids, ranges, cu(bg), W, H)
    assert np.isinf(ref["image"][..., C - 1]).any()
    np.testing.assert_array_equal(host(nc), ref["n_contrib"])
    assert_features(host(out), ref["image"])


# 943 tiles (7 past a multiple of 8), 273, 294, 209 and 6363 tiles, corner tiles of
# 1 x 1; 273 to 294 tiles evenly filled and crowded
@pytest.mark.parametrize("C,depth,W,H,crowd", [
    (1, True, 641, 359, False), (2, False, 641, 359, False), (3, False, 641, 359, False),
    (3, True, 641, 359, False), (4, True, 641, 359, True), (4, False, 331, 195, False),
    (4, False, 331, 195, True), (1, True, 331, 195, True), (4, True, 289, 167, False),
    (4, True, 289, 167, True), (2, False, 335, 211, True), (3, True, 335, 211, False),
    (3, True, 335, 211, True), (3, True, 1601, 1007, False), (1, False, 1601, 1007, True)])
def test_render_of_odd_frames_matches_oracle(C, depth, W, H, crowd):
    """Images, T, contributor counts, depth and gradients through the public render
    (which takes the binning's order), Gaussians up to and past every edge."""
    from gpu_util import assert_bits, cu, host, oracle_backward, oracle_forward, rel_err
    from mlx3d_amd.cameras import Camera
    from mlx3d_amd.splatting import render_gaussian_features

    import torch

    n = 4000
    rng = np.random.default_rng(100 * C + W)
    cam = Camera.look_at(eye=(0.0, 0.0, -4.0), width=W, height=H)
    half = 4.0 * 0.5 * H / cam.fy  # of the frame's height in the plane of the means
    f32 = lambda a: np.ascontiguousarray(a, np.float32)  # noqa: E731
    means = f32(rng.uniform(-1.05, 1.05, (n, 3)) * [half * W / H, half, 0.5])
    if crowd:
        means[n // 4:, :2] *= np.float32(0.04)
    quats, scales = f32(rng.standard_normal((n, 4))), f32(rng.uniform(0.005, 0.06, (n, 3)))
    opac, feats = f32(rng.uniform(0.02, 0.95, n)), f32(rng.standard_normal((n, C)))
    bg = rng.random(C, dtype=np.float32)
    t = [cu(a).requires_grad_(True) for a in (means, quats, scales, opac, feats)]
    out = render_gaussian_features(cam, *t, background=cu(bg), return_depth=depth)
    pre, f, ids, ranges, r = oracle_forward(cam, means, quats, scales, opac, colors=feats, bg=bg,
                                            depth=depth)
    nc, lists = r["n_contrib"], ranges[:, 1] - ranges[:, 0]
    assert (lists.max() * lists.size >= 8 * lists.sum()) == crowd
    assert min(nc[0].max(), nc[-1].max(), nc[:, 0].max(), nc[:, -1].max()) > 0
    np.testing.assert_array_equal(host(out["n_contrib"]), nc)
    assert_bits(host(out["features"]), r["image"], "image")
    assert_bits(host(out["final_T"]), r["final_T"], "final_T")
    if depth:
        assert_bits(host(out["depth"]), r["depth"], "depth")
    g_img = rng.standard_normal((H, W, C)).astype(np.float32)
    g_a = rng.standard_normal((H, W)).astype(np.float32)
    torch.autograd.backward([out["features"], out["alpha"]], [cu(g_img), cu(g_a)])
    g = oracle_backward(cam, means, quats, scales, opac, pre, f, ids, ranges, r, g_img, g_a, bg=bg)
    for name, a in zip(("means", "quats", "scales", "opacities", "features"), t):
        # the repository's bound for gradients of this chain (tests/test_gpu_parity.py)
        assert rel_err(host(a.grad), g[name]) < 1e-3, name


@pytest.mark.parametrize("W,H", [(64, 64), (328, 200), (641, 359)])
def test_order_holds_the_bands_lengths(W, H):
    """Behind the order's T words: each band's longest list and its number of
    entries, from the binning's placement and from the forward's own launch."""
    from gpu_util import cu, host
    from mlx3d_amd.cameras import Camera
    from mlx3d_amd.splatting import render_gaussians
    from mlx3d_amd.splatting.rasterize import raster_forward, tile_order_buffer

    rng = np.random.default_rng(W)
    n = 2000
    cam = Camera.look_at(eye=(0.0, 0.0, -4.0), width=W, height=H)
    t = [cu(np.asarray(a, np.float32)) for a in (
        rng.standard_normal((n, 3)) * 0.7, rng.standard_normal((n, 4)),
        rng.uniform(0.02, 0.1, (n, 3)), rng.uniform(0.1, 0.9, n), rng.random((n, 3)))]
    t[0].requires_grad_(True)
    out = render_gaussians(cam, *t[:4], colors=t[4])
    placed = out["image"].grad_fn.saved_tensors[-1]  # the backward has not run
    ranges, ids = out["tile_ranges"], out["sorted_ids"]
    T = ranges.shape[0]
    own = tile_order_buffer(W, H, ranges.device)
    raster_forward(out["means2d"].detach(), cu(np.ones((n, 4), np.float32)), t[4], ids, ranges,
                   None, W, H, tile_order=own)
    lists = host(ranges[:, 1] - ranges[:, 0])
    cuts = np.cumsum([0] + [T // 8 + (x < T % 8) for x in range(8)])
    bands = [lists[a:b] for a, b in zip(cuts[:-1], cuts[1:])]
    want = [b.max() for b in bands] + [b.sum() for b in bands]
    for order in (placed, own):
        np.testing.assert_array_equal(host(order)[2 * T:2 * T + 16], want)

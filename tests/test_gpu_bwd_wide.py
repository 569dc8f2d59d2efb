"""The backward for five channels and more (lanes are Gaussians): list lengths
around its buckets (16), its chunks (64) and its buffer (80), partial tiles and
quadrants, every channel block, non-finite inputs, and the geometry record with
its split form, against the oracle."""

from __future__ import annotations

import importlib

import numpy as np
import pytest
import torch

from gpu_util import cu, host, say
from mlx3d_amd.splatting import bin_gaussians
from oracle import oracle as O

pytestmark = pytest.mark.gpu

# the module (the package's attribute of that name is the function)
RASTERIZE = importlib.import_module("mlx3d_amd.splatting.rasterize")


def _scene(n, C, W, H, seed):
    """n 2D Gaussians that all reach every tile of a small image; every 40th
    is a needle (conic past the plain bound) down a column of pixel centres,
    opacities from faint to 1."""
    rng = np.random.default_rng(seed)
    m2 = np.stack([rng.uniform(-2, W + 2, n), rng.uniform(-2, H + 2, n)], 1).astype(np.float32)
    a, c = rng.uniform(0.005, 0.2, n), rng.uniform(0.005, 0.2, n)
    b = rng.uniform(-0.8, 0.8, n) * np.sqrt(a * c)
    op = rng.uniform(0.003, 1.0, n).astype(np.float32)
    op[op < 0.3] *= 0.1  # long lists before a pixel stops
    a[7::40], c[7::40], b[7::40], op[7::40] = 1e3, 1e-4, 0.0, 0.4
    m2[7::40] = np.floor(rng.uniform(0, 1, m2[7::40].shape) * [W, H]) + 0.5
    if n == 1:
        m2[0], op[0] = (W // 2 + 0.3, H // 2 + 0.8), 0.7
    con = np.stack([a, b, c], 1).astype(np.float32)
    feats = rng.standard_normal((n, C)).astype(np.float32)
    depths = rng.uniform(1, 2, n).astype(np.float32)
    radii = np.full(n, 64.0, np.float32)
    ids, ranges, _, _ = bin_gaussians(cu(m2), cu(radii), cu(depths), W, H)
    return m2, con, op, feats, ids, ranges, rng


def _alpha(m2, con, op, px, py):
    """(alpha, G, dx, dy) of (L, P) pairs in the kernels' float32 (fused steps
    rounded once from float64; float32 products are exact there)."""
    f = np.float32
    dx = m2[:, :1] - px[None].astype(f)
    dy = m2[:, 1:] - py[None].astype(f)
    A, B, C = f(-0.5) * con[:, :1], -con[:, 1:2], f(-0.5) * con[:, 2:]
    inner = (B.astype(np.float64) * dy + A * dx).astype(f)
    power = (inner.astype(np.float64) * dx + (C * dy) * dy).astype(f)
    G = O.splat_expf(power)
    alpha = np.minimum(f(0.99), op[:, None] * G)
    return np.where((power <= 0) & (alpha >= f(1.0 / 255.0)), alpha, f(0)), G, dx, dy


def _terms(m2, con, op, feats, ids, ranges, n_contrib, W, H, bg, g_img, g_T):
    """Every gradient in 64 bits, the sum of its terms' sizes (each product's and
    each summand's absolute value) and the most Gaussians a pixel composites."""
    d = np.float64
    n, C = feats.shape
    val = dict(means2d=np.zeros((n, 2)), conics=np.zeros((n, 3)), opacities=np.zeros(n),
               features=np.zeros((n, C)))
    size = {k: np.zeros_like(v) for k, v in val.items()}
    most = 0
    tiles_x = (W + 15) // 16
    for tile, (lo, hi) in enumerate(ranges):
        ty, tx = divmod(tile, tiles_x)
        y, x = np.mgrid[16 * ty:min(16 * ty + 16, H), 16 * tx:min(16 * tx + 16, W)]
        y, x, order = y.ravel(), x.ravel(), ids[lo:hi]
        al, G, dx, dy = _alpha(m2[order], con[order], op[order], x + 0.5, y + 0.5)
        al = np.where(np.arange(hi - lo)[:, None] < n_contrib[y, x][None], al, 0).astype(d)
        most = max(most, int((al > 0).sum(0).max(initial=0)))
        T = np.cumprod(np.concatenate([np.ones((1, y.size)), 1.0 - al]), 0)
        T, T_end = T[:-1], T[-1]
        g = g_img[y, x].astype(d)
        f = feats[order].astype(d)
        for out, cg, end in ((val, f @ g.T, g @ bg.astype(d) + g_T[y, x]),
                             (size, np.abs(f) @ np.abs(g).T,
                              np.abs(g) @ np.abs(bg).astype(d) + np.abs(g_T[y, x]))):
            sign = -1.0 if out is val else 1.0
            w = al * T * cg
            behind = T_end * end + w[::-1].cumsum(0)[::-1] - w
            h = np.where(al > 0, G * (T * cg + sign * behind / (1.0 - al)), 0.0)
            o, (a, b, c) = op[order].astype(d)[:, None], con[order].astype(d).T[..., None]
            ab = (lambda v: v) if out is val else np.abs
            dx_, dy_ = ab(dx.astype(d)), ab(dy.astype(d))
            parts = dict(
                means2d=np.stack([(sign * o * h * (ab(a) * dx_ + ab(b) * dy_)).sum(1),
                                  (sign * o * h * (ab(c) * dy_ + ab(b) * dx_)).sum(1)], 1),
                conics=np.stack([(sign * 0.5 * o * h * dx_ * dx_).sum(1),
                                 (sign * o * h * dx_ * dy_).sum(1),
                                 (sign * 0.5 * o * h * dy_ * dy_).sum(1)], 1),
                opacities=h.sum(1), features=(al * T) @ (g if out is val else np.abs(g)))
            for k, v in parts.items():
                np.add.at(out[k], order, v)
    return val, size, most


def _both(m2, con, op, feats, ids, ranges, W, H, bg, g_img, g_T):
    from mlx3d_amd.splatting.rasterize import (pack_conic_opacity, raster_backward_geometry,
                                               raster_forward, split_geometry)

    ref = O.raster_fwd(m2, con, op, feats, host(ids), host(ranges), W, H, bg=bg)
    rg = O.raster_bwd(m2, con, op, feats, host(ids), host(ranges), W, H, ref["final_T"],
                      ref["n_contrib"], g_img, grad_final_T=g_T, bg=bg)
    assert ref["n_contrib"].max() > 0
    co = pack_conic_opacity(cu(con), cu(op))
    _, fT, nc, _, _ = raster_forward(cu(m2), co, cu(feats), ids, ranges, cu(bg), W, H)
    np.testing.assert_array_equal(host(nc), ref["n_contrib"])
    rec, gf = raster_backward_geometry(cu(m2), co, cu(feats), ids, ranges, cu(bg), W, H, fT, nc,
                                       cu(g_img), cu(g_T))
    gm, gc, go = split_geometry(rec)
    got = {"means2d": gm, "conics": gc, "opacities": go, "features": gf}
    assert gf.is_contiguous()
    if rec.shape[1] == 8:
        assert float(rec[:, 6:].abs().max()) == 0.0
    return {k: (host(v), np.asarray(rg[k])) for k, v in got.items()}, ref["n_contrib"]


def _edges(n, C, W, H):
    m2, con, op, feats, ids, ranges, rng = _scene(n, C, W, H, 100 + n + C)
    bg = rng.random(C, dtype=np.float32)
    g_img = rng.standard_normal((H, W, C)).astype(np.float32)
    g_T = rng.standard_normal((H, W)).astype(np.float32)
    both, n_contrib = _both(m2, con, op, feats, ids, ranges, W, H, bg, g_img, g_T)
    val, size, most = _terms(m2, con, op, feats, host(ids), host(ranges), n_contrib, W, H, bg,
                             g_img, g_T)
    # Of the size of a gradient's terms (2^-24 each): T in front of an entry has
    # two roundings an entry ahead of it (1 - alpha, the product) and three an
    # entry behind (a reciprocal of 1 ulp, the product): 5 L; the colour behind
    # the same again and a sum: 6 L; c . g: C; the sums over the pixels: P; the
    # other products of a term: 16
    bound = (11 * most + C + W * H + 16) * 2.0 ** -24
    for k, (a, b) in both.items():
        e = np.abs(a - val[k])
        worst = float((e[size[k] > 0] / size[k][size[k] > 0]).max())
        say(f"  n={n} C={C} {W}x{H} {k}: {worst:.2e} of the terms (bound {bound:.1e})")
        assert (e <= bound * size[k]).all(), k
        assert float(np.abs(a - b).max() / (np.abs(b).max() + 1e-30)) < 1e-4, k
        needles = b[7::40]
        assert needles.size == 0 or (np.abs(needles).max(axis=-1) > 0).any(), k


@pytest.mark.parametrize("n,C,W,H", [(1, 5, 1, 1), (15, 8, 23, 9), (16, 9, 16, 16),
                                     (17, 16, 7, 23), (79, 17, 23, 9), (80, 32, 17, 15),
                                     (81, 5, 33, 8), (400, 12, 23, 9), (400, 37, 16, 17),
                                     (33, 33, 17, 9), (64, 34, 9, 17), (65, 36, 16, 16)])
def test_wide_backward_list_edges(n, C, W, H):
    _edges(n, C, W, H)


@pytest.mark.parametrize("n,C,W,H", [(1, 5, 1, 1), (17, 8, 7, 23), (81, 10, 33, 8),
                                     (80, 11, 17, 15), (16, 15, 16, 16), (400, 10, 23, 9),
                                     (400, 12, 23, 9)])
def test_wide_backward_whole_lines(n, C, W, H, monkeypatch):
    """The features' gradient gathered in the record or in rows of 16."""
    monkeypatch.setattr(RASTERIZE, "_whole_lines", lambda n, C, d: True)
    _edges(n, C, W, H)


@pytest.mark.parametrize("C", [7, 13])
def test_render_features_in_whole_lines(C, monkeypatch):
    """A feature render whose Gaussians reach many tiles takes those rows by
    itself and gives the gradients of the packed ones."""
    from mlx3d_amd.cameras import Camera
    from mlx3d_amd.splatting import render_gaussian_features

    rng = np.random.default_rng(C)
    n, W, H = 3000, 639, 361
    raw = (rng.uniform(-1, 1, (n, 3)), rng.standard_normal((n, 4)),
           rng.uniform(0.15, 0.4, (n, 3)), rng.uniform(0.01, 0.2, n), rng.standard_normal((n, C)))
    cam = Camera.look_at(eye=(0, 0, -3.0), width=W, height=H)
    g = cu(rng.standard_normal((H, W, C)).astype(np.float32))
    taken, grads = [], []
    rule = RASTERIZE._whole_lines
    for force in (None, False):
        monkeypatch.setattr(RASTERIZE, "_whole_lines", lambda *a, force=force: taken.append(
            rule(*a) if force is None else force) or taken[-1])
        t = [cu(np.asarray(a, np.float32)).requires_grad_(True) for a in raw]
        render_gaussian_features(cam, *t)["features"].backward(g)
        grads.append([host(x.grad) for x in t])
    assert taken == [True, False]
    for name, a, b in zip(("means", "quats", "scales", "opacities", "features"), *grads):
        # the same sums, in the order the atomics came
        np.testing.assert_allclose(a, b, rtol=0, atol=2e-5 * np.abs(b).max(), err_msg=name)


@pytest.mark.parametrize("C", [6, 32])
def test_wide_backward_non_finite(C):
    """An infinite feature and a NaN cotangent reach exactly the gradients
    that composite with them."""
    W, H, n = 23, 9, 60
    m2, con, op, feats, ids, ranges, rng = _scene(n, C, W, H, 7 + C)
    con[:, [0, 2]] += 0.3  # small footprints: most pairs do not meet
    feats[20, 1] = np.inf
    g_img = rng.standard_normal((H, W, C)).astype(np.float32)
    g_img[4, 11, C - 1] = np.nan
    bg = np.zeros(C, np.float32)
    g_T = np.zeros((H, W), np.float32)
    both, _ = _both(m2, con, op, feats, ids, ranges, W, H, bg, g_img, g_T)
    for k, (a, b) in both.items():
        fin = np.isfinite(b)
        say(f"  C={C} {k}: {int((~fin).sum())} of {fin.size} non-finite")
        np.testing.assert_array_equal(np.isfinite(a), fin, err_msg=k)
        assert fin.any()
        e = float(np.abs(a[fin] - b[fin]).max() / (np.abs(b[fin]).max() + 1e-30))
        assert e < 1e-4, k


@pytest.mark.parametrize("plain", [True, False])
@pytest.mark.parametrize("by_pixel", [True, False])
@pytest.mark.parametrize("C", [5, 9, 17])
def test_wide_backward_behind_opaque(C, by_pixel, plain):
    """The colour behind an opaque entry, which dL/dalpha divides by 1 - alpha =
    0.01: stacks of three Gaussians, each on one pixel alone (the middle one at the
    0.99 clamp, a dim one behind it), against 64 bits, in list orders that put a
    stack's entries side by side and a layer apart."""
    from mlx3d_amd.splatting.rasterize import (pack_conic_opacity, raster_backward_geometry,
                                               raster_forward)

    W = H = 32
    P, L = W * H, 3
    rng = np.random.default_rng(C)
    layer, pixel = np.divmod(np.arange(L * P), P)
    m2 = np.stack([pixel % W + 0.5, pixel // W + 0.5], 1).astype(np.float32)
    con = np.tile(np.array([30.0, 0.0, 30.0 if plain else 1e9], np.float32), (L * P, 1))
    op = np.array([0.3, 1.0, 0.5], np.float32)[layer]
    feats = rng.uniform(0.5, 1.0, (L * P, C)).astype(np.float32)
    feats[layer == 2] *= np.float32(0.01)
    g_img = rng.uniform(0.5, 1.0, (H, W, C)).astype(np.float32)
    depths = 1.0 + (pixel * L + layer if by_pixel else layer * P + pixel).astype(np.float32)
    ids, ranges, _, _ = bin_gaussians(cu(m2), cu(np.ones(L * P, np.float32)), cu(depths), W, H)
    co = pack_conic_opacity(cu(con), cu(op))
    _, fT, nc, _, _ = raster_forward(cu(m2), co, cu(feats), ids, ranges, None, W, H)
    rec, _ = raster_backward_geometry(cu(m2), co, cu(feats), ids, ranges, None, W, H, fT, nc,
                                      cu(g_img), None)
    got = host(rec)[:, 5].astype(np.float64).reshape(L, P)  # dL/dopacity = dL/dalpha (G = 1)
    # alpha is min(0.99, opacity) to the bit, so 64 bits start from the same values
    alpha = np.minimum(np.float32(0.99), op).astype(np.float64).reshape(L, P)
    cg = (feats.astype(np.float64).reshape(L, P, C) * g_img.reshape(1, P, C)).sum(-1)
    T = np.cumprod(np.concatenate([np.ones((1, P)), 1.0 - alpha[:-1]]), 0)
    term = alpha * T * cg
    behind = term[::-1].cumsum(0)[::-1] - term
    want = T * cg - behind / (1.0 - alpha)
    scale = T * cg + behind / (1.0 - alpha)
    # every term is positive.  T: three roundings of 1 - alpha and three products
    # ahead, a reciprocal (1 ulp) and a product an entry back; c . g: C
    # products and sums; alpha T, the sum behind, its quotient, the difference
    # and h / opacity: at most (6 + 9 + C + 8) 2^-24 of the terms' size
    e = np.abs(got - want) / scale
    say(f"  C={C} by_pixel={by_pixel} plain={plain}: largest error {e.max(1)} of the terms")
    assert e.max() < (23 + C) * 2.0 ** -24

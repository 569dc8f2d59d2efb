"""The measured workloads of the splatting path.

Each case is one call sequence of a user's program on seeded synthetic
scenes: viewing a model, one differentiable render with its backward, a
feature render, a render through a calibrated lens, and a training step.
``listed()`` are the fixed cases, ``draw(rng)`` another one of the same
ranges, ``prepare`` the state such a program holds, ``run`` one pass through
the public entry points, ``work`` the bytes and operations the pass cannot do
without, ``exact`` what ``run`` returns in 64 bits by plain torch.
"""

import math

import torch

from mlx3d_amd.cameras import Camera
from mlx3d_amd.losses import l1_loss
from mlx3d_amd.splatting import (GaussianModel, GaussianTrainer, TrainerConfig, render_gaussians,
                                 render_gaussian_features)

TILE = 16
GROUPS = ("means", "scales", "quats", "opacities", "sh_dc", "sh_rest")
# learning rates of a refinement run: a hundredth of the trainer's defaults,
# so that a scene keeps its statistics however many steps are timed
RATES = {"means": 1.6e-6, "scales": 5e-5, "quats": 1e-5, "opacities": 5e-4, "sh_dc": 2.5e-5,
         "sh_rest": 1.25e-6}
LAMBDA = 0.2
THICKNESS = 1e-4
FISHEYE = (0.05, -0.02, 0.004, -0.001)
BROWN = (0.08, -0.03, -0.004, 0.003, 0.01)


def listed():
    return [
        # a viewer's thumbnail of a fresh point-cloud initialisation: DC colour
        # only, isotropic Gaussians, with depth; launches and host time count
        dict(name="preview_256", kind="view", scene="blob", n=10_000, degree=0, width=256,
             height=256, antialias=False, depth=True, morton=False),
        # interactive viewing of a small model in a window of odd size
        dict(name="view_odd_720p", kind="view", scene="box", n=100_000, degree=3, width=1279,
             height=717, antialias=False, depth=False, morton=False),
        # frames of a full-size model, antialiased, rows in spatial order
        dict(name="view_1080p", kind="view", scene="shells", n=1_000_000, degree=3, width=1920,
             height=1080, antialias=True, depth=False, morton=True),
        # optimisation against a photograph with a calibrated fisheye: unscented
        # projection and tight tile lists, activated parameters, own SH tensor
        dict(name="lens_square", kind="lens", scene="box", n=300_000, degree=2, width=1021,
             height=1021, antialias=True, lens="fisheye", refine=True),
        # one iteration of a user's own training loop (L1, backward to the raw
        # parameters) on a small model
        dict(name="iter_720p", kind="iter", scene="box", n=100_000, degree=3, width=1280,
             height=720, antialias=False, morton=False),
        # the same on a full-size model: the headline configuration
        dict(name="iter_1080p", kind="iter", scene="shells", n=1_000_000, degree=3, width=1920,
             height=1080, antialias=True, morton=True),
        # the same on a large table in creation order with a few percent of very
        # large Gaussians (sky, walls): long tile lists
        dict(name="iter_heavy", kind="iter", scene="heavy", n=3_000_000, degree=3, width=1920,
             height=1080, antialias=False, morton=False),
        # distilling a 32-channel feature field, with depth
        dict(name="features_32", kind="features", scene="box", n=500_000, channels=32, width=1280,
             height=720, normalize=False, depth=True),
        # a normalised map of a few semantic channels at video size
        dict(name="features_12", kind="features", scene="shells", n=60_000, channels=12, width=641,
             height=479, normalize=True, depth=False),
        # early training, while density control gathers its statistics
        dict(name="train_early", kind="train", scene="shells", n=50_000, degree=1, width=801,
             height=599, antialias=False, method="vanilla", collect=True),
        # late training of a full-size model: photometric loss, Adam on all groups
        dict(name="train_1080p", kind="train", scene="shells", n=1_000_000, degree=3, width=1920,
             height=1080, antialias=True, method="vanilla", collect=False),
        # training surfels with the depth and normal regularisers
        dict(name="train_2dgs", kind="train", scene="shells", n=200_000, degree=2, width=960,
             height=540, antialias=False, method="2dgs", collect=False),
    ]


def draw(rng):
    def log_int(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    kind = rng.choice(("view", "view", "iter", "iter", "lens", "features", "train", "train"))
    # widths from a thumbnail to full HD, landscape to square
    width = log_int(200, 1920)
    height = max(128, min(1080, int(width / rng.uniform(1.0, 1.8))))
    # no more than two Gaussians a pixel: a table is trained at its images' scale
    case = dict(kind=kind, scene=rng.choice(("blob", "box", "shells", "heavy")),
                n=min(log_int(5_000, 900_000), 2 * width * height), width=width, height=height)
    if kind in ("view", "iter"):
        case.update(degree=rng.randint(0, 3), antialias=rng.random() < 0.5,
                    morton=rng.random() < 0.5)
        if kind == "view":
            case["depth"] = rng.random() < 0.3
    elif kind == "lens":
        case.update(n=min(case["n"], 400_000), degree=rng.randint(0, 3),
                    antialias=rng.random() < 0.5, lens=rng.choice(("fisheye", "brown")),
                    refine=rng.random() < 0.5)
    elif kind == "features":
        case.update(n=min(case["n"], 500_000), channels=rng.choice((1, 2, 4, 5, 8, 13, 16, 24, 32)),
                    normalize=rng.random() < 0.5, depth=rng.random() < 0.5)
    else:
        method = rng.choice(("vanilla", "vanilla", "2dgs"))
        if method == "2dgs":
            case["n"] = min(case["n"], 150_000)
        case.update(degree=rng.randint(0, 3), antialias=rng.random() < 0.5, method=method,
                    collect=method == "vanilla" and rng.random() < 0.5)
    return case


# ------------------------------------------------------------------ inputs
def _camera(case, gen):
    """A seeded view from a distance of 4 to 5 towards the centre, 60 degrees high."""
    u = torch.rand(3, generator=gen, device="cuda").tolist()
    radius = {"blob": 4.0, "box": 4.2, "shells": 5.0, "heavy": 5.0}[case["scene"]]
    th, ph = 2.0 * math.pi * u[0], math.radians(60.0 * u[1] - 30.0)
    eye = torch.tensor([math.cos(ph) * math.sin(th), math.sin(ph), -math.cos(ph) * math.cos(th)],
                       dtype=torch.float64) * radius
    z = -eye / eye.norm()
    x = torch.linalg.cross(z, torch.tensor([0.0, 1.0, 0.0], dtype=torch.float64))
    x = x / x.norm()
    R = torch.stack([x, torch.linalg.cross(z, x), z]).float()
    t = (-(R.double() @ eye)).float()
    f = float(torch.tensor(case["height"] / (2.0 * math.tan(math.radians(30.0)))).float())
    return dict(R=R, t=t, f=f, cx=case["width"] / 2.0, cy=case["height"] / 2.0)


def _inputs(case, seed):
    """Raw parameters (log-scales, opacity logits), camera and target, from the seed alone."""
    gen = torch.Generator(device="cuda").manual_seed(1 + 7919 * int(seed))
    n, scene = case["n"], case["scene"]

    def uniform(*shape):
        return torch.rand(*shape, generator=gen, device="cuda")

    def normal(*shape):
        return torch.randn(*shape, generator=gen, device="cuda")

    logit = normal(n)
    if scene == "blob":  # a fresh initialisation: opacity 0.1, isotropic until it is trained
        means = 0.5 * normal(n, 3)
        scales = (-3.2 - math.log(n / 10_000) / 3 + 0.4 * normal(n, 1)).expand(n, 3).contiguous()
        if case["kind"] != "view":
            scales = scales + 0.3 * normal(n, 3)
        logit = torch.full((n,), math.log(0.1 / 0.9), device="cuda")
    elif scene == "box":
        means = 3.0 * uniform(n, 3) - 1.5
        scales = -4.0 - math.log(n / 100_000) / 3 + 0.5 * normal(n, 3)
    elif scene == "shells":  # surfaces and floaters
        shell = n - n * 3 // 10
        d = normal(shell, 3)
        d = d / d.norm(dim=1, keepdim=True)
        means = torch.cat([d * (1.0 + 2.0 * uniform(shell, 1)) + 0.02 * normal(shell, 3),
                           8.0 * uniform(n - shell, 3) - 4.0])
        scales = -4.5 - math.log(n / 1_000_000) / 3 + 0.7 * normal(n, 3)
        logit = 1.5 * logit
    else:  # heavy: 3 % of the Gaussians two orders larger than the others
        means = 6.0 * uniform(n, 3) - 3.0
        scales = torch.where(uniform(n, 1) < 0.03, -1.5 + 0.3 * normal(n, 3),
                             -5.0 - math.log(n / 3_000_000) / 3 + 0.5 * normal(n, 3))
    quats = normal(n, 4)
    quats = quats / quats.norm(dim=1, keepdim=True)
    if scene == "blob" and case["kind"] == "view":
        quats = torch.zeros_like(quats)
        quats[:, 0] = 1.0
    K = (case.get("degree", 0) + 1) ** 2
    p = dict(means=means, quats=quats, scales=scales, opacities=logit,
             sh_dc=uniform(n, 1, 3) - 0.5, sh_rest=0.05 * normal(n, K - 1, 3))
    if case.get("method") == "2dgs":  # surfels, thinner than the trainer's cap
        p["scales"][:, 2] = math.log(THICKNESS) - 0.1 * uniform(n)
    C = case.get("channels", 3)
    if case["kind"] == "features":
        p["features"] = normal(n, C)
    cam = _camera(case, gen)
    # a photograph: smooth structure and some grain
    coarse = uniform(1, C, 12, 16)
    smooth = torch.nn.functional.interpolate(coarse, size=(case["height"], case["width"]),
                                             mode="bilinear", align_corners=False)[0]
    target = (0.9 * smooth.permute(1, 2, 0) + 0.1 * uniform(case["height"], case["width"], C))
    return {k: v.contiguous() for k, v in p.items()}, cam, target.contiguous()


def _lens(case):
    if case.get("lens") == "fisheye":
        return dict(distortion=FISHEYE, fisheye=True)
    return dict(distortion=BROWN) if case.get("lens") == "brown" else {}


def prepare(case, seed):
    p, c, target = _inputs(case, seed)
    kind = case["kind"]
    s = dict(case=case, target=target,
             camera=Camera(R=c["R"], t=c["t"], fx=c["f"], fy=c["f"], cx=c["cx"], cy=c["cy"],
                           width=case["width"], height=case["height"], **_lens(case)))
    if kind in ("view", "iter", "train"):
        m = GaussianModel({k: p[k] for k in GROUPS}, sh_degree=case["degree"])
        m.active_sh_degree = case["degree"]
        if case.get("morton"):
            m.reorder_spatial()
        s["model"] = m
    if kind == "iter":
        s["model"].requires_grad_(True)
    elif kind == "lens":
        s["params"] = {"means": p["means"], "quats": p["quats"], "scales": torch.exp(p["scales"]),
                       "opacities": torch.sigmoid(p["opacities"]),
                       "sh": torch.cat([p["sh_dc"], p["sh_rest"]], dim=1)}
    elif kind == "features":
        s["params"] = {"means": p["means"], "quats": p["quats"], "scales": torch.exp(p["scales"]),
                       "opacities": torch.sigmoid(p["opacities"]), "features": p["features"]}
    if kind in ("lens", "features"):
        s["params"] = {k: v.contiguous().requires_grad_(True) for k, v in s["params"].items()}
    if kind == "train":
        two_d = case["method"] == "2dgs"
        config = TrainerConfig(
            method=case["method"], antialias=case["antialias"], lambda_dssim=LAMBDA,
            lr_means=RATES["means"], lr_means_final=0.01 * RATES["means"],
            lr_scales=RATES["scales"], lr_quats=RATES["quats"], lr_opacities=RATES["opacities"],
            lr_sh_dc=RATES["sh_dc"], lr_sh_rest=RATES["sh_rest"], two_d_thickness=THICKNESS,
            lambda_2d_depth_variance=0.1 if two_d else 0.0,
            lambda_2d_normal_consistency=0.05 if two_d else 0.0,
            # statistics are gathered, but the table keeps its size
            densify_from=0 if case["collect"] else 500,
            densify_until=10 ** 9 if case["collect"] else 0, densify_every=10 ** 9,
            opacity_reset_every=10 ** 9)
        s["trainer"] = GaussianTrainer(s["model"], config)
    return s


# -------------------------------------------------------------------- runs
def _backward(loss, params):
    loss.backward()
    grads = {k: v.grad for k, v in params.items()}
    for v in params.values():
        v.grad = None
    return grads


def run(s):
    case = s["case"]
    kind = case["kind"]
    if kind == "view":
        with torch.no_grad():
            out = s["model"].render(s["camera"], antialias=case["antialias"],
                                    return_depth=case["depth"])
        got = {"image": out["image"], "alpha": out["alpha"]}
        if case["depth"]:
            got["depth"] = out["depth"]
        return got
    if kind == "iter":
        out = s["model"].render(s["camera"], antialias=case["antialias"])
        loss = l1_loss(out["image"], s["target"])
        return {"image": out["image"].detach(), "loss": loss.detach(),
                "grads": _backward(loss, s["model"].params)}
    if kind == "lens":
        p = s["params"]
        out = render_gaussians(s["camera"], p["means"], p["quats"], p["scales"], p["opacities"],
                               sh=p["sh"], sh_degree=case["degree"], antialias=case["antialias"],
                               projection="ut", refine_tiles=case["refine"])
        loss = l1_loss(out["image"], s["target"])
        return {"image": out["image"].detach(), "loss": loss.detach(),
                "grads": _backward(loss, p)}
    if kind == "features":
        p = s["params"]
        out = render_gaussian_features(s["camera"], p["means"], p["quats"], p["scales"],
                                       p["opacities"], p["features"], normalize=case["normalize"],
                                       return_depth=case["depth"])
        loss = l1_loss(out["features"], s["target"])
        got = {"features": out["features"].detach(), "alpha": out["alpha"].detach(),
               "loss": loss.detach(), "grads": _backward(loss, p)}
        if case["depth"]:
            got["depth"] = out["depth"]
        return got
    trainer = s["trainer"]
    stats = trainer.step(s["camera"], s["target"])
    got = {"loss": stats["loss"]}
    for k in GROUPS:
        state = trainer.optimizers[k].state[k]
        got[k] = {"value": trainer.model.params[k], "m": state["m"], "v": state["v"]}
    if case["collect"]:
        got["statistics"] = {"accum": trainer.grad_accum, "count": trainer.grad_count}
    return got


def work(case):
    n, pixels, kind = case["n"], case["width"] * case["height"], case["kind"]
    C = case.get("channels", 3)
    floats = 11 + (C if kind == "features" else 3 * (case["degree"] + 1) ** 2)
    geometry = 5 if case.get("method") == "2dgs" else 0
    # Gaussians that a pixel composites, as these scenes have them on average
    depth = {"blob": 40, "box": 50, "shells": 60, "heavy": 25}[case["scene"]]
    forward = n * (300 + 2 * floats) + pixels * depth * (25 + 2 * (C + geometry))
    size = 4 * n * floats
    if kind == "view":
        return {"bytes": size + 4 * pixels * (C + 1 + case["depth"]), "flops": forward}
    flops = 3 * forward
    image = 4 * pixels * (2 * C + 1)  # the image and its target
    if kind == "train":
        # parameters and both moments, read and written; a window of the loss
        return {"bytes": 6 * size + image,
                "flops": flops + pixels * C * 300 + 12 * n * floats}
    return {"bytes": 2 * size + image, "flops": flops}


def tolerance(case):
    # Against 64 bits, images are off by up to 1e-5 and gradients by up to
    # 9e-4 (surfels: 8e-3, their footprints are nearly singular), mostly from
    # the few pixels and Gaussians on the other side of the alpha or
    # transmittance threshold ("max"); sums in another order alone change
    # gradients by 1e-6 to 6e-6.
    if case["kind"] == "view":
        return {"rel": 4e-5, "max": 0.1}
    return {"rel": 1e-2, "max": 0.2} if case.get("method") == "2dgs" else {"rel": 3e-3, "max": 0.1}


# ------------------------------------------------- the same values in 64 bits
def _rotation(q):
    q = q / q.norm(dim=1, keepdim=True)
    w, x, y, z = q.unbind(1)
    return torch.stack([1 - 2 * (y * y + z * z), 2 * (x * y - w * z), 2 * (x * z + w * y),
                        2 * (x * y + w * z), 1 - 2 * (x * x + z * z), 2 * (y * z - w * x),
                        2 * (x * z - w * y), 2 * (y * z + w * x), 1 - 2 * (x * x + y * y)],
                       1).view(-1, 3, 3)


def _mul3(a, b):
    """(..., 3, 3) products as sums (no library product)."""
    return (a[..., :, :, None] * b[..., None, :, :]).sum(-2)


def _distort(case, x, y):
    if case.get("lens") == "fisheye":
        r = torch.sqrt(x * x + y * y)
        th = torch.atan(r)
        k1, k2, k3, k4 = FISHEYE
        t2 = th * th
        s = th * (1 + t2 * (k1 + t2 * (k2 + t2 * (k3 + t2 * k4)))) / r.clamp(min=1e-9)
        return x * s, y * s
    if case.get("lens") == "brown":
        k1, k2, p1, p2, k3 = BROWN
        r2 = x * x + y * y
        s = 1 + r2 * (k1 + r2 * (k2 + r2 * k3))
        return (x * s + 2 * p1 * x * y + p2 * (r2 + 2 * x * x),
                y * s + p1 * (r2 + 2 * y * y) + 2 * p2 * x * y)
    return x, y


def _project64(case, cam, means, quats, scales):
    """Screen means, conics, camera z, radii and antialiasing factors."""
    R, t = cam["R"].double().cuda(), cam["t"].double().cuda()
    f, cx, cy = cam["f"], cam["cx"], cam["cy"]

    def to_camera(p):
        return (p[..., None, :] * R).sum(-1) + t

    pc = to_camera(means)
    z = pc[:, 2]
    axes = _rotation(quats) * scales[:, None, :]  # columns
    if case["kind"] == "lens":
        off = math.sqrt(3.0) * axes.transpose(1, 2)
        q = to_camera(means[:, None, :] + torch.cat([off, -off], 1))
        x, y = _distort(case, q[..., 0] / q[..., 2], q[..., 1] / q[..., 2])
        u6, v6 = f * x + cx, f * y + cy
        u, v = u6.mean(1), v6.mean(1)
        du, dv = u6 - u[:, None], v6 - v[:, None]
        a0, b, c0 = (du * du).mean(1), (du * dv).mean(1), (dv * dv).mean(1)
    else:
        zs = z.clamp(min=1e-6)
        u, v = f * pc[:, 0] / zs + cx, f * pc[:, 1] / zs + cy
        lx, ly = 1.3 * (0.5 * case["width"] / f), 1.3 * (0.5 * case["height"] / f)
        tx, ty = (pc[:, 0] / zs).clamp(-lx, lx) * zs, (pc[:, 1] / zs).clamp(-ly, ly) * zs
        M = (R[None, :, :, None] * axes[:, None, :, :]).sum(2)  # camera-space axes
        ju = (f / zs)[:, None] * M[:, 0] - (f * tx / zs ** 2)[:, None] * M[:, 2]
        jv = (f / zs)[:, None] * M[:, 1] - (f * ty / zs ** 2)[:, None] * M[:, 2]
        a0, b, c0 = (ju * ju).sum(1), (ju * jv).sum(1), (jv * jv).sum(1)
    a, c = a0 + 0.3, c0 + 0.3
    det = a * c - b * b
    ds = det.clamp(min=1e-12)
    comp = torch.ones_like(det)
    if case.get("antialias"):
        comp = torch.sqrt((a0 * c0 - b * b).clamp(min=0.0) / ds)
    mid = 0.5 * (a + c)
    radius = torch.ceil(3 * torch.sqrt(mid + torch.sqrt((mid * mid - det).clamp(min=0.01))))
    valid = (z > float(torch.tensor(0.01).float())) & (det > 0)
    return (torch.stack([u, v], 1), torch.stack([c / ds, -b / ds, a / ds], 1), z,
            torch.where(valid, radius, 0.0).detach(), torch.where(valid, comp, 0.0))


def _colour64(case, cam, means, sh):
    """max(0, 0.5 + the SH expansion) along the view directions (no gradient to the means)."""
    center = -(cam["R"].double() * cam["t"].double()[:, None]).sum(0).cuda()
    d = means.detach() - center
    x, y, z = (d / d.norm(dim=1, keepdim=True).clamp(min=1e-8)).unbind(1)
    xx, yy, zz = x * x, y * y, z * z
    basis = [torch.full_like(x, 0.28209479177387814)]
    if case["degree"] > 0:
        k = 0.4886025119029199
        basis += [-k * y, k * z, -k * x]
    if case["degree"] > 1:
        k = 1.0925484305920792
        basis += [k * x * y, -k * y * z, 0.31539156525252005 * (2 * zz - xx - yy), -k * x * z,
                  0.5462742152960396 * (xx - yy)]
    if case["degree"] > 2:
        a, b, c = 0.5900435899266435, 2.890611442640554, 0.4570457994644658
        basis += [-a * y * (3 * xx - yy), b * x * y * z, -c * y * (4 * zz - xx - yy),
                  0.3731763325901154 * z * (2 * zz - 3 * xx - 3 * yy),
                  -c * x * (4 * zz - xx - yy), 0.5 * b * z * (xx - yy), -a * x * (xx - 3 * yy)]
    return (0.5 + (torch.stack(basis, 1)[:, :, None] * sh).sum(1)).clamp(min=0.0)


def _lists64(case, xy, radius, z):
    """(ids, start, count per tile): each tile's Gaussians front to back."""
    W, H = case["width"], case["height"]
    tx, ty = -(-W // TILE), -(-H // TILE)
    x, y, r = xy[:, 0], xy[:, 1], radius
    on = (r > 0) & (x + r >= 0) & (x - r < W) & (y + r >= 0) & (y - r < H)
    x0, x1 = (torch.floor((x + s * r) / TILE).clamp(0, tx - 1).long() for s in (-1, 1))
    y0, y1 = (torch.floor((y + s * r) / TILE).clamp(0, ty - 1).long() for s in (-1, 1))
    order = torch.argsort(z.float(), stable=True)
    order = order[on[order]]
    w = (x1 - x0 + 1)[order]
    count = w * (y1 - y0 + 1)[order]
    rank = torch.repeat_interleave(torch.arange(order.numel(), device="cuda"), count)
    k = torch.arange(rank.numel(), device="cuda") - (torch.cumsum(count, 0) - count)[rank]
    tile = (y0[order][rank] + k // w[rank]) * tx + x0[order][rank] + k % w[rank]
    tile, by = torch.sort(tile, stable=True)
    num = torch.bincount(tile, minlength=tx * ty)
    return order[rank[by]], torch.cumsum(num, 0) - num, num


def _chunks(num, most):
    """Tiles of similar list length, at most `most` (entry, pixel) pairs a group."""
    by = torch.argsort(num, descending=True)
    lengths = num[by].tolist()
    at = 0
    while at < len(lengths) and lengths[at] > 0:
        size = max(1, min(len(lengths) - at, most // (256 * lengths[at])))
        tiles = by[at:at + size]
        yield tiles[num[tiles] > 0], lengths[at]
        at += size


def _weights64(case, lists, tiles, length, xy, conic, opacity):
    """The group's (ids, pixel index, inside, dx, dy, G, alpha, T, keep), T in front of each entry."""
    ids, start, num = lists
    W, H = case["width"], case["height"]
    k = torch.arange(length, device="cuda")
    on = k[None, :] < num[tiles][:, None]
    g = ids[(start[tiles][:, None] + k[None, :]).clamp(max=ids.numel() - 1)]
    q = torch.arange(256, device="cuda")
    tx = -(-W // TILE)
    px = (tiles % tx)[:, None] * TILE + q[None, :] % TILE
    py = (tiles // tx)[:, None] * TILE + q[None, :] // TILE
    inside = (px < W) & (py < H)
    pid = torch.where(inside, py * W + px, 0)
    dx = xy[g, 0][:, :, None] - (px[:, None, :] + 0.5)
    dy = xy[g, 1][:, :, None] - (py[:, None, :] + 0.5)
    c = conic[g]
    G = torch.exp(-0.5 * (c[:, :, 0, None] * dx * dx + c[:, :, 2, None] * dy * dy)
                  - c[:, :, 1, None] * dx * dy)
    alpha = (opacity[g][:, :, None] * G).clamp(max=0.99)
    alpha = torch.where((alpha >= 1.0 / 255.0) & on[:, :, None], alpha, 0.0)
    after = torch.cumprod(1.0 - alpha, 1)
    T = torch.cat([torch.ones_like(after[:, :1]), after[:, :-1]], 1)
    keep = torch.cumsum((after < 1e-4).to(torch.int32), 1) == 0  # before the first crossing
    return g, pid, inside, dx, dy, G, torch.where(keep, alpha, 0.0), torch.where(keep, T, 0.0), keep


def _composite64(case, lists, xy, conic, opacity, feats, depths):
    """(sums of weighted features, transmittance left, weighted depth) per pixel."""
    pixels = case["width"] * case["height"]
    out = torch.zeros(pixels, feats.shape[1], dtype=torch.float64, device="cuda")
    left = torch.ones(pixels, dtype=torch.float64, device="cuda")
    deep = torch.zeros_like(left)
    for tiles, length in _chunks(lists[2], 1 << 26):
        g, pid, inside, _, _, _, alpha, T, _ = _weights64(case, lists, tiles, length, xy, conic,
                                                          opacity)
        w = (alpha * T).transpose(1, 2).contiguous()
        at = pid[inside]
        out[at] = torch.bmm(w, feats[g])[inside]
        left[at] = torch.prod(1.0 - alpha, 1)[inside]
        deep[at] = (w * depths[g][:, None, :]).sum(2)[inside]
    return out, left, deep


def _composite64_bwd(case, lists, xy, conic, opacity, feats, left, g_out, g_left):
    """Gradients of the composite: screen means, conics, opacities, features.  The clamp of
    alpha at 0.99 passes the gradient on, as the framework's does."""
    gx, gc = torch.zeros_like(xy), torch.zeros_like(conic)
    go, gf = torch.zeros_like(opacity), torch.zeros_like(feats)
    for tiles, length in _chunks(lists[2], 1 << 25):
        g, pid, inside, dx, dy, G, alpha, T, keep = _weights64(case, lists, tiles, length, xy,
                                                               conic, opacity)
        cot = torch.where(inside[:, :, None], g_out[pid], 0.0)
        rest = torch.where(inside, (left * g_left)[pid], 0.0)
        w = alpha * T
        cg = torch.bmm(feats[g], cot.transpose(1, 2).contiguous())
        s = w * cg
        later = s.sum(1, keepdim=True) - torch.cumsum(s, 1) + rest[:, None, :]
        live = alpha > 0
        da = torch.where(live, T * cg - later / (1.0 - alpha), 0.0)
        dG = da * G
        d = opacity[g][:, :, None] * dG  # cotangent of the power
        c = conic[g]
        a, b, cc = c[:, :, 0, None], c[:, :, 1, None], c[:, :, 2, None]
        flat = g.reshape(-1)
        gx.index_add_(0, flat, torch.stack([-(d * (a * dx + b * dy)).sum(2),
                                            -(d * (b * dx + cc * dy)).sum(2)], 2).view(-1, 2))
        gc.index_add_(0, flat, torch.stack([-0.5 * (d * dx * dx).sum(2), -(d * dx * dy).sum(2),
                                            -0.5 * (d * dy * dy).sum(2)], 2).view(-1, 3))
        go.index_add_(0, flat, dG.sum(2).view(-1))
        gf.index_add_(0, flat, torch.bmm(w, cot).view(-1, feats.shape[1]))
    return gx, gc, go, gf


def _blur64(x):
    """Separable Gaussian window (11, sigma 1.5) with zero padding, over (H, W, C)."""
    k = torch.exp(-0.5 * (torch.arange(11, dtype=torch.float64) - 5) ** 2 / 1.5 ** 2)
    k = (k / k.sum()).tolist()
    H, W = x.shape[:2]
    p = torch.nn.functional.pad(x, (0, 0, 5, 5))
    x = sum(k[i] * p[:, i:i + W] for i in range(11))
    p = torch.nn.functional.pad(x, (0, 0, 0, 0, 5, 5))
    return sum(k[i] * p[i:i + H] for i in range(11))


def _ssim64(p, t):
    mp, mt = _blur64(p), _blur64(t)
    vp, vt, c = _blur64(p * p) - mp * mp, _blur64(t * t) - mt * mt, _blur64(p * t) - mp * mt
    return ((2 * mp * mt + 1e-4) * (2 * c + 9e-4)
            / ((mp * mp + mt * mt + 1e-4) * (vp + vt + 9e-4))).mean()


def _geometry64(case, cam, F, alpha):
    """Depth variance and normal consistency of the rendered surfels."""
    W, H = case["width"], case["height"]
    ok = (alpha > 0.05).double()
    var = ((F[..., 1] - F[..., 0] ** 2).clamp(min=0.0) * ok).sum() / ok.sum().clamp(min=1.0)
    x = ((torch.arange(W, device="cuda").double() + 0.5 - cam["cx"]) / cam["f"]).expand(H, W)
    y = ((torch.arange(H, device="cuda").double() + 0.5 - cam["cy"]) / cam["f"])[:, None].expand(H, W)
    pc = torch.stack([x, y, torch.ones_like(x)], 2) * F[..., :1] - cam["t"].double().cuda()
    P = (pc[..., :, None] * cam["R"].double().cuda()).sum(-2)

    def unit(v):
        return v / v.norm(dim=-1, keepdim=True).clamp(min=1e-8)

    n = unit(torch.linalg.cross(P[:-1, 1:] - P[:-1, :-1], P[1:, :-1] - P[:-1, :-1]))
    quad = ok[:-1, :-1] * ok[:-1, 1:] * ok[1:, :-1] * ok[1:, 1:]
    off = 1.0 - (unit(F[:-1, :-1, 2:5]) * n).sum(-1).abs()
    return 0.1 * var + 0.05 * (off * quad).sum() / quad.sum().clamp(min=1.0)


def exact(case, seed):
    kind = case["kind"]
    p, cam, target = _inputs(case, seed)
    if kind in ("lens", "features"):  # the call takes activated values
        p["scales"], p["opacities"] = torch.exp(p["scales"]), torch.sigmoid(p["opacities"])
    if case.get("morton"):
        # the table's rows as the framework stores them: a pure reordering of the inputs
        m = GaussianModel({k: p[k] for k in GROUPS}, sh_degree=case["degree"])
        m.reorder_spatial()
        p = dict(m.params)
    raw = {k: v.double().requires_grad_(True) for k, v in p.items()}
    if kind == "lens":
        raw["sh"] = torch.cat([raw.pop("sh_dc"), raw.pop("sh_rest")], 1).detach().requires_grad_(True)
    direct = kind in ("lens", "features")
    scales = raw["scales"] if direct else torch.exp(raw["scales"])
    opac = raw["opacities"] if direct else torch.sigmoid(raw["opacities"])
    xy, conic, z, radius, comp = _project64(case, cam, raw["means"], raw["quats"], scales)
    oe = opac * comp
    if kind == "features":
        feats = raw["features"]
    else:
        sh = raw["sh"] if kind == "lens" else torch.cat([raw["sh_dc"], raw["sh_rest"]], 1)
        feats = _colour64(case, cam, raw["means"], sh)
    surfels = case.get("method") == "2dgs"
    if surfels:
        n = _rotation(raw["quats"])[:, :, 2]
        center = -(cam["R"].double() * cam["t"].double()[:, None]).sum(0).cuda()
        facing = (n * (center - raw["means"].detach())).sum(1, keepdim=True) < 0
        feats = torch.cat([feats, z[:, None], z[:, None] ** 2, torch.where(facing, -n, n)], 1)
    flat = [v.detach().contiguous() for v in (xy, conic, oe, feats)]
    lists = _lists64(case, flat[0], radius, z.detach())
    out, left, deep = _composite64(case, lists, *flat, z.detach())
    H, W = case["height"], case["width"]
    out.requires_grad_(True)
    left.requires_grad_(True)
    image, alpha = out.view(H, W, -1), 1.0 - left.view(H, W)
    depth = torch.where(alpha > 1e-6, deep.view(H, W) / alpha.clamp(min=1e-6), 0.0).detach()
    if kind == "view":
        got = {"image": image.detach(), "alpha": alpha.detach()}
        if case["depth"]:
            got["depth"] = depth
        return got
    t64 = target.double()
    if case.get("normalize"):
        image = torch.where(alpha[..., None] > 1e-6, image / alpha[..., None].clamp(min=1e-6), 0.0)
    if kind == "train":
        rgb = image[..., :3]
        loss = (1 - LAMBDA) * (rgb - t64).abs().mean() + LAMBDA * (1 - _ssim64(rgb, t64))
        if surfels:
            a = alpha[..., None]
            loss = loss + _geometry64(
                case, cam, torch.where(a > 1e-6, image[..., 3:] / a.clamp(min=1e-6), 0.0),
                alpha.detach())
    else:
        loss = (image - t64).abs().mean()
    g_out, g_left = torch.autograd.grad(loss, (out, left), allow_unused=True)
    g_left = torch.zeros_like(left) if g_left is None else g_left
    gx, gc, go, gf = _composite64_bwd(case, lists, *flat, left.detach(), g_out, g_left)
    names = list(raw)
    grads = dict(zip(names, torch.autograd.grad((xy, conic, oe, feats), [raw[k] for k in names],
                                                (gx, gc, go, gf), allow_unused=True)))
    grads = {k: torch.zeros_like(raw[k]) if g is None else g for k, g in grads.items()}
    if kind != "train":
        if kind == "iter":
            grads = {k: grads[k] for k in GROUPS}
        elif kind == "features":
            grads = {k: grads[k] for k in ("means", "quats", "scales", "opacities", "features")}
        name = "features" if kind == "features" else "image"
        got = {name: image.detach(), "loss": loss.detach(), "grads": grads}
        if kind == "features":
            got["alpha"] = alpha.detach()
            if case["depth"]:
                got["depth"] = depth
        return got
    got = {"loss": float(loss.detach())}
    for k in GROUPS:  # the first Adam update
        m, v = 0.1 * grads[k], 0.001 * grads[k] ** 2
        value = raw[k].detach() - RATES[k] * m / (torch.sqrt(v) + 1e-15)
        if surfels and k == "scales":
            value[:, 2].clamp_(max=math.log(THICKNESS))
        got[k] = {"value": value, "m": m, "v": v}
    if case["collect"]:
        seen = (radius > 0).double()
        size = 0.5 * torch.tensor([W, H], dtype=torch.float64, device="cuda")
        got["statistics"] = {"accum": (gx * size).norm(dim=1) * seen, "count": seen}
    return got

"""The workloads whose time on the GPU matters, each as a user's program calls the package.

A case is a plain dict:

  path     "raster"   rasterize_projected_gaussians (2D splats)
           "pinhole"  rasterize_pinhole_gaussians (3D splats, projection included)
           "project"  project_pinhole_gaussians alone
  train    forward and backward (every gradient comes back), or an image under no_grad
  H, W, B, G   image size, images, splats per image
  lo, hi   2D standard deviations in pixels, uniform
  cluster  80% of the means in eight clusters of 20 px, depths on ten planes (2D)
  logit    mean of the opacity's logit (0: opacities around 0.5; -2: translucent, long tile lists)
  pose     the camera pose is a parameter too (its gradient comes back)
"""
import math
import os
import sys

import torch

sys.path.insert(0, os.path.join(os.getcwd(), "fast-mac-gsplat_amd"))
import torch_gsplat_bridge_fast as gs  # noqa: E402

THRESHOLD = 1.0 / 255.0
STOP = 1e-4
MAX_ALPHA = 0.99
NEAR = 1e-4


def _raster(name, train, H, W, B, G, lo, hi, cluster=False, logit=0.0):
    return dict(name=name, path="raster", train=train, H=H, W=W, B=B, G=G, lo=lo, hi=hi, cluster=cluster,
                logit=logit, pose=False)


def _pinhole(name, train, H, W, B, G, logit=0.0, pose=False, path="pinhole"):
    return dict(name=name, path=path, train=train, H=H, W=W, B=B, G=G, lo=0.0, hi=0.0, cluster=False, logit=logit,
                pose=pose)


def listed():
    return [
        # a thumbnail or a preview while something is edited: nothing but the call's own cost
        _raster("eval_thumb", False, 96, 131, 1, 300, 1.0, 8.0),
        # fitting a small image, thousands of steps: launches and host time
        _raster("train_512sq_512", True, 512, 512, 1, 512, 1.0, 8.0),
        # a batch of ragged small images in one call (dataset crops)
        _raster("train_ragged_b5", True, 203, 341, 5, 4001, 0.5, 6.0),
        # ordinary screen size, 64K splats: a training step and a frame
        _raster("train_1080p_64k", True, 1080, 1920, 1, 65536, 0.5, 6.0),
        _raster("eval_1080p_64k", False, 1080, 1920, 1, 65536, 0.5, 6.0),
        # the headline size: a training step and a frame at 4096 x 4096
        _raster("train_4096sq_64k", True, 4096, 4096, 1, 65536, 1.0, 12.0),
        _raster("eval_4096sq_64k", False, 4096, 4096, 1, 65536, 1.0, 12.0),
        # hot tiles: most splats of four images in a few clusters
        _raster("train_clustered_b4", True, 512, 1024, 4, 65536, 1.0, 8.0, cluster=True),
        # a frame of a translucent 3D scene (low opacities: long lists before a pixel is opaque)
        _pinhole("eval_3d_translucent", False, 1080, 1920, 1, 200003, logit=-2.0),
        # fitting a 3D scene and the camera poses, two views a step, odd sizes
        _pinhole("train_3d_pose_b2", True, 822, 1237, 2, 100003, pose=True),
        # the largest: a training step of a million 3D splats at 4096 x 4096
        _pinhole("train_3d_4096sq_1m", True, 4096, 4096, 1, 1 << 20),
        # the projection by itself, for a program with a rasterizer or culling of its own
        _pinhole("project_1m", True, 4096, 4096, 1, 1 << 20, path="project"),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.random()
    if kind < 0.10:
        c = _pinhole("", True, 1080, 1920, rng.choice((1, 1, 2)), _log(rng, 1000, 500000), path="project",
                     pose=rng.random() < 0.5)
    elif kind < 0.40:
        W = _log(rng, 320, 4096)
        H = max(200, min(4096, int(W * rng.uniform(0.5, 1.1))))
        B = rng.choice((1, 1, 1, 2)) if W <= 2048 else 1
        logit = rng.choice((0.0, 0.0, 0.0, -2.0))
        most = (1 << 17 if logit else 1 << 19) // B
        c = _pinhole("", rng.random() < 0.6, H, W, B, min(_log(rng, 5000, most), max(5000, H * W // 4)), logit=logit,
                     pose=rng.random() < 0.3)
    elif kind < 0.52:
        W = _log(rng, 400, 1400)
        H = max(200, int(W * rng.uniform(0.5, 1.0)))
        B = rng.choice((1, 2, 3, 4))
        c = _raster("", rng.random() < 0.7, H, W, B, min(_log(rng, 4000, 65536), H * W // 8), 1.0, 8.0, cluster=True)
    else:
        W = _log(rng, 96, 4096)
        H = max(64, min(4096, int(W * rng.uniform(0.5, 1.3))))
        B = rng.choice((1, 1, 1, 2, 4, 7))
        B = max(1, min(B, (1 << 24) // (H * W)))
        G = min(_log(rng, 200, 131072), max(200, H * W // 8))
        G = max(1, min(G, (1 << 18) // B))
        hi = round(rng.uniform(4.0, 12.0), 2)
        c = _raster("", rng.random() < 0.6, H, W, B, G, round(rng.uniform(0.5, 1.0), 2), hi,
                    logit=rng.choice((0.0, 0.0, 0.0, -1.0)))
    c.pop("name")
    return c


# --- inputs -----------------------------------------------------------------------------------


def _rand(g, *shape):
    return torch.rand(*shape, generator=g, device=g.device)


def _normal(g, *shape):
    return torch.randn(*shape, generator=g, device=g.device)


def _scene_2d(case, seed):
    """Means uniform over the image (or clustered), sigmas U(lo, hi), any angle, opacities
    sigmoid(N(logit, 1)), depths U(0.1, 10) (clustered: on ten planes)."""
    g = torch.Generator(device="cuda").manual_seed(seed)
    H, W, B, G = case["H"], case["W"], case["B"], case["G"]
    size = torch.tensor([W, H], dtype=torch.float32, device="cuda")
    means = _rand(g, B, G, 2) * size
    depths = 0.1 + 9.9 * _rand(g, B, G)
    if case["cluster"]:
        centres = _rand(g, B, 8, 2) * size
        which = torch.randint(0, 8, (B, G), generator=g, device="cuda")
        near = torch.gather(centres, 1, which[..., None].expand(B, G, 2)) + 20.0 * _normal(g, B, G, 2)
        means = torch.where(_rand(g, B, G, 1) < 0.8, near, means)
        depths = torch.randint(1, 11, (B, G), generator=g, device="cuda") + 0.05 * _normal(g, B, G)
    sigma = case["lo"] + (case["hi"] - case["lo"]) * _rand(g, B, G, 2)
    angle = math.pi * _rand(g, B, G)
    c, s = torch.cos(angle), torch.sin(angle)
    ix, iy = sigma[..., 0] ** -2, sigma[..., 1] ** -2
    conics = torch.stack([c * c * ix + s * s * iy, c * s * (ix - iy), s * s * ix + c * c * iy], dim=-1)
    opacities = torch.sigmoid(case["logit"] + _normal(g, B, G))
    t = [means, conics, _rand(g, B, G, 3), opacities, depths]
    return [x[0].contiguous() if B == 1 else x.contiguous() for x in t], g


def _scene_3d(case, seed):
    """Means uniform in a cube of side 10 seen from 15 away, log-normal scales around 0.05 with a
    tenth of the splats ten times as large, any rotation."""
    g = torch.Generator(device="cuda").manual_seed(seed)
    W, H, B, G = case["W"], case["H"], case["B"], case["G"]
    means = 10.0 * _rand(g, B, G, 3) - 5.0
    scales = torch.exp(-3.0 + 0.5 * _normal(g, B, G, 3))
    scales = torch.where(_rand(g, B, G, 1) < 0.1, 10.0 * scales, scales)
    quats = torch.nn.functional.normalize(_normal(g, B, G, 4), dim=-1)
    opacities = torch.sigmoid(case["logit"] + _normal(g, B, G))
    colors = _rand(g, B, G, 3)
    c2w = torch.eye(4, device="cuda").repeat(B, 1, 1)
    c2w[:, 2, 3] = -15.0
    c2w[:, :2, 3] = 0.2 * _normal(g, B, 2)
    t = [means, scales, quats, opacities, colors, c2w]
    f = 3500.0 * W / 4096.0
    return [x[0].contiguous() if B == 1 else x.contiguous() for x in t], (f, f, W / 2.0, H / 2.0), g


def prepare(case, seed):
    H, W, B, G = case["H"], case["W"], case["B"], case["G"]
    lead = () if B == 1 else (B,)
    s = {"case": case, "config": gs.RasterConfig(height=H, width=W, background=(0.1, 0.2, 0.3))}
    if case["path"] == "raster":
        t, g = _scene_2d(case, seed)
        s["inputs"], s["leaves"] = t, t[:4]
    else:
        t, s["camera"], g = _scene_3d(case, seed)
        s["inputs"] = t
        s["leaves"] = t[:4] if case["path"] == "project" else t[:5]
        if case["pose"]:
            s["leaves"] = s["leaves"] + [t[5]]
    if case["train"]:
        for x in s["leaves"]:
            x.requires_grad_(True)
        if case["path"] == "project":
            # the sizes of gradients that a rasterizer gives back
            s["weights"] = [_normal(g, *lead, G, 2), _normal(g, *lead, G, 3), _normal(g, *lead, G),
                            _normal(g, *lead, G)]
        else:
            s["weights"] = _rand(g, *lead, H, W, 3)
    return s


def _forward(s):
    t, path = s["inputs"], s["case"]["path"]
    if path == "raster":
        return gs.rasterize_projected_gaussians(*t, s["config"])
    if path == "pinhole":
        return gs.rasterize_pinhole_gaussians(*t[:5], *s["camera"], camera_to_world=t[5], near_plane=NEAR,
                                              config=s["config"])
    return gs.project_pinhole_gaussians(*t[:4], *s["camera"], camera_to_world=t[5], near_plane=NEAR)


def run(s):
    if not s["case"]["train"]:
        with torch.no_grad():
            return _forward(s)
    for x in s["leaves"]:
        x.grad = None
    out = _forward(s)
    if s["case"]["path"] == "project":
        torch.autograd.backward(out, s["weights"])
        return [x.detach() for x in out], [x.grad for x in s["leaves"]]
    out.backward(s["weights"])
    return out.detach(), [x.grad for x in s["leaves"]]


# --- what a pass cannot do without ------------------------------------------------------------


def work(case):
    """bytes: the inputs once, the image once, for training its gradient once and the gradients
    once.  flops: 24 for each pixel a splat is visible at in the forward and 60 in the backward (an
    ellipse of 2 pi ln(255 o) sx sy pixels, o around its median), no more than the layers after
    which a pixel is opaque; about 150 and 400 a splat for the projection."""
    H, W, B, G = case["H"], case["W"], case["B"], case["G"]
    px, n = B * H * W, B * G
    o = 1.0 / (1.0 + math.exp(-case["logit"]))
    if case["path"] == "raster":
        area = 2.0 * math.pi * max(math.log(255.0 * o), 0.5) * ((case["lo"] + case["hi"]) / 2.0) ** 2
        inout, grads, flops = 40 * n, 36 * n, 0
    else:
        # scale 0.05 (0.5 for a tenth) at distance 15
        s = 3500.0 * W / 4096.0 * 0.05 / 15.0
        area = 2.0 * math.pi * max(math.log(255.0 * o), 0.5) * (0.9 * s * s + 0.1 * 100.0 * s * s + 0.3)
        flops = (550 if case["train"] else 150) * n
        if case["path"] == "project":
            return {"bytes": 44 * n + 28 * n + ((28 + 44 + 44) * n if case["train"] else 0), "flops": flops}
        inout, grads = 56 * n, 56 * n
    layers = math.log(1.0 / STOP) / -math.log(1.0 - o / 2.0)
    seen = min(area * n, layers * px)
    return {"bytes": inout + 12 * px + (12 * px + grads if case["train"] else 0),
            "flops": flops + (84 if case["train"] else 24) * seen}


def tolerance(case):
    """32-bit sums give 5e-7 (the gradients are atomic sums: the same inputs twice differ by that).
    Four times the difference from 64 bits leaves room for the decisions that rounding can turn at
    single pixels: a visible splat at the threshold (1e-5 of the result), in 3D the order of two
    splats at the same depth too.  Whole splats never differ by much against the largest values."""
    if case["path"] == "project":
        return {"rel": 6e-6, "max": 1e-2}
    return {"rel": 4e-5 if case["path"] == "raster" else 2e-4, "max": 5e-2}


# --- the same in 64 bits ----------------------------------------------------------------------


def _project64(means, scales, quats, opacities, c2w, camera):
    r, i, j, k = quats.unbind(-1)
    rot = torch.stack([1 - 2 * (j * j + k * k), 2 * (i * j - r * k), 2 * (i * k + r * j),
                       2 * (i * j + r * k), 1 - 2 * (i * i + k * k), 2 * (j * k - r * i),
                       2 * (i * k - r * j), 2 * (j * k + r * i), 1 - 2 * (i * i + j * j)], dim=-1)
    m = rot.reshape(*quats.shape[:-1], 3, 3) * scales[..., None, :]
    world = c2w[:, None, :3, :3]
    cam = ((means - c2w[:, None, :3, 3])[..., None, :] @ world)[..., 0, :]
    m = world.transpose(-1, -2) @ m
    x, y, z = cam.unbind(-1)
    front = z > NEAR
    z1 = torch.where(front, z, torch.ones_like(z))
    x, y = torch.where(front, x, 0 * x), torch.where(front, y, 0 * y)
    fx, fy, cx, cy = camera
    jac = torch.stack([torch.stack([fx / z1, 0 * z1, -fx * x / z1 ** 2], -1),
                       torch.stack([0 * z1, fy / z1, -fy * y / z1 ** 2], -1)], -2)
    half = jac @ m
    cov = half @ half.transpose(-1, -2)
    a, b, c = cov[..., 0, 0] + 0.3, cov[..., 0, 1], cov[..., 1, 1] + 0.3
    det = torch.clamp(a * c - b * b, min=1e-6)
    return (torch.stack([fx * x / z1 + cx, fy * y / z1 + cy], -1), torch.stack([c / det, -b / det, a / det], -1),
            torch.where(front, opacities, 0 * opacities), z)


def _lists(means, conics, opacities, depths, H, W):
    """Splats of each 16 x 16 tile in depth order: every tile that the box of the pixels where alpha
    can reach the threshold touches.  The box is the rasterizer's own: it takes the conic's
    determinant as 1e-8 at least, which cuts splats of over about a hundred pixels off.  Returns the
    splat of each pair, and where each tile starts."""
    G = means.shape[0]
    a, b, c = conics.unbind(-1)
    det = torch.clamp(a * c - b * b, min=1e-8)
    ok = opacities > THRESHOLD
    tau = 2.0 * torch.log(torch.where(ok, opacities, torch.ones_like(opacities)) / THRESHOLD)
    ex, ey = torch.sqrt(tau * c / det), torch.sqrt(tau * a / det)
    nx, ny = (W + 15) // 16, (H + 15) // 16

    def span(m, e, pixels):
        lo = torch.floor(m - e - 0.5).clamp(0, pixels).long()
        hi = torch.ceil(m + e - 0.5).clamp(-1, pixels - 1).long()
        return lo // 16, torch.where(hi >= lo, hi // 16 - lo // 16 + 1, 0 * lo)

    tx, wx = span(means[:, 0], ex, W)
    ty, wy = span(means[:, 1], ey, H)
    order = torch.argsort(depths, stable=True)
    tx, ty, wx = tx[order], ty[order], wx[order]
    count = torch.where(ok[order], wx * wy[order], 0 * wx)
    first = torch.cumsum(count, 0) - count
    rank = torch.repeat_interleave(torch.arange(G, device=means.device), count)
    k = torch.arange(rank.numel(), device=means.device) - first[rank]
    w = wx[rank]
    tile = (ty[rank] + k // w) * nx + tx[rank] + k % w
    del k, w
    tile, at = torch.sort(tile.int(), stable=True)
    splat = order[rank[at]].int()
    starts = torch.searchsorted(tile, torch.arange(nx * ny + 1, device=means.device, dtype=torch.int32))
    return splat, starts


def _alphas(p, ids, px, py):
    """Alpha of splats ids [t, k] at the pixels px, py [t, 256] -> [t, k, 256]; -1 is no splat."""
    means, conics, _, opacities = p
    i = ids.clamp(min=0).long()
    dx, dy = px[:, None] - means[i][..., 0, None], py[:, None] - means[i][..., 1, None]
    q = conics[i]
    power = -0.5 * (q[..., 0, None] * dx * dx + 2 * q[..., 1, None] * dx * dy + q[..., 2, None] * dy * dy)
    alpha = torch.clamp(opacities[i][..., None] * torch.exp(power), max=MAX_ALPHA)
    seen = (power <= 0) & (alpha >= THRESHOLD) & (ids >= 0)[..., None]
    return torch.where(seen, alpha, torch.zeros_like(alpha))


def _image64(p, depths, H, W, background, weights):
    """One image, and the gradients of its weighted sum (weights: None, no gradients), in 64 bits."""
    dev = depths.device
    nx, ny = (W + 15) // 16, (H + 15) // 16
    splat, starts = _lists(p[0], p[1], p[3], depths, H, W)
    if weights is not None:
        p = [x.detach().requires_grad_(True) for x in p]
    length = starts[1:] - starts[:-1]
    most = 1 << 23

    def groups(n):
        """Tiles of like list lengths, so many at a time that a [t, k, 256] tensor is small."""
        order = torch.argsort(n, descending=True)
        sizes, at = n[order].tolist(), 0
        while at < len(sizes):
            t = max(1, min(len(sizes) - at, most // (256 * max(1, sizes[at]))))
            yield order[at:at + t], sizes[at]
            at += t

    def pixels(t):
        l = torch.arange(256, device=dev)
        return (t % nx)[:, None] * 16 + l % 16, (t // nx)[:, None] * 16 + l // 16

    def ids_of(t, lo, hi):
        k = torch.arange(lo, hi, device=dev)
        inside = k < length[t][:, None]
        return torch.where(inside, splat[(starts[t][:, None] + k).clamp(max=max(0, splat.numel() - 1))],
                           torch.full_like(splat[:1], -1)) if splat.numel() else torch.full_like(inside, -1, dtype=torch.int32)

    need = length.clone()
    with torch.no_grad():  # how much of its list a tile walks before it is opaque
        step = 64
        long_tiles = torch.nonzero(length > step)[:, 0]
        for chunk in long_tiles.split(512):
            live, T, at = chunk, torch.ones(len(chunk), 256, dtype=torch.float64, device=dev), 0
            while len(live):
                x, y = pixels(live)
                T = T * torch.prod(1 - _alphas(p, ids_of(live, at, at + step), x + 0.5, y + 0.5), dim=1)
                at += step
                out = (x >= W) | (y >= H)
                stopped = ((T <= STOP) | out).all(dim=1)
                need[live[stopped]] = torch.clamp(length[live[stopped]], max=at)
                go = ~stopped & (length[live] > at)
                live, T = live[go], T[go]
    img = torch.zeros(ny * 16, nx * 16, 3, dtype=torch.float64, device=dev)
    bg = torch.tensor(background, dtype=torch.float64, device=dev)
    if weights is not None:
        wide = torch.zeros_like(img)
        wide[:H, :W] = weights
    for t, k in groups(need):
        x, y = pixels(t)
        with torch.enable_grad() if weights is not None else torch.no_grad():
            ids = ids_of(t, 0, max(1, k))
            a = _alphas(p, ids, x + 0.5, y + 0.5)
            after = torch.cumprod(1 - a.detach(), dim=1)
            before = torch.cat([torch.ones_like(after[:, :1]), after[:, :-1]], dim=1)
            a = torch.where(before > STOP, a, torch.zeros_like(a))
            logs = torch.cumsum(torch.log1p(-a), dim=1)
            T = torch.exp(torch.cat([torch.zeros_like(logs[:, :1]), logs[:, :-1]], dim=1))
            c = p[2][ids.clamp(min=0).long()]
            block = ((T * a).transpose(1, 2) @ c) + torch.exp(logs[:, -1])[..., None] * bg
            img[y, x] = block.detach()
            if weights is not None:
                (block * wide[y, x]).sum().backward()
    return img[:H, :W], None if weights is None else [x.grad if x.grad is not None else torch.zeros_like(x) for x in p]


def exact(case, seed):
    s = prepare(case, seed)
    B, path = case["B"], case["path"]

    def batch(x):
        return (x[None] if B == 1 else x).detach().double()

    def back(x):
        return x[0] if B == 1 else x

    t = [batch(x) for x in s["inputs"]]
    if path == "raster":
        flat, leaves = t, None
    else:
        leaves = [x.requires_grad_(case["train"]) for x in t[:4]]
        c2w = t[5].requires_grad_(case["train"] and case["pose"])
        m, q, o, z = _project64(*leaves, c2w, s["camera"])
        if path == "project":
            want = leaves + ([c2w] if case["pose"] else [])
            w = [batch(x) for x in s["weights"]]
            grads = torch.autograd.grad([m, q, o, z], want, w)
            return [back(x.detach()) for x in (m, q, o, z)], [back(x) for x in grads]
        flat = [m, q, t[4], o, z]
    images, grads = [], []
    for b in range(B):
        p = [x[b].detach() for x in flat[:4]]
        w = batch(s["weights"])[b] if case["train"] else None
        img, g = _image64(p, flat[4][b].detach(), case["H"], case["W"], s["config"].background, w)
        images.append(img)
        grads.append(g)
    img = back(torch.stack(images))
    if not case["train"]:
        return img
    g = [torch.stack([x[i] for x in grads]) for i in range(4)]
    if path == "raster":
        return img, [back(x) for x in g]
    want = leaves + ([c2w] if case["pose"] else [])
    got = torch.autograd.grad([m, q, o], want, [g[0], g[1], g[3]])
    return img, [back(x) for x in list(got[:4]) + [g[2]] + list(got[4:])]

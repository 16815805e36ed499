"""The host path in C++ (csrc/host.cpp) against the Python path that takes every
call it leaves: same results, gradients and refusals, and it does leave what is
not the plain case."""
import threading

import pytest
import torch
from torch.utils.checkpoint import checkpoint

from torch_gsplat_bridge_fast import (RasterConfig, project_pinhole_gaussians, rasterize_pinhole_gaussians,
                                      rasterize_projected_gaussians)
from torch_gsplat_bridge_fast import _lib, _ops
from torch_gsplat_bridge_fast import project as project_mod
from torch_gsplat_bridge_fast import rasterize as rasterize_mod
from torch_gsplat_bridge_fast.scenes import make_scene_2d, make_scene_3d

pytestmark = pytest.mark.gpu

KEYS = ("means2d", "conics", "colors", "opacities", "depths")
# the direct path, the one-call binning, the tile-sorted binning
SIZES = [(1, 300, 96, 131), (2, 5000, 130, 170), (2, 9000, 260, 530)]


def _scene(B, G, H, W, batched=True, seed=1):
    sc = make_scene_2d(0, seed=seed, G=G, B=B, H=H, W=W)
    ts = [sc[k].cuda() for k in KEYS]
    return ts if batched else [t[0].contiguous() for t in ts]


def _plan(cfg, ts):
    """The config's plan (a first call makes it, and the shape's capacity)."""
    with torch.no_grad():
        rasterize_projected_gaussians(*ts, cfg)
        rasterize_projected_gaussians(*ts, cfg)
    plan = rasterize_mod._plan(cfg)
    assert plan is not None
    return plan


def _python(ts, cfg):
    if ts[0].ndim == 2:
        return rasterize_mod._rasterize_batched(*(t.unsqueeze(0) for t in ts), cfg).squeeze(0)
    return rasterize_mod._rasterize_batched(*ts, cfg)


def _leaves(ts, need):
    return [t.clone().requires_grad_(bool(n)) for t, n in zip(ts, need)]


@pytest.mark.parametrize("B,G,H,W", SIZES)
@pytest.mark.parametrize("need", [(1, 1, 1, 1, 1), (1, 1, 1, 1, 0), (0, 1, 0, 0, 0), (0, 0, 0, 1, 1)])
def test_matches_python(B, G, H, W, need):
    batched = B > 1
    ts = _scene(B, G, H, W, batched)
    cfg = RasterConfig(height=H, width=W, background=(0.1, 0.2, 0.3))
    plan = _plan(cfg, ts)
    w = torch.rand((B, H, W, 3) if batched else (H, W, 3), generator=torch.Generator().manual_seed(2)).cuda()
    a, b = _leaves(ts, need), _leaves(ts, need)
    img = plan.run(*a, True)
    ref = _python(b, cfg)
    assert img is not None and img.shape == ref.shape and torch.equal(img, ref) and img.requires_grad
    img.backward(w, retain_graph=True)
    img.backward(w)
    ref.backward(w, retain_graph=True)
    ref.backward(w)
    for x, y in zip(a, b):
        assert (x.grad is None) == (y.grad is None)
        if x.grad is not None:
            assert x.grad.shape == x.shape
            torch.testing.assert_close(x.grad, y.grad, rtol=1e-4, atol=1e-5 * float(y.grad.abs().max()) + 1e-7)
    with pytest.raises(RuntimeError, match="second time"):
        img.backward(w)
    with torch.no_grad():
        out = plan.run(*a, True)
    assert torch.equal(out, ref) and not out.requires_grad


@pytest.mark.parametrize("B,G,H,W", SIZES)
def test_strides_hooks_and_streams(B, G, H, W):
    """Strided inputs, saved-tensor hooks (the buffers go to host memory and back), another stream and
    an upstream graph give the plain call's gradients."""
    ts = _scene(B, G, H, W)
    cfg = RasterConfig(height=H, width=W)
    _plan(cfg, ts)
    w = torch.rand(B, H, W, 3, generator=torch.Generator().manual_seed(2)).cuda()

    def step(leaves, args, grad=w):
        img = rasterize_projected_gaussians(*args, cfg)
        img.backward(grad)
        return img.detach(), [x.grad for x in leaves[:4]]

    leaves = _leaves(ts, (1, 1, 1, 1, 0))
    want = step(leaves, leaves)

    def close(got):
        assert torch.equal(got[0], want[0])
        for x, y in zip(got[1], want[1]):
            torch.testing.assert_close(x, y, rtol=1e-4, atol=1e-5 * float(y.abs().max()))

    wide = [torch.stack([t, t], dim=-1)[..., 0].detach().requires_grad_(k < 4) for k, t in enumerate(ts)]
    assert not any(t.is_contiguous() for t in wide)
    close(step(wide, wide))
    x = _leaves(ts, (1, 1, 1, 1, 0))
    close(step(x, [t * 1.0 for t in x[:4]] + [x[4]], w.transpose(1, 2).contiguous().transpose(1, 2)))
    x = _leaves(ts, (1, 1, 1, 1, 0))
    packed = []
    with torch.autograd.graph.saved_tensors_hooks(lambda t: packed.append(t.shape) or t.cpu(), lambda t: t.cuda()):
        close(step(x, x))
    assert packed
    x = _leaves(ts, (1, 1, 1, 1, 0))
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        got = step(x, x)
    torch.cuda.current_stream().wait_stream(side)
    close(got)


@pytest.mark.parametrize("kind,B,G,H,W", [
    ("uniform", 1, 16384, 512, 272),     # the fewest splats, 2^9 + 32 tiles
    ("ties", 1, 4999, 512, 1024),        # the fewest tiles
    ("uniform", 1, 131072, 1080, 1920),
    ("uniform", 2, 131072, 800, 1100),   # the most
    ("uniform", 1, 131072, 4096, 4095),  # buckets above 8192 pairs
    ("ties", 3, 21845, 300, 400),        # depth ties, three images
    ("special", 2, 20001, 333, 517),     # NaN, infinite and signed zero depths
    ("uniform", 1, 70001, 4096, 4096),   # 2^16 tiles, 256 a bucket
    ("long", 1, 30000, 400, 400),        # lists above the hand-off length, below the limit
    ("hot tile", 1, 20000, 600, 600),    # a tile above the limit: binned by the other path
    ("hot bucket", 1, 60000, 600, 600),  # a bucket above the limit
    ("culled", 1, 20002, 600, 600),
])
def test_tile_sorted_matches_python(kind, B, G, H, W):
    g = torch.Generator().manual_seed(5)
    sc = make_scene_2d(1, seed=3, G=G, B=B, H=H, W=W)
    if kind == "ties":
        sc["depths"] = torch.randint(0, 9, (B, G), generator=g).float()
    if kind == "special":
        for k, v in enumerate((float("nan"), float("inf"), -float("inf"), -0.0, 0.0)):
            sc["depths"][:, k::7] = v
    if kind == "long":
        sc["conics"] = sc["conics"] * 0.3
        sc["opacities"] = 0.05 + 0.0 * sc["opacities"]
    if kind == "hot tile":
        sc["means2d"][:, :900] = 300.0 + 2.0 * torch.rand(B, 900, 2, generator=g)
        sc["opacities"] = 0.3 * sc["opacities"]
    if kind == "hot bucket":
        sc["means2d"][:, :40000] = torch.rand(B, 40000, 2, generator=g) * torch.tensor([600.0, 20.0])
        sc["opacities"] = 0.3 * sc["opacities"]
    if kind == "culled":
        sc["opacities"] = 0.0 * sc["opacities"]
    ts = [sc[k].cuda() for k in KEYS]
    cfg = RasterConfig(height=H, width=W, background=(0.1, 0.2, 0.3))
    _plan(cfg, ts)
    rasterize_mod._plans.clear()           # (a plan that has seen no skewed scene)
    plan = rasterize_mod._make_plan(cfg)
    L = _lib.lib()
    meta = rasterize_mod._meta(cfg, B, G)
    key = (0, B, G, H, W)
    cap = _ops._capacity.get(key, 0)
    if kind == "culled":
        cap = _ops._capacity[key] = 10000
    assert L.gsplat_hip_tile_workspace_bytes(meta, cap) > 0
    w = torch.rand(B, H, W, 3, generator=g).cuda()
    b = _leaves(ts, (1, 1, 1, 1, 0))
    ref = _python(b, cfg)
    ref.backward(w)
    n = _ops.bin_gaussians(meta, *[t.reshape(B * G, -1).squeeze(-1) for t in ts]).n_pairs
    hot = kind.startswith("hot")
    for k, cap in enumerate((cap, cap, max(1, n), max(1, n // 2))):   # the last: too small, binned again
        _ops._capacity[key] = cap
        a = _leaves(ts, (1, 1, 1, 1, 0))
        with _ops.LaunchTrace() as trace:
            img = plan.run(*a, True)
        names = [name for name, _ in trace.launches]
        # (a skewed scene is tried once, then binned at once)
        assert ("tile_sort_kernel" in names) == (not hot or k == 0)
        assert ("emit_kernel<true>" in names) == (hot or cap < n)
        assert torch.equal(img, ref)
        img.backward(w)
        for x, y in zip(a[:4], b[:4]):
            torch.testing.assert_close(x.grad, y.grad, rtol=1e-4, atol=1e-5 * float(y.grad.abs().max()) + 1e-7)
        with torch.no_grad():
            assert torch.equal(plan.run(*ts, True), ref)


def test_skewed_shape_is_tried_again():
    """A scene with a tile list too long for the tile sort sends its shape's next 1024 calls to the one-call
    binning, then the tile sort is tried again, and 2048 calls after a second such scene."""
    B, G, H, W = 1, 20007, 600, 600
    even, hot = _scene(B, G, H, W), _scene(B, G, H, W)
    hot[0][:, :900] = 300.0 + 2.0 * torch.rand(B, 900, 2, generator=torch.Generator().manual_seed(5)).cuda()
    hot[3] = 0.3 * hot[3]
    cfg = RasterConfig(height=H, width=W, background=(0.1, 0.3, 0.3))
    plan = _plan(cfg, even)
    want = _python(even, cfg), _python(hot, cfg)

    def launches(ts, ref):
        with _ops.LaunchTrace() as trace, torch.no_grad():
            img = plan.run(*ts, True)
        assert torch.equal(img, ref)
        return [name for name, _ in trace.launches]

    for calls in (1024, 2048):
        assert "tile_sort_kernel" in launches(even, want[0])
        names = launches(hot, want[1])
        assert "tile_sort_kernel" in names and "emit_kernel<true>" in names
        assert "tile_sort_kernel" not in launches(even, want[0])
        with torch.no_grad():
            for _ in range(calls - 2):
                plan.run(*even, True)
        assert "tile_sort_kernel" not in launches(even, want[0])
    assert "tile_sort_kernel" in launches(even, want[0])


@pytest.mark.parametrize("B,G,H,W", SIZES)
def test_new_configs_checkpointed(B, G, H, W):
    """A background per step on a shape whose capacity is known: each config's first call is checkpointed,
    and its recomputation saves what it saved."""
    ts = _scene(B, G, H, W)
    with torch.no_grad():
        rasterize_projected_gaussians(*ts, RasterConfig(height=H, width=W))
    w = torch.rand(B, H, W, 3, generator=torch.Generator().manual_seed(2)).cuda()
    for step in range(3):
        cfg = RasterConfig(height=H, width=W, background=(0.5, 0.25, 0.125 * step))
        a, b = _leaves(ts, (1, 1, 1, 1, 0)), _leaves(ts, (1, 1, 1, 1, 0))
        img = checkpoint(rasterize_projected_gaussians, *a, cfg, use_reentrant=False)
        img.backward(w)
        ref = _python(b, cfg)
        ref.backward(w)
        assert torch.equal(img, ref)
        for x, y in zip(a[:4], b[:4]):
            torch.testing.assert_close(x.grad, y.grad, rtol=1e-4, atol=1e-5 * float(y.grad.abs().max()) + 1e-7)
    sc = make_scene_3d(seed=4, G=G, H=H, W=W)
    ts = [torch.cat([sc[k].cuda()] * B) for k in ("means3d", "scales", "quats", "opacities", "colors")]
    cam = (250.0, 250.0, W / 2, H / 2)
    with torch.no_grad():
        rasterize_pinhole_gaussians(*ts, *cam, config=RasterConfig(height=H, width=W))
    for step in range(2):
        cfg = RasterConfig(height=H, width=W, background=(0.75, 0.25, 0.125 * step))
        x = _leaves(ts, (1, 1, 1, 1, 1))
        checkpoint(lambda *t: rasterize_pinhole_gaussians(*t, *cam, config=cfg), *x, use_reentrant=False).backward(w)
        assert all(bool(t.grad.abs().sum() > 0) for t in x)


def test_threads_share_a_plan():
    """Threads with streams of their own, one config, different scenes."""
    B, G, H, W = SIZES[1]
    cfg = RasterConfig(height=H, width=W)
    scenes = [_scene(B, G, H, W, seed=s) for s in range(4)]
    _plan(cfg, scenes[0])
    want = [_python(s, cfg) for s in scenes]
    torch.cuda.synchronize()
    bad = []

    def work(k):
        stream = torch.cuda.Stream()
        with torch.cuda.stream(stream), torch.no_grad():
            for _ in range(20):
                img = rasterize_projected_gaussians(*scenes[k], cfg)
                stream.synchronize()
                if not torch.equal(img, want[k]):
                    bad.append(k)

    threads = [threading.Thread(target=work, args=(k,)) for k in range(4)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not bad


def test_refusals_stay():
    """With the config's plan known, inputs that were refused are refused with the same errors."""
    B, G, H, W = SIZES[0]
    ts = _scene(B, G, H, W)
    cfg = RasterConfig(height=H, width=W)
    _plan(cfg, ts)

    def bad(k, t, match, err=ValueError):
        args = list(ts)
        args[k] = t
        with pytest.raises(err, match=match):
            rasterize_projected_gaussians(*args, cfg)

    bad(0, ts[0].double(), "must be float32")
    bad(1, ts[1].cpu(), "same device")
    bad(1, ts[1][:, :-1], "dimensions must match")
    bad(2, ts[2][..., :2], "last dim = 3")
    bad(3, ts[3][0], "rank")
    with pytest.raises(ValueError, match="ROCm device"):
        rasterize_projected_gaussians(*(t.cpu() for t in ts), cfg)
    with pytest.raises(ValueError, match="at least one Gaussian"):
        rasterize_projected_gaussians(*(t[:, :0] for t in ts), cfg)
    with pytest.raises(RuntimeError):   # no vmap rule
        torch.vmap(lambda m: rasterize_projected_gaussians(m, *ts[1:], cfg))(torch.stack([ts[0]] * 2))
    with pytest.raises(Exception):      # no jvp
        torch.func.jvp(lambda m: rasterize_projected_gaussians(m, *ts[1:], cfg), (ts[0],), (ts[0],))
    # vmap used in this thread before does not keep later calls off the host path
    assert rasterize_mod._plan(cfg).run(*ts, True) is not None


@pytest.mark.parametrize("batched", [False, True])
def test_projection_matches_python(batched):
    G = 3000
    sc = make_scene_3d(seed=4, G=G, H=200, W=300)
    ts = [sc[k].cuda() for k in ("means3d", "scales", "quats", "opacities", "colors")]
    ts = [torch.cat([t, t.flip(1)]) if batched else t[0].contiguous() for t in ts]
    ts[3] = ts[3].unsqueeze(-1)   # [.., 1] opacities
    c2w = sc["camera_to_world"].cuda()
    cfg = RasterConfig(height=200, width=300)
    cam = (250.0, 250.0, 150.0, 100.0)

    def run(native):
        if not native:
            project_mod._project_plain, keep = (lambda *a: None), project_mod._project_plain
        try:
            x = [t.clone().requires_grad_(True) for t in ts]
            pose = c2w.clone().requires_grad_(True)
            out = project_pinhole_gaussians(*x[:4], *cam, camera_to_world=pose)
            (out[0].sum() * 1e-3 + out[1].square().sum() + out[2].sum() + 0.1 * out[3].sum()).backward()
            g1 = [t.grad.clone() for t in x[:4]] + [pose.grad.clone()]
            for t in (*x, pose):
                t.grad = None
            imgs = []
            for _ in range(3):
                img = rasterize_pinhole_gaussians(*x, *cam, camera_to_world=pose, config=cfg)
                imgs.append(img.detach())
            img.square().mean().backward()
            return out, g1, imgs[-1], [t.grad for t in x] + [pose.grad]
        finally:
            if not native:
                project_mod._project_plain = keep

    a, b = run(True), run(False)
    for x, y in zip(a[0], b[0]):
        assert x.shape == y.shape and torch.equal(x, y)
    assert torch.equal(a[2], b[2])
    for x, y in zip(a[1] + a[3], b[1] + b[3]):
        assert x.shape == y.shape
        torch.testing.assert_close(x, y, rtol=1e-4, atol=1e-5 * float(y.abs().max()))
    with pytest.raises(ValueError, match="quats must have shape"):
        project_pinhole_gaussians(ts[0], ts[1], ts[2][..., :3], ts[3], *cam)
    with pytest.raises(ValueError, match="must be float32"):
        project_pinhole_gaussians(ts[0].double(), *ts[1:4], *cam)

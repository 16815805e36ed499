"""The sliced forward and backward of dense scenes against the unsliced path:
the image bit for bit (both walk the same splats of every tile in the same
order), the gradients up to the order of their atomic sums."""
import pytest
import torch
import torch.utils.checkpoint

from torch_gsplat_bridge_fast import RasterConfig, _lib, _ops, _slices, rasterize_projected_gaussians

pytestmark = pytest.mark.gpu


def _scene(B, G, H, W, seed, sigma=(4.0, 20.0), logit=0.0, depth="uniform", cover=1.0):
    """Splats over the left `cover` of the image; depth ties with depth="planes"."""
    g = torch.Generator().manual_seed(seed)
    means = torch.rand(B, G, 2, generator=g) * torch.tensor([W * cover, float(H)])
    sig = sigma[0] + torch.rand(B, G, 2, generator=g) * (sigma[1] - sigma[0])
    th = torch.rand(B, G, generator=g) * 3.14159
    c, s = torch.cos(th), torch.sin(th)
    ix, iy = sig[..., 0] ** -2, sig[..., 1] ** -2
    conics = torch.stack([c * c * ix + s * s * iy, c * s * (ix - iy), s * s * ix + c * c * iy], -1)
    depths = torch.rand(B, G, generator=g) * 10 if depth == "uniform" else \
        torch.randint(0, 40, (B, G), generator=g).float()
    if depth == "one":
        depths = torch.ones(B, G)
    opac = torch.sigmoid(logit + torch.randn(B, G, generator=g))
    if depth == "veil":  # the left 45% nearly transparent: most of its splats touch live tiles
        opac = torch.where(means[..., 0] < 0.45 * W, 0.02 * opac, opac)
        depths = torch.rand(B, G, generator=g) * 10
    if depth == "split":  # near: the left half opaque, the right 40% translucent; behind, inside the left half: the rest
        part = torch.rand(B, G, generator=g)
        x, y = means.unbind(-1)
        far = part >= 0.7
        x = torch.where(far, 0.15 * W + 0.15 * x, torch.where(part < 0.6, 0.5 * x, W - 0.4 * x))
        means = torch.stack([x, torch.where(far, 0.25 * H + 0.45 * y, y)], -1)
        opac = torch.where((part >= 0.6) & ~far, 0.02 + 0.0 * opac, opac)
        depths = torch.rand(B, G, generator=g) + 5.0 * far
    t = [means, conics, torch.rand(B, G, 3, generator=g), opac, depths]
    return [x.cuda().contiguous() for x in t]


def _flat(ts):
    return [t.reshape(-1, t.shape[-1]) if t.ndim == 3 else t.reshape(-1) for t in ts]


def _unsliced(meta, ts, w):
    st = _ops.bin_gaussians(meta, *_flat(ts))
    img, T, last, stop, ws = _ops.render_forward(meta, st, save_state=True)
    grads = _ops.render_backward(meta, st, T, last, stop, w, ws)
    return st, img, T, stop, grads


def _sliced(monkeypatch, meta, ts, w, budget, cap, save_state=True):
    key = (0, meta.batch, meta.gaussians_per_batch, meta.height, meta.width)
    monkeypatch.setattr(_slices, "MIN_PAIRS", 0)
    monkeypatch.setattr(_slices, "MIN_PAIRS_PER_TILE", 0)
    monkeypatch.setitem(_ops._capacity, key, cap)
    plan = _slices._Plan(cap)
    plan.budget = budget
    monkeypatch.setitem(_slices._plans, key, plan)
    got = _slices.render(meta, _flat(ts), save_state=save_state)
    if got is None or not save_state:
        return got, None
    st, (img, T, last) = got
    out = _ops.gradient_buffers(meta.batch, meta.gaussians_per_batch, img.device)
    grads = _slices.backward(meta, st.tensors(), st.plain(), T, last, w, out)
    st.check_status()
    return got, grads


CASES = [
    # B, G, H, W, sigma, logit, depth, cover, budget
    (1, 20000, 200, 300, (4.0, 20.0), 0.0, "uniform", 1.0, 256),    # opaque but for some edges
    (1, 20000, 200, 300, (4.0, 20.0), 0.0, "planes", 0.6, 400),     # depth ties, an empty side
    (2, 9001, 203, 341, (4.0, 20.0), 0.0, "uniform", 0.9, 220),     # ragged, two images
    (3, 5000, 64, 80, (2.0, 9.0), 0.0, "planes", 1.0, 300),         # tiles of three images in one bitmap word
    (1, 30000, 160, 160, (4.0, 30.0), -1.0, "uniform", 0.8, 900),   # lists over 128: continuation, segments
    (1, 350000, 512, 512, (1.0, 6.0), 0.5, "veil", 1.0, 400),       # a back of over 131,072 splats
    (1, 20000, 200, 300, (4.0, 20.0), 0.0, "uniform", 1.0, 100000),  # the front holds every splat, no live tile
    (1, 20000, 200, 300, (4.0, 20.0), 0.0, "uniform", 0.6, 100000),  # the same with live tiles: no back either
    (1, 20000, 200, 300, (2.0, 5.0), 0.0, "split", 1.0, 390),        # what the front leaves out touches no live tile
]


@pytest.mark.parametrize("B,G,H,W,sigma,logit,depth,cover,budget", CASES)
def test_sliced_matches_unsliced(monkeypatch, B, G, H, W, sigma, logit, depth, cover, budget):
    ts = _scene(B, G, H, W, 3, sigma, logit, depth, cover)
    meta = _lib.make_raster_meta(H, W, B, G, 1 / 255, 1e-4, (0.1, 0.2, 0.3))
    w = torch.rand(B, H, W, 3, generator=torch.Generator().manual_seed(1)).cuda()
    st, img, T, stop, ref = _unsliced(meta, ts, w)
    # (the front's slots grow with budget / capacity: at this ratio they hold every splat)
    whole = budget >= 100000 or depth == "split"
    cap = max(st.n_pairs, (4 * budget * st.num_tiles // 3 + 1) if whole else 2 * budget * st.num_tiles)
    got, grads = _sliced(monkeypatch, meta, ts, w, budget, cap)
    key = (0, B, G, H, W)
    assert got is not None, f"the scene was meant to be sliced (budget now {_slices._plans[key].budget})"
    state, (img2, T2, last2) = got
    assert torch.equal(img, img2) and torch.equal(T, T2)
    if whole:
        assert not state.has_back
        assert bool((T > 1e-4).any()) == (cover < 1 or depth == "split")
        layout = state.plain()[1][0][0]
        front_offsets = state.tensors()[2][layout[2]:layout[2] + 4 * (st.num_tiles + 1)].view(torch.int32)
        assert (int(front_offsets[-1]) < st.n_pairs) == (depth == "split")
    if depth == "veil":
        assert state.plain()[1][1][1] > 131072  # the back's slots
    for a, b in zip(grads, ref):
        torch.testing.assert_close(a, b, rtol=1e-4, atol=1e-5 * float(b.abs().max()))
    # a second backward on the same state: the gradient records are zero again
    again = _slices.backward(meta, state.tensors(), state.plain(), T2, last2, w,
                             _ops.gradient_buffers(B, G, img.device))
    for a, b in zip(again, ref):
        torch.testing.assert_close(a, b, rtol=1e-4, atol=1e-5 * float(b.abs().max()))
    # the eval forward
    got, _ = _sliced(monkeypatch, meta, ts, w, budget, cap, save_state=False)
    assert torch.equal(got[1][0], img)


def test_fronts_that_do_not_suit_return_none(monkeypatch):
    """One depth for all (no front can be chosen) and a translucent scene: the caller is sent to the
    unsliced path and the shape's budget is raised or given up."""
    for kw in (dict(depth="one"), dict(logit=-4.0)):
        ts = _scene(1, 20000, 200, 300, 5, **kw)
        meta = _lib.make_raster_meta(200, 300, 1, 20000, 1 / 255, 1e-4, (0, 0, 0))
        st = _ops.bin_gaussians(meta, *_flat(ts))
        got, _ = _sliced(monkeypatch, meta, ts, None, 32, max(st.n_pairs, 64 * st.num_tiles), save_state=False)
        assert got is None
        assert _slices._plans[(0, 1, 20000, 200, 300)].budget in (0, 64)


def test_negative_threshold_is_not_sliced(monkeypatch):
    """The slots a slice leaves over hold splats of opacity 0, visible below a threshold of 0: such a config
    goes unsliced, also where the shape has been sliced with another threshold."""
    ts = _scene(1, 20000, 200, 300, 3)
    meta = _lib.make_raster_meta(200, 300, 1, 20000, 1 / 255, 1e-4, (0, 0, 0))
    n = _ops.bin_gaussians(meta, *_flat(ts)).n_pairs
    cap = max(n, 2 * 256 * 247)
    assert _sliced(monkeypatch, meta, ts, None, 256, cap, save_state=False)[0] is not None
    meta = _lib.make_raster_meta(200, 300, 1, 20000, -0.1, 1e-4, (0, 0, 0))
    assert _slices.render(meta, _flat(ts), save_state=False) is None


def test_public_calls_take_the_slices(monkeypatch):
    """rasterize_projected_gaussians on a dense scene: the second and later calls of the shape are
    sliced and give the first call's image, through autograd too."""
    monkeypatch.setattr(_slices, "MIN_PAIRS", 1 << 18)
    monkeypatch.setattr(_slices, "FIRST_BUDGET", 96)
    seen = []
    orig = _slices.render
    monkeypatch.setattr(_slices, "render", lambda *a, **k: seen.append(orig(*a, **k)) or seen[-1])
    B, G, H, W = 1, 40001, 190, 310
    ts = _scene(B, G, H, W, 11)
    cfg = RasterConfig(height=H, width=W, background=(0.1, 0.2, 0.3))
    imgs, grads = [], []
    for k in range(4):
        leaves = [t[0].clone().requires_grad_(True) for t in ts]
        img = rasterize_projected_gaussians(*leaves, cfg)
        img.square().mean().backward()
        imgs.append(img.detach())
        grads.append([t.grad for t in leaves])
    with torch.no_grad():
        imgs.append(rasterize_projected_gaussians(*[t[0] for t in ts], cfg))
    assert any(s is not None for s in seen)
    for img in imgs[1:]:
        assert torch.equal(img, imgs[0])
    for g in grads[1:]:
        for a, b in zip(g, grads[0]):
            torch.testing.assert_close(a, b, rtol=1e-4, atol=1e-5 * float(b.abs().max()))


def test_checkpointed_calls(monkeypatch):
    """Non-reentrant checkpointing of a shape that is sliced otherwise: the recomputation saves what the
    first pass saved, call after call."""
    monkeypatch.setattr(_slices, "MIN_PAIRS", 1 << 18)
    monkeypatch.setattr(_slices, "FIRST_BUDGET", 96)   # too small: the first sliced call raises it
    seen = []
    orig = _slices.render
    monkeypatch.setattr(_slices, "render", lambda *a, **k: seen.append(orig(*a, **k)) or seen[-1])
    B, G, H, W = 1, 40005, 190, 310
    cfg = RasterConfig(height=H, width=W, background=(0.1, 0.2, 0.3))
    ts = _scene(B, G, H, W, 11)
    w = torch.rand(B, H, W, 3, generator=torch.Generator().manual_seed(1)).cuda()

    def step(checkpointed):
        leaves = [t.clone().requires_grad_(k < 4) for k, t in enumerate(ts)]
        img = torch.utils.checkpoint.checkpoint(rasterize_projected_gaussians, *leaves, cfg, use_reentrant=False) \
            if checkpointed else rasterize_projected_gaussians(*leaves, cfg)
        img.backward(w)
        return [img.detach()] + [t.grad for t in leaves[:4]]

    want = step(False)
    for checkpointed in (True, False, True, False, True):
        got = step(checkpointed)
        assert torch.equal(got[0], want[0])
        for a, b in zip(got[1:], want[1:]):
            torch.testing.assert_close(a, b, rtol=1e-4, atol=1e-5 * float(b.abs().max()))
    assert any(x is not None for x in seen)


def test_views_of_different_density(monkeypatch):
    """A dense view and one with few visible splats by turns on one shape, whose remembered capacity is
    the dense one's when the sparse one comes: each call gives the unsliced image and gradients, and the
    dense view is sliced whenever the capacity is its own."""
    monkeypatch.setattr(_slices, "MIN_PAIRS", 1 << 18)
    seen = {}
    orig = _slices.render

    def render(*a, **k):
        seen[call] = orig(*a, **k)
        return seen[call]

    monkeypatch.setattr(_slices, "render", render)
    B, G, H, W = 1, 40003, 190, 310
    cfg = RasterConfig(height=H, width=W, background=(0.1, 0.2, 0.3))
    meta = _lib.make_raster_meta(H, W, B, G, 1 / 255, 1e-4, (0.1, 0.2, 0.3))
    monkeypatch.delitem(_ops._capacity, (0, B, G, H, W), raising=False)
    monkeypatch.delitem(_slices._plans, (0, B, G, H, W), raising=False)
    dense = _scene(B, G, H, W, 11)
    sparse = _scene(B, G, H, W, 12, sigma=(1.0, 3.0))
    sparse[3] = torch.where(torch.arange(G, device="cuda") < 3000, sparse[3], 0.0 * sparse[3]).contiguous()
    w = torch.rand(B, H, W, 3, generator=torch.Generator().manual_seed(1)).cuda()
    want = {}
    for name, ts in (("dense", dense), ("sparse", sparse)):
        monkeypatch.delitem(_ops._capacity, (0, B, G, H, W), raising=False)
        _, img, _, _, ref = _unsliced(meta, ts, w)
        want[name] = img, ref
    monkeypatch.delitem(_ops._capacity, (0, B, G, H, W), raising=False)
    names = ("dense", "dense", "sparse", "dense", "sparse", "dense", "dense", "sparse")
    for call, name in enumerate(names):
        leaves = [t.clone().requires_grad_(k < 4) for k, t in enumerate(dense if name == "dense" else sparse)]
        img = rasterize_projected_gaussians(*leaves, cfg)
        img.backward(w)
        assert torch.equal(img, want[name][0])
        for a, b in zip(leaves[:4], want[name][1]):
            torch.testing.assert_close(a.grad, b, rtol=1e-4, atol=1e-5 * float(b.abs().max()))
    for call in (1, 2, 4, 6, 7):   # (3 and 5 find the capacity that the sparse view left)
        assert seen[call] is not None, (call, names[call])


@pytest.mark.parametrize("B,G,H,W,sigma", [
    (1, 2999, 300, 500, (6.0, 20.0)),     # 8 splats per wavefront: dozens of pairs per splat
    (2, 70001, 400, 500, (8.0, 16.0)),    # 16: as dense, over 131,072 splats in the batch
    (3, 90001, 400, 500, (8.0, 16.0)),    # 32: as dense, over 262,144 splats in the batch
    (1, 16384, 300, 500, (0.5, 2.0)),     # 16: few splats
    (1, 16385, 300, 500, (0.5, 2.0)),     # 32
])
def test_walk_widths(monkeypatch, B, G, H, W, sigma):
    """The one-call binning at each number of splats per wavefront against the staged calls (always
    32): the same offsets, tile ranges and lists."""
    ts = _scene(B, G, H, W, 7, sigma)
    meta = _lib.make_raster_meta(H, W, B, G, 1 / 255, 1e-4, (0, 0, 0))
    key = (0, B, G, H, W)
    monkeypatch.delitem(_ops._capacity, key, raising=False)
    ref = _ops.bin_gaussians(meta, *_flat(ts))   # staged: the shape's first binning
    n = ref.n_pairs
    if sigma[0] > 1:
        assert n >= 24 * B * G
    for cap in (n, n + 1, n + n // 4):
        with _ops.LaunchTrace() as trace:
            got = _ops._bin_fast(meta, *_flat(ts), cap, key)
        assert "emit_kernel<true>" in [name for name, _ in trace.launches]
        assert got.n_pairs == n
        got.check_status()
        assert torch.equal(got.perm, ref.perm)
        assert torch.equal(got.splat_offsets, ref.splat_offsets)
        assert torch.equal(got.tile_offsets, ref.tile_offsets)
        assert torch.equal(got.binned_ids, ref.binned_ids)
        assert torch.equal(got.packed, ref.packed)

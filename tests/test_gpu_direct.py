"""The direct path of small scenes against the staged binning and forward: the
same records, tile lists, image and stops bit for bit, the gradients up to the
order of their atomic sums."""
import pytest
import torch

from torch_gsplat_bridge_fast import _lib, _ops
from torch_gsplat_bridge_fast.scenes import make_scene_2d

pytestmark = pytest.mark.gpu

KEYS = ("means2d", "conics", "colors", "opacities", "depths")


def _flat(sc, B, G):
    return [sc[k].reshape(B * G, -1).squeeze(-1).contiguous().cuda() for k in KEYS]


@pytest.mark.parametrize("B,G,H,W,kind", [
    (1, 1, 16, 16, "uniform"),
    (1, 15, 33, 47, "ties"),          # below one group of ranks
    (2, 64, 40, 50, "uniform"),
    (3, 65, 64, 17, "special"),       # NaN, infinite and signed zero depths
    (1, 129, 100, 100, "uniform"),    # one above the hand-off length
    (5, 401, 203, 341, "ties"),
    (1, 300, 96, 131, "big"),         # splats larger than the image, off-screen centres
    (1, 4095, 150, 200, "ties"),
    (2, 4096, 150, 200, "uniform"),   # the most splats
    (1, 768, 2048, 2048, "uniform"),  # the most tiles x splats
    (1, 900, 48, 48, "faint"),        # lists of hundreds: continuation and segments
    (1, 4000, 850, 870, "faint"),     # the same in 2970 tiles: more segments than records
    (1, 50, 32, 32, "culled"),        # nothing visible
])
def test_direct_matches_staged(B, G, H, W, kind):
    sc = make_scene_2d(0, seed=G, G=G, B=B, H=H, W=W)
    if kind in ("ties", "special"):
        sc["depths"] = torch.randint(0, 5, (B, G), generator=torch.Generator().manual_seed(1)).float()
    if kind == "special":
        sc["depths"][:, ::7] = float("nan")
        sc["depths"][:, 1::7] = float("inf")
        sc["depths"][:, 2::7] = -float("inf")
        sc["depths"][:, 3::7] = -0.0
    if kind == "big":
        sc["means2d"] = sc["means2d"] * 3.0 - 100.0
        sc["conics"] = sc["conics"] * 1e-3
    if kind == "faint":
        sc["opacities"] = 0.02 + 0.0 * sc["opacities"]
        sc["conics"] = sc["conics"] * 0.05
    if kind == "culled":
        sc["opacities"] = 0.001 + 0.0 * sc["opacities"]
    flat = _flat(sc, B, G)
    meta = _lib.make_raster_meta(H, W, B, G, 1 / 255, 1e-4, (0.1, 0.2, 0.3))
    key = (0, B, G, H, W)
    _ops._capacity.pop(key, None)
    ref = _ops.bin_gaussians(meta, *flat)
    img, T, last, stop, ws = _ops.render_forward(meta, ref, save_state=True)
    st, (img2, T2, last2, stop2, ws2) = _ops.direct_render(meta, flat, save_state=True)
    assert torch.equal(st.packed.view(torch.int32), ref.packed.view(torch.int32))
    tiles = ref.num_tiles
    counts = ref.tile_counts.tolist()
    offs = ref.tile_offsets.tolist()
    assert st.tile_offsets[:tiles].tolist() == [t * G for t in range(tiles)]
    for t in {0, tiles // 2, tiles - 1} | set(range(0, tiles, max(1, tiles // 97))):
        assert torch.equal(st.pairs[t * G:t * G + counts[t]], ref.pairs[offs[t]:offs[t + 1]]), f"tile {t}"
    assert torch.equal(img2, img) and torch.equal(T2, T) and torch.equal(stop2, stop)
    w = torch.rand(B, H, W, 3, generator=torch.Generator().manual_seed(2)).cuda()
    want = _ops.render_backward(meta, ref, T, last, stop, w, ws)
    for _ in range(2):  # the gradient records are zero again after a backward
        got = _ops.render_backward(meta, st, T2, last2, stop2, w, ws2)
        for a, b in zip(got, want):
            torch.testing.assert_close(a, b, rtol=1e-4, atol=1e-5 * max(1.0, float(b.abs().max())), equal_nan=True)
    _, (img3, *_) = _ops.direct_render(meta, flat, save_state=False)
    assert torch.equal(img3, img)


def test_direct_limits():
    """Above 4096 splats an image or 12 * 2^20 tiles x splats the caller gets None."""
    for G, H, W in ((4097, 32, 32), (769, 2048, 2048)):
        sc = make_scene_2d(0, seed=1, G=G, H=H, W=W)
        meta = _lib.make_raster_meta(H, W, 1, G, 1 / 255, 1e-4, (0, 0, 0))
        assert _ops.direct_render(meta, _flat(sc, 1, G), save_state=False) is None


@pytest.mark.parametrize("G,H,W", [
    (3000, 16, 16),        # one tile
    (20000, 511, 1009),    # 2048 tiles, the most that are composited by several wavefronts each
    (20000, 513, 990),     # 2046 tiles of 33 rows, the last cut
    (20000, 512, 1025),    # 2080 tiles: one wavefront each
])
def test_wavefronts_per_tile(G, H, W):
    """Image, stops and gradients with the workspace (several wavefronts per tile in images of few
    tiles, continuation in others) against those without it (one wavefront per tile throughout)."""
    L = _lib.lib()
    sc = make_scene_2d(0, seed=3, G=G, B=1, H=H, W=W)
    sc["opacities"] = 0.3 * sc["opacities"]
    flat = _flat(sc, 1, G)
    meta = _lib.make_raster_meta(H, W, 1, G, 1 / 255, 1e-4, (0.1, 0.2, 0.3))
    _ops._capacity.pop((0, 1, G, H, W), None)
    st = _ops.bin_gaussians(meta, *flat)
    out = _ops.render_forward(meta, st, save_state=True)
    one = [torch.empty_like(t) for t in out[:4]]
    p = _lib.ptr
    _lib.check(L.gsplat_hip_render_forward(meta, p(st.packed), p(st.tile_offsets), p(st.pairs), *map(p, one),
                                           st.capacity, None, 0, _lib.stream_of(one[0])), "render_forward")
    for a, b in zip(out[:4], one):
        assert torch.equal(a, b)
    w = torch.rand(1, H, W, 3, generator=torch.Generator().manual_seed(2)).cuda()
    got = _ops.render_backward(meta, st, *out[1:4], w, out[4])
    want = _ops.render_backward(meta, st, *one[1:], w, None)
    for a, b in zip(got, want):
        torch.testing.assert_close(a, b, rtol=1e-4, atol=1e-5 * float(b.abs().max()))

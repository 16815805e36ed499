"""gsplat_hip_tile_render called directly: its offsets, lists and report against the staged binning, and
the groups of tiles it leaves out."""
import pytest
import torch

from torch_gsplat_bridge_fast import _lib, _ops
from torch_gsplat_bridge_fast.scenes import make_scene_2d

pytestmark = pytest.mark.gpu

KEYS = ("means2d", "conics", "colors", "opacities", "depths")
LIST, BUCKET = 512, 16384   # kTileList, kTileBucket
WORK = 1 << 20              # kTileWorkSmall, kTileWork: a bucket's list lengths squared, up to 64K splats and above


def _tile_render(meta, flat, cap, fill):
    """(host words, tile_offsets, binned_ids (pre-filled with `fill`), image, stops)"""
    L, p = _lib.lib(), _lib.ptr
    B, G, H, W = meta.batch, meta.gaussians_per_batch, meta.height, meta.width
    tiles = B * ((H + 15) // 16) * ((W + 15) // 16)
    ws_bytes = L.gsplat_hip_tile_workspace_bytes(meta, cap)
    assert ws_bytes > 0
    ws = torch.empty(ws_bytes, dtype=torch.uint8, device="cuda")
    rws = torch.empty(L.gsplat_hip_render_workspace_bytes(meta, cap), dtype=torch.uint8, device="cuda")
    packed = torch.empty(B * G, 16, device="cuda")
    offsets = torch.empty(tiles + 1, dtype=torch.int32, device="cuda")
    ids = torch.full((cap,), fill, dtype=torch.int32, device="cuda")
    words = torch.zeros(4, dtype=torch.int32, pin_memory=True)
    img, T = torch.empty(B, H, W, 3, device="cuda"), torch.empty(B, H, W, device="cuda")
    last = torch.empty(B, H, W, dtype=torch.int32, device="cuda")
    stop = torch.empty(tiles, dtype=torch.int32, device="cuda")
    _lib.check(L.gsplat_hip_tile_render(meta, *map(p, flat), cap, p(packed), p(offsets), p(ids), words.data_ptr(),
                                        p(img), p(T), p(last), p(stop), p(ws), ws_bytes, p(rws), rws.numel(),
                                        _lib.stream_of(img)), "tile_render")
    torch.cuda.synchronize()
    assert int(words[3]) == 1
    return words.tolist(), offsets, ids, img, stop


@pytest.mark.parametrize("kind,B,G,H,W", [
    ("uniform", 1, 16384, 512, 272),
    ("ties", 3, 21845, 300, 400),
    ("uniform", 1, 70001, 4096, 4096),   # 256 tiles a bucket
    ("culled", 1, 20002, 600, 600),      # no pair at all
    ("hot tile", 1, 20000, 600, 600),
    ("hot bucket", 1, 60000, 600, 600),
    ("hot tile", 1, 40000, 900, 800),    # 2850 tiles: the forward of a wavefront per tile
])
def test_tile_render_lists(kind, B, G, H, W):
    """Offsets and ids of the staged binning; where a list or a bucket is too long, the skew bit, and an
    image that is the staged one outside those buckets and the background inside them."""
    print(f"tile render {kind} {B}x{H}x{W} G={G}", flush=True)
    g = torch.Generator().manual_seed(5)
    sc = make_scene_2d(1, seed=3, G=G, B=B, H=H, W=W)
    if kind == "ties":
        sc["depths"] = torch.randint(0, 9, (B, G), generator=g).float()
    if kind == "hot tile":
        sc["means2d"][:, :900] = 300.0 + 2.0 * torch.rand(B, 900, 2, generator=g)
        sc["opacities"] = 0.3 * sc["opacities"]
    if kind == "hot bucket":
        sc["means2d"][:, :40000] = torch.tensor([0.0, 296.0]) + torch.rand(B, 40000, 2, generator=g) * torch.tensor([600.0, 20.0])
        sc["opacities"] = 0.3 * sc["opacities"]
    if kind == "culled":
        sc["opacities"] = 0.0 * sc["opacities"]
    bg = (0.1, 0.2, 0.3)
    flat = [sc[k].reshape(B * G, -1).squeeze(-1).contiguous().cuda() for k in KEYS]
    meta = _lib.make_raster_meta(H, W, B, G, 1 / 255, 1e-4, bg)
    ref = _ops.bin_gaussians(meta, *flat)
    img, _, _, stop, _ = _ops.render_forward(meta, ref, save_state=True)
    n, counts = ref.n_pairs, ref.tile_counts.long()
    gid = torch.arange(B * G, device="cuda")
    orig = gid // G * G + ref.perm.long()
    want = orig[ref.binned_ids.long()]
    T = ref.num_tiles
    per = 1 << ((T - 1).bit_length() - 8)    # tiles a bucket
    bucket = torch.arange(T, device="cuda") // per
    size, work, hot = (torch.zeros(256, dtype=torch.long, device="cuda").index_add_(0, bucket, x)
                       for x in (counts, counts * counts, (counts > LIST).long()))
    bad = (size > BUCKET) | (work > (WORK if B * G <= 65536 else 3 * WORK // 2)) | (hot > 0)
    assert bool(bad.any()) == kind.startswith("hot")
    first_bad = int(bad.nonzero()[0]) if bad.any() else 0
    before = first_bad * per - 1             # the tile before a group that is left out
    # whatever the ids held: a splat of that tile, so that a range over them would show
    fill = int(want[int(ref.tile_offsets[before])]) if bad.any() else 0
    if bad.any():
        assert before >= 0 and int(counts[before]) > 0
    words, offsets, ids, img2, stop2 = _tile_render(meta, flat, max(1, n), fill)
    assert words[0] == n and words[1] == 0
    assert bool(words[2] & 2) == bool(bad.any())
    skip = bad[bucket]
    assert torch.equal(offsets[:-1][~skip], ref.tile_offsets[:-1][~skip]) and int(offsets[-1]) == n
    inside = ~torch.repeat_interleave(skip, counts)
    assert torch.equal(ids[:n][inside].long(), want[inside])
    # (above 2048 tiles, lists above the hand-off length are left to the caller's continuation)
    whole = ~skip & ((counts <= _lib.HANDOFF_PAIRS) | (T <= 2048))
    assert before < 0 or bool(whole[before])
    ny, nx = (H + 15) // 16, (W + 15) // 16

    def pixels(tiles):
        return tiles.reshape(B, ny, nx).repeat_interleave(16, 1).repeat_interleave(16, 2)[:, :H, :W]

    assert torch.equal(img2[pixels(whole)], img[pixels(whole)]) and torch.equal(stop2[whole], stop[whole])
    out = img2[pixels(skip)]
    assert torch.equal(out, torch.tensor(bg, device="cuda").expand_as(out))

"""GPU parity of the row spans (binning.hip, span_constants) with the oracle, which tests every
tile of a splat's box.  Bar: bit-exact."""
import numpy as np
import pytest
import torch

from oracle import tile_oracle as TO
from torch_gsplat_bridge_fast import _lib, _ops

pytestmark = pytest.mark.gpu

KEYS = ("means2d", "conics", "colors", "opacities", "depths")


@pytest.mark.parametrize("seed,B,H,W,G,lo,hi,ratio", [
    (1, 1, 203, 341, 4000, 2.0, 60.0, (0.03, 1.0)),    # ragged last row and column
    (2, 2, 513, 1025, 3000, 8.0, 120.0, (0.06, 0.13)),  # 1 - r^2 on both sides of 2^-7 at 45 degrees
    (3, 1, 1, 4097, 2000, 0.3, 300.0, (0.001, 1.0)),   # one row, needles
    (4, 1, 4097, 3, 2000, 0.3, 300.0, (0.001, 1.0)),   # one column
    (5, 1, 260, 530, 140000, 0.3, 6.0, (0.05, 1.0)),   # the original-order emit
])
def test_binning_row_spans(gpu, seed, B, H, W, G, lo, hi, ratio):
    """Every axis ratio, angle and size, centres off-screen, opacities from the threshold up, and
    conics that no span is computed for (zero, negative, infinite, NaN entries)."""
    print(f"row spans seed={seed} {B}x{H}x{W} G={G}", flush=True)
    rng = np.random.default_rng(seed)
    n = B * G
    m = np.stack([rng.uniform(-0.2 * W - 20, 1.2 * W + 20, n), rng.uniform(-0.2 * H - 20, 1.2 * H + 20, n)], -1)
    s1 = np.exp(rng.uniform(np.log(lo), np.log(hi), n))
    s2 = s1 * rng.uniform(*ratio, n)
    th = rng.uniform(0, np.pi, n)
    c, s = np.cos(th), np.sin(th)
    ix, iy = 1 / s1 ** 2, 1 / s2 ** 2
    q = np.stack([c * c * ix + s * s * iy, c * s * (ix - iy), s * s * ix + c * c * iy], -1).astype(np.float32)
    odd = np.array([0.0, -1.0, np.inf, -np.inf, np.nan, 1e-8, 1e-9, 1e30, 1e-30], np.float32)
    for k in range(90):
        q[k, k % 3] = odd[k // 3 % 9]
    m[90:100] = np.round(m[90:100] / 16) * 16 + 0.5   # on the tiles' edges
    o = np.exp(rng.uniform(np.log(1.0 / 255.0 * 1.0001), 0.0, n))
    sc = {k: torch.from_numpy(np.asarray(v, np.float32)).reshape(B, G, *v.shape[1:]) for k, v in dict(
        means2d=m, conics=q, colors=rng.uniform(0, 1, (n, 3)), opacities=o, depths=rng.uniform(0.1, 10, n)).items()}
    with np.errstate(all="ignore"):
        ob = TO.bin_scene(TO.make_meta(H, W, B, G), TO.Scene(*(sc[k].numpy() for k in KEYS), B, G))
    meta = _lib.make_raster_meta(H, W, B, G, 1.0 / 255.0, 1e-4, (0.0, 0.0, 0.0))
    flat = [sc[k].flatten(0, 1).to(gpu) for k in KEYS]
    for _ in range(2):   # the four-call binning, then the one-call path with the remembered buffer
        st = _ops.bin_gaussians(meta, *flat)
        np.testing.assert_array_equal(st.tile_counts.cpu().numpy(), ob.tile_counts)
        np.testing.assert_array_equal(st.tile_offsets.cpu().numpy(), ob.tile_offsets)
        np.testing.assert_array_equal(st.binned_ids.cpu().numpy(), ob.binned_ids)

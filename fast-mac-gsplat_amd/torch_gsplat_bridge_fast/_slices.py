"""The sliced forward and backward of dense scenes (gsplat_hip_front_render and
following in gsplat_hip.h).

Where tiles list hundreds of pairs but are opaque after a few dozen, the
nearest splats alone (the front) are binned and composited first, and the
tiles that stay transparent (the live tiles) are then done again from their
whole lists (the back).  The image, stops and gradients are those of the
unsliced path.  A shape is sliced when the pair count of its last binning
makes the front a small part of it; the front's budget per tile follows the
stops that the shape's last sliced call reported, and a shape whose tiles do
not turn opaque early goes back to the unsliced path.

What a sliced forward saves differs from call to call (the budget follows the
calls before it, and there may be no back).  Where saved tensors go through
hooks, a training forward is not sliced: non-reentrant checkpointing compares
what its recomputation saves with what the first pass saved.
"""
from __future__ import annotations

import ctypes
import itertools
from typing import Optional

import torch
from torch import Tensor

from . import _lib, _ops
from ._lib import check, ptr

# Slicing pays above MIN_PAIRS + MIN_PAIRS_PER_TILE * tiles pairs: the binning of the whole scene grows
# with its pairs, the slices' own launches and the host's wait between them do not (about 250 us), and
# the live tiles composited twice grow with the image.  3D scenes, forward + backward, whole against
# sliced: 4096^2, 122M pairs 2720 -> 1480 us; 4000 x 3000, 46M 1435 -> 1016 us; 1080p, 21.6M 960 -> 820 us;
# 1080p translucent, 20M 1355 -> 1290 us; below the line 2048^2, 21M 1071 -> 1093 us; 4000 x 3000, 13.7M
# 983 -> 1000 us; 1080p translucent, 8M 1083 -> 1245 us.
MIN_PAIRS = 14 << 20
MIN_PAIRS_PER_TILE = 512
# Box tiles per tile that the front of a shape's first sliced call takes.
FIRST_BUDGET = 192
MAX_SLOTS = 1 << 17     # splats per image of the two-launch depth order


class _Plan:
    """What a shape's calls have shown: the front's budget (box tiles per tile; 0: not worth slicing)
    and the pair capacity it was chosen for."""
    __slots__ = ("budget", "capacity")

    def __init__(self, capacity: int):
        self.budget = FIRST_BUDGET
        self.capacity = capacity


_plans: dict = {}


def _budget(key: tuple, tiles: int) -> Optional[_Plan]:
    """The plan of a shape that is to be sliced, else None."""
    cap = _ops._capacity.get(key)
    # (the capacity is a quarter above the pairs it was taken from)
    if cap is None or 4 * cap < 5 * (MIN_PAIRS + MIN_PAIRS_PER_TILE * tiles) or _ops._staged():
        return None
    plan = _plans.get(key)
    if plan is None or cap > 2 * plan.capacity or 2 * cap < plan.capacity:
        if len(_plans) > 256:
            _plans.clear()
        plan = _plans[key] = _Plan(cap)
    if plan.budget == 0 or 4 * plan.budget * tiles > 3 * cap:
        return None
    return plan


class _SliceRows:
    """A ring of pinned host words per device, one 16-word row per front."""
    RING = 256

    def __init__(self):
        self.tensor = torch.zeros((self.RING, 16), dtype=torch.int32, pin_memory=True)
        self.rows = self.tensor.numpy()
        self.base = self.tensor.data_ptr()
        self.calls = itertools.count()


class _Row:
    """Adapts a 16-word row to _ops._ReportReady, which polls word 3 of a 4-word row."""
    __slots__ = ("row",)

    def __init__(self, row):
        self.row = row

    def __getitem__(self, k):
        return self.row[15 if k == 3 else k]


_rows: dict = {}


_sizes: dict = {}


def _slice_sizes(meta: _lib.RasterMeta, key: tuple, slots: int, capacity: int, save_state: bool) -> tuple:
    """Byte offsets of a slice's parts.  Kept until the backward: (packed, pairs, tile_offsets,
    tile_stop, render workspace, end); only until the forward is enqueued: (splats, binning workspace,
    end)."""
    k = (key, slots, capacity, save_state)
    v = _sizes.get(k)
    if v is None:
        L = _lib.lib()
        B, H, W = meta.batch, meta.height, meta.width
        tiles = B * ((H + 15) // 16) * ((W + 15) // 16)
        m = _lib.RasterMeta.from_buffer_copy(meta)
        m.gaussians_per_batch = slots

        def offsets(*sizes):
            out = [0]
            for n in sizes:
                out.append(out[-1] + (n + 255) // 256 * 256)
            return tuple(out)

        v = (offsets(B * slots * 4 * _lib.RECORD_FLOATS, 4 * capacity, 4 * (tiles + 1), 4 * tiles,
                     L.gsplat_hip_render_workspace_bytes(m, capacity if save_state else 0)),
             offsets(L.gsplat_hip_slice_splats_bytes(B, slots), L.gsplat_hip_bin_workspace_bytes(m, capacity)))
        if len(_sizes) > 256:
            _sizes.clear()
        _sizes[k] = v
    return v


class _Slice:
    """One slice's buffers: `kept` for the backward, `used` by the forward."""
    __slots__ = ("slots", "capacity", "layout", "kept", "used")

    def __init__(self, meta: _lib.RasterMeta, key: tuple, slots: int, capacity: int, save_state: bool, device):
        self.slots, self.capacity = slots, capacity
        keep, use = _slice_sizes(meta, key, slots, capacity, save_state)
        self.layout = keep
        self.kept = torch.empty(keep[-1], dtype=torch.uint8, device=device)
        self.used = (torch.empty(use[-1], dtype=torch.uint8, device=device), use)

    def struct(self) -> _lib.Slice:
        return _struct(self.kept, self.layout, self.slots, self.capacity, self.used)


def _struct(kept: Tensor, o: tuple, slots: int, capacity: int, used=None) -> _lib.Slice:
    p = kept.data_ptr()
    s = _lib.Slice()
    s.capacity, s.slots = capacity, slots
    s.packed, s.binned_ids, s.tile_offsets, s.tile_stop = p, p + o[1], p + o[2], p + o[3]
    s.render_workspace, s.render_workspace_bytes = p + o[4], o[5] - o[4]
    if used is not None:
        q, u = used[0].data_ptr(), used[1]
        s.splats, s.splats_bytes = q, u[1]
        s.bin_workspace, s.bin_workspace_bytes = q + u[1], u[2] - u[1]
    return s


class SlicedState:
    """What a sliced forward leaves for its backward: tensors() for autograd to save, and plain()."""

    def __init__(self, front: _Slice, back: Optional[_Slice], live_list: Tensor, n_live: int, records: Optional[Tensor],
                 back_state: Optional[_ops.BinState]):
        self._tensors = (live_list, records, front.kept) + (() if back is None else (back.kept,))
        self.n_live = n_live
        self._slices = tuple((x.layout, x.slots, x.capacity) for x in (front, back) if x is not None)
        self._back_state = back_state

    @property
    def has_back(self) -> bool:
        return len(self._slices) > 1

    def tensors(self) -> tuple:
        return self._tensors

    def plain(self) -> tuple:
        return self.n_live, self._slices

    def release(self) -> None:
        """Drops the tensors (autograd holds those it needs)."""
        self._tensors = ()

    def check_status(self) -> None:
        if self._back_state is not None:
            self._back_state.check_status()


def _report(row) -> tuple:
    """(status, live tiles, slots, fresh, box tiles, back tiles, stops, opaque tiles) of a front's row."""
    w = [int(row[k]) & 0xffffffff for k in range(12)]
    return w[0], w[1], w[2], w[3], *(w[4 + 2 * k] | w[5 + 2 * k] << 32 for k in range(4))


def _adapt(plan: _Plan, tiles: int, live: int, box: int, back: int, stops: int, opaque: int) -> None:
    """The shape's next budget.  A front that left more than a quarter of the work to the back was too
    small; otherwise the budget is the box tiles (about 1.3 per pair) of the opaque tiles' mean stop and
    a margin for the tiles above it."""
    if 4 * back > box:
        plan.budget *= 2
    elif opaque > 0:
        want = (3 * stops // (2 * opaque) + 24 + 31) // 32 * 32
        if 5 * want < 4 * plan.budget or 4 * want > 5 * plan.budget:
            plan.budget = want
    if 2 * plan.budget * tiles > box:
        plan.budget = 0


def _step_up(n: int) -> int:
    """n or a little more: a multiple of an eighth of the power of two below it, and of 256."""
    step = max(256, 1 << max(0, n.bit_length() - 4))
    return (max(n, 1) + step - 1) // step * step


def render(meta: _lib.RasterMeta, flat, *, save_state: bool):
    """(SlicedState, (img, final_T, last)) if this shape is sliced and the scene turned out to suit it,
    else None (the caller takes the unsliced path).  Raises if a binning of the front failed; the
    caller runs check_status() for the back's."""
    means2d = flat[0]
    dev = means2d.device
    B, G, H, W = meta.batch, meta.gaussians_per_batch, meta.height, meta.width
    key = (dev.index, B, G, H, W)
    tpi = ((H + 15) // 16) * ((W + 15) // 16)
    plan = _budget(key, B * tpi)
    if plan is None or (save_state and _lib.host().saved_tensor_hooks()):
        return None
    L = _lib.lib()
    ws_bytes = L.gsplat_hip_slice_workspace_bytes(meta)
    if ws_bytes == 0:   # not a scene that can be sliced
        return None
    cap = _ops._capacity[key]
    budget = plan.budget
    # as many splats as the budget holds at the scene's mean pairs per splat (the nearest are larger)
    slots = min(G, MAX_SLOTS, (524288 // B) & ~4095, (int(1.1 * budget * tpi * B * G / cap) // 4096 + 1) * 4096)
    if slots <= 0:
        return None
    front = _Slice(meta, key, slots, B * budget * tpi, save_state, dev)
    img = torch.empty((B, H, W, 3), dtype=torch.float32, device=dev)
    final_T = last = records = None
    if save_state:
        final_T = torch.empty((B, H, W), dtype=torch.float32, device=dev)
        last = torch.empty((B, H, W), dtype=torch.int32, device=dev)
        records = torch.empty((B * G, _lib.GRAD_RECORD_FLOATS), dtype=torch.float32, device=dev)
    live_list = _ops._empty(B * tpi, torch.int32, dev)
    ws = _ops._empty(ws_bytes, torch.uint8, dev)
    rows = _rows.get(dev.index)
    if rows is None:
        rows = _rows[dev.index] = _SliceRows()
    slot = next(rows.calls) % rows.RING
    args = [ptr(t) for t in flat]
    stream = torch.cuda.current_stream(dev).cuda_stream
    check(L.gsplat_hip_front_render(meta, *args, front.struct(), ptr(img), ptr(final_T), ptr(last), ptr(records),
                                    ptr(live_list), ptr(ws), ws.numel(), rows.base + 64 * slot, stream),
          "gsplat_hip_front_render")
    row = rows.rows[slot]
    _ops._ReportReady(_Row(row), dev).synchronize()
    status, live, back_slots, fresh, box, back_tiles, stops, opaque = _report(row)
    if status:
        raise RuntimeError(f"binning failed with device status {status:#x} (a decoupled look-back wait gave up); the "
                           "results of this call are invalid")
    # (the box tiles bound the pairs: a much sparser scene lowers the shape's capacity, and says nothing
    # about the scenes that raise it again)
    if _ops._headroom(box) < cap // 2:
        _ops._capacity[key] = _ops._headroom(box)
        _plans.pop(key, None)
    else:
        _adapt(plan, B * tpi, live, box, back_tiles, stops, opaque)
    if live == 0 or fresh == 0:
        return SlicedState(front, None, live_list, 0, records, None), (img, final_T, last)
    if 2 * back_tiles > box or back_tiles > _ops.MAX_PAIRS:
        return None
    # (in steps of 1/8 of a power of two, so that a scene's next calls find the sizes known)
    slots = min(G, _step_up(back_slots))
    back = _Slice(meta, key, slots, min(_step_up(back_tiles), _ops.MAX_PAIRS), save_state, dev)
    d = _ops._device_bin.get(dev.index)
    if d is None:
        d = _ops._device_bin[dev.index] = _ops._DeviceBinState(dev)
    slot = d.slot()
    check(L.gsplat_hip_back_render(meta, *args, back.struct(), ptr(img), ptr(final_T), ptr(last), ptr(live_list), live,
                                   ptr(ws), ws.numel(), d.ring_base + 16 * slot, stream,
                                   _ops._side_stream(dev).cuda_stream, d.inputs.cuda_event, d.count.cuda_event),
          "gsplat_hip_back_render")
    ready = _ops._ReportReady(d.ring[slot], dev)
    # (without the tensors: only the status is read from it)
    st = _ops.BinState(None, None, None, None, None, back.capacity, d.ring, ready, None, None, (slot, 0), d.ring,
                       (slot, 1), ready, d, d.calls - 1, (slot, 2))
    return SlicedState(front, back, live_list, live, records, st), (img, final_T, last)


def backward(meta: _lib.RasterMeta, tensors: tuple, plain: tuple, final_T: Tensor, last: Tensor, grad_img: Tensor,
             out: tuple) -> tuple:
    """The gradients into the buffers `out` (_ops.gradient_buffers); tensors and plain: SlicedState's."""
    n_live, slices = plain
    live_list, records, *kept = tensors
    front, back = [_struct(k, *x) for k, x in zip(kept, slices)] + [None] * (2 - len(slices))
    grad_img = grad_img.contiguous()
    g_m, g_q, g_c, g_o = out
    with _ops._timed("render_backward"):
        check(_lib.lib().gsplat_hip_sliced_backward(
            meta, front, back, ptr(live_list), n_live, ptr(final_T), ptr(last), ptr(grad_img), ptr(records), ptr(g_m),
            ptr(g_q), ptr(g_c), ptr(g_o), _lib.stream_of(grad_img)), "gsplat_hip_sliced_backward")
    return out

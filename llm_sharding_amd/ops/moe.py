"""Bindings and weights of the mixture-of-experts kernels (csrc/kernels/moe.hip).

The conventions of :mod:`.hip` hold: shapes are checked on the host, launches go to torch's current
stream, nothing falls back to another implementation."""
from __future__ import annotations

import ctypes
import functools
from typing import Optional

import torch

from . import hip
from .hip import _check, _p, _req, _stream, lib
from .packing import fuse_gate_up, pack_b, pack_f32
from .stream import is_f32, pad2


def pad128(n: int) -> int:
    return -(-n // 128) * 128


DOWN, GLU, RELU2 = 0, 1, 2  # MoeUp in csrc/kernels/moe.h


class RouteArgs(ctypes.Structure):
    _fields_ = [("correction", ctypes.c_void_p), ("sigmoid", ctypes.c_int), ("groups", ctypes.c_int), ("keep", ctypes.c_int),
                ("scale", ctypes.c_float)]


class Pick(ctypes.Structure):  # csrc/kernels/moe.h MoePick
    _fields_ = [("nt", ctypes.c_int * 2), ("step", (ctypes.c_float * 2) * 4), ("own", ctypes.c_float * 4)]


HEIGHTS = (128, 192, 256, 320)  # of the bf16 kernel's tiles of 256 columns (MOE_ROWS)
# us of such a tile on every CU, as measured in the projection GEMM: a 64-deep K step, and its start and end; and what low ones take
# more because they read an expert's weights more often
HEIGHT_COST = ((0.84, 3.8, 1.06), (1.09, 6.1, 1.03), (1.36, 7.9, 1.0), (1.70, 9.9, 1.0))


@functools.lru_cache(maxsize=256)
def pick(*products) -> Optional[Pick]:
    """What :func:`group` chooses a height from for both of the experts' products [(columns, k)]: what a round of such tiles takes;
    None: not for these."""
    if any(n % 256 or k % 64 for n, k in products):
        return None
    p = Pick(tuple(n // 256 for n, _ in products))
    for i, (step, own, more) in enumerate(HEIGHT_COST):
        p.step[i] = tuple(more * (k // 64 * step) for _, k in products)
        p.own[i] = more * own
    return p


def heights(pairs: int, experts: int, rows: int, f32, *products) -> Optional[Pick]:
    """:func:`pick` where the height is picked when the pairs are counted: bf16 tiles of ``rows`` >= 128, in tables that lsa_moe_group
    takes with heights (2^19 tiles of the lowest). None: tiles of ``rows``."""
    return pick(*products) if rows >= 128 and not f32 and max_tiles(pairs, experts, HEIGHTS[0]) < 1 << 19 else None


def route_args(s=None, correction=None) -> RouteArgs:
    """How the experts of ``s`` (a MoeSpec; None: softmax over the largest logits) are chosen."""
    if s is None:
        return RouteArgs(None, 0, 1, 1, 1.0)
    _req(correction is None or (correction.dtype == torch.float32 and correction.numel() == s.experts
                                and correction.is_contiguous()), "route: correction")
    return RouteArgs(_p(correction), int(s.sigmoid), s.groups, s.keep, float(s.scale))


class Experts:
    """The experts' products, one after another: gate and up interleaved by 16 rows [E][2 ff][width] (without gates
    up alone [E][ff][width]) and down [E][width][ff], sizes padded to 128, packed for the matrix kernels
    of their type."""

    def __init__(self, gate: Optional[list], up: list, down: list):
        self.ff, self.width = pad128(up[0].shape[0]), pad128(up[0].shape[1])
        self.f32 = is_f32(up[0].dtype)
        self.kind = RELU2 if gate is None else GLU
        lay = pack_f32 if self.f32 else pack_b
        ups = [pad2(u, self.ff, self.width) for u in up]
        if gate is not None:
            ups = [fuse_gate_up(pad2(g, self.ff, self.width), u) for g, u in zip(gate, ups)]
        self.up = torch.stack([lay(u) for u in ups])
        self.up_n = ups[0].shape[0]
        self.down = torch.stack([lay(pad2(d, self.width, self.ff)) for d in down])
        self.experts = len(up)

    def tensors(self) -> list:
        return [self.up, self.down]


def tile_rows(pairs: int, experts: int, f32: bool, cols: Optional[int] = None) -> int:
    """Pairs per tile: what an expert gets on average, rounded to a kernel's size. ``cols``: of the narrower of the two products (None:
    wide enough)."""
    mean = pairs / experts  # (a second tile of an expert reads its weights again)
    if f32:  # 64 x 128 and 128 rows x 256 columns: 90 pairs an expert 3907 and 4155 us a pass (Runidra 2k), 183 6000 and 5662, 104
        # 3780 and 3804 (Dumizen 2k), 141 4568 and 4440. The large ones keep a CU for more than twice as long and are for products with as
        # many as 160 of them: 8 experts of 1024 x 2048, 136 pairs each 51 and 122 us, 32 experts 145 and 138. With narrow ones (gemm)
        # 1.02 times the fastest of all three, worst 1.45 (just under 112 pairs); by the pairs alone 1.37, worst 4.0 (270 products
        # of 2 to 32 experts, 768 to 4096 columns and 26 to 400 pairs evenly drawn, profiles/cost_moe_f32.csv).
        if mean > 112 and (cols is None or experts * max(1.0, mean / 128 + 0.5) * -(-cols // 256) >= 160):
            return 128
        return next((n for n in (16, 32) if mean <= 0.75 * n), 64)
    return next((n for n in (16, 32, 64) if mean <= 0.75 * n), 128 if mean <= 320 else 256)


def narrow_tiles(pairs: int, experts: int, rows: int, cols: int) -> bool:
    """Whether tiles of 64 rows have 64 columns instead of 128 (fp32): where there are no more of those than CUs, with 3/8 of a tile
    more per expert than its pairs fill. 1024 x 2048: 128 tiles 30 and 46 us, 256 33 and 48, 288 58 and 50."""
    n = min(experts, pairs)
    return rows == 64 and n * max(1.0, pairs / n / 64 + 0.375) * -(-cols // 64) <= 256


def max_tiles(pairs: int, experts: int, rows: int) -> int:
    return min(experts, pairs) + pairs // rows


def route(logits, rows: int, experts: int, top: int, expert, weight, how: Optional[RouteArgs] = None) -> None:
    """fp32 router logits -> chosen experts and their weights [rows * top]."""
    how = how or route_args()
    _req(logits.dtype == torch.float32 and logits.stride(1) == 1 and logits.shape[0] >= rows
         and logits.shape[1] >= experts, "route: logits")
    _req(expert.dtype == torch.int32 and weight.dtype == torch.float32 and min(expert.numel(), weight.numel()) >= rows * top,
         "route: outputs")
    _check(lib().lsa_moe_route(ctypes.byref(how), _p(logits), logits.stride(0), rows, experts, top, _p(expert), _p(weight), _stream()),
           "lsa_moe_route")


def group(expert, pairs: int, experts: int, rows: int, order, place, tiles, spare=None, heights: Optional[Pick] = None) -> int:
    """Pairs sorted by expert (``order``; ``place`` is its inverse) and their tiles; returns the table's length. ``spare``: int32
    scratch, as long as the pairs, that lets many of them have several workgroups. ``heights`` (:func:`pick`): the tiles are as high
    as the pairs make best, ``rows`` is the lowest; for :func:`gemm` with ``rows`` 0."""
    n = max_tiles(pairs, experts, rows)
    _req(all(t.dtype == torch.int32 for t in (expert, order, place, tiles)) and tiles.numel() >= 4 * n
         and min(expert.numel(), order.numel(), place.numel()) >= pairs, "group: shapes")
    _req(spare is None or (spare.dtype == torch.int32 and spare.is_contiguous()), "group: scratch")
    _check(lib().lsa_moe_group(_p(expert), pairs, experts, rows, n, _p(order), _p(place), _p(tiles), _p(spare),
                               0 if spare is None else spare.numel(), heights, _stream()), "lsa_moe_group")
    return n


def route_group(logits, rows: int, experts: int, top: int, tile: int, expert, weight, order, place, tiles,
                how: Optional[RouteArgs] = None, spare=None, heights: Optional[Pick] = None) -> int:
    """:func:`route` and :func:`group`, in one launch where there are few rows (and the height is given)."""
    pairs, how = rows * top, how or route_args()
    if rows > 16 or experts > 256 or heights is not None:
        route(logits, rows, experts, top, expert, weight, how)
        return group(expert, pairs, experts, tile, order, place, tiles, spare, heights)
    n = max_tiles(pairs, experts, tile)
    _req(logits.dtype == torch.float32 and logits.stride(1) == 1 and logits.shape[0] >= rows
         and logits.shape[1] >= experts and weight.dtype == torch.float32 and weight.numel() >= pairs, "route: shapes")
    _req(all(t.dtype == torch.int32 for t in (expert, order, place, tiles)) and tiles.numel() >= 4 * n
         and min(expert.numel(), order.numel(), place.numel()) >= pairs, "group: shapes")
    _check(lib().lsa_moe_route_group(ctypes.byref(how), _p(logits), logits.stride(0), rows, experts, top, _p(expert), _p(weight), tile, n,
                                     _p(order), _p(place), _p(tiles), _stream()), "lsa_moe_route_group")
    return n


def gemm(tiles, n_tiles: int, rows: int, order, top: int, a, w, n: int, k: int, out, pairs: int, up: int) -> None:
    """One product of every tile's expert: ``up`` (GLU / RELU2) from rows of h (``a``) to out [pairs, n / 2 or n], or
    DOWN from the sorted pairs (``a`` [pairs, k]) to out [pairs, n]. ``rows`` 0: tiles of the height that :func:`group` chose."""
    _req(a.dtype == w.dtype == out.dtype and a.stride(1) == 1 and a.shape[1] >= k and out.stride(1) == 1
         and out.shape[0] >= pairs and out.shape[1] >= (n // 2 if up == GLU else n) and order.numel() >= pairs
         and (a.shape[0] * top >= pairs if up else a.shape[0] >= pairs), "moe: shapes")
    _req(w[0].numel() == n * k and w.is_contiguous(), "moe: weights")
    f32 = is_f32(a.dtype)
    if (rows > 64 or not rows) and not f32:
        _check(lib().lsa_moe_gemm_big(up, _p(tiles), n_tiles, rows, _p(order), top, _p(a), a.shape[0] if up else 0,
                                      a.stride(0), _p(w), n, k, _p(out), out.stride(0), _stream()), "lsa_moe_gemm_big")
        return
    narrow = bool(f32) and narrow_tiles(pairs, w.shape[0], rows, n)
    _check(lib().lsa_moe_gemm(f32, up, _p(tiles), n_tiles, rows, narrow, _p(order), top, _p(a), a.stride(0), _p(w),
                              n, k, _p(out), out.stride(0), _stream()), "lsa_moe_gemm")


def declare(L: ctypes.CDLL) -> None:
    """Signatures of these entry points (called by hip.load_library)."""
    vp, i, ra = ctypes.c_void_p, ctypes.c_int, ctypes.POINTER(RouteArgs)
    hip.set_signatures(L, {
        "lsa_moe_route": [ra, vp, i, i, i, i, vp, vp, vp],
        "lsa_moe_group": [vp, i, i, i, i, vp, vp, vp, vp, i, ctypes.POINTER(Pick), vp],
        "lsa_moe_route_group": [ra, vp, i, i, i, i, vp, vp, i, i, vp, vp, vp, vp],
        "lsa_moe_gemm_big": [i, vp, i, i, vp, i, vp, i, i, vp, i, i, vp, i, vp],
        "lsa_moe_gemm": [i, i, vp, i, i, i, vp, i, vp, i, vp, i, i, vp, i, vp],
    })

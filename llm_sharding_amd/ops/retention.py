"""Bindings of the retention kernels (csrc/kernels/retention*.hip).

The conventions of :mod:`.hip` hold: shapes are checked on the host, launches go to torch's current
stream, nothing falls back to another implementation."""
from __future__ import annotations

import ctypes

import torch

from . import hip
from .delta import check_runs  # noqa: F401  (one run per slot and step, as there)
from .hip import _check, _p, _req, _stream, lib
from .paged_attn import PAGE
from .stream import is_f32


class RetArgs(ctypes.Structure):
    _fields_ = ([(n, ctypes.c_void_p) for n in ("inp", "state", "cos", "sin", "decay", "runs", "slot", "pos", "table", "out")]
                + [(n, ctypes.c_int) for n in ("ldi", "ldo", "oq", "ok", "ov", "og", "heads", "dim", "vdim", "dk", "dv",
                                               "rot_dims", "max_pages", "n_pages")]
                + [(n, ctypes.c_float) for n in ("k_scale", "eps", "oscale")])


def make_args(s, decay, state, inp, cols: tuple, out, rot, eps: float, table, n_pages: int, slot=None, pos=None, runs=None,
              oscale: float = 1.0) -> RetArgs:
    """``state`` fp32 [slots, heads, *s.state_dims]; ``cols``: first columns of q, k, v and gate in ``inp``; ``rot``:
    (cos, sin, dims) or None; ``runs`` int32 [n, 4] (row0, rows, slot, pos0), checked by :func:`check_runs`, or
    ``slot`` / ``pos`` int32 [rows]; ``oscale``: factor of the output."""
    _req(state.dtype == decay.dtype == torch.float32 and state.is_contiguous() and decay.numel() == s.heads
         and tuple(state.shape[1:]) == (s.heads,) + s.state_dims, "retention: state")
    kc, vc = (s.heads * n for n in s.state_dims)
    _req(inp.dtype == out.dtype and inp.stride(1) == out.stride(1) == 1 and out.shape[0] >= inp.shape[0]
         and out.shape[1] >= vc and inp.shape[1] >= max(cols[0] + kc, cols[1] + kc, cols[2] + vc, cols[3] + vc),
         "retention: inputs")
    _req((runs is None) != (slot is None), "retention: runs or rows")
    _req(table.dtype == torch.int32 and table.shape[0] <= state.shape[0], "retention: page table")
    for t in (runs, slot, pos):
        _req(t is None or (t.dtype == torch.int32 and t.is_contiguous()), "retention: int32 rows")
    cos, sin, dims = rot if rot is not None else (None, None, 0)
    _req(rot is None or (cos.dtype == sin.dtype == torch.float32 and cos.is_contiguous() and sin.is_contiguous()
                         and cos.shape == sin.shape == (cos.shape[0], dims // 2)
                         and cos.shape[0] >= table.shape[1] * PAGE), "retention: rotation tables")
    return RetArgs(_p(inp), _p(state), _p(cos), _p(sin), _p(decay), _p(runs), _p(slot), _p(pos), _p(table), _p(out),
                   inp.stride(0), out.stride(0), *cols, s.heads, s.dim, s.vdim, *s.state_dims, dims, table.shape[1], n_pages,
                   float(s.k_scale), float(eps), float(oscale))


CHUNK = 64  # rows per chunk (C in csrc/kernels/retention_chunk.hip)


def chunk_size(s) -> bool:
    """The chunked kernels take this size."""
    return max(s.state_dims) <= 128 and (s.rot is None or s.rot.dims % 16 == 0)


def segments(s, runs: list, want: int, least: int = 4 * CHUNK) -> tuple:
    """Runs (row0, rows, slot, pos0) cut into segments, so that the chunked kernel has about ``want`` workgroups, of
    ``least`` rows at least: (items int32 [n, 8] (RetItem), workspace entries, longest item, several per run)."""
    per = s.heads * (2 if s.state_dims[1] == 128 else 1)
    items, entry, several = [], 0, False
    parts = max(1, -(-want // (per * len(runs))))
    for row0, n, slot, pos0 in runs:
        length = -(-max(least, -(-n // parts)) // CHUNK) * CHUNK
        k = max(1, -(-n // length))
        items += [[row0 + i * length, min(length, n - i * length), slot, pos0 + i * length, entry, i, k, length]
                  for i in range(k)]
        entry += k
        several |= k > 1
    return torch.tensor(items, dtype=torch.int32), entry, max(i[1] for i in items), several


def chunked(a: RetArgs, s, items, longest: int, several: bool, ws, o32) -> None:
    """The segments of checked runs, bf16: ``items`` (device), ``ws`` fp32 [entries, heads, *s.state_dims] (with several
    segments per run), ``o32`` fp32 [rows, heads dv]."""
    _req(o32.dtype == torch.float32 and o32.stride(1) == 1 and o32.shape[1] >= s.heads * s.state_dims[1], "retention: read-outs")
    _req(items.dtype == torch.int32 and items.is_contiguous() and items.shape[1] == 8, "retention: segments")
    _req(not several or (ws.dtype == torch.float32 and ws.is_contiguous()), "retention: workspace")
    _check(lib().lsa_ret_chunked(ctypes.byref(a), _p(items), items.shape[0], longest, int(several), _p(ws), _p(o32),
                                 o32.stride(0), _stream()), "lsa_ret_chunked")


def steps(a: RetArgs, dtype, n: int, longest: int = 0) -> None:
    """n runs (or rows), step by step; ``longest``: none has more rows (0: not known)."""
    _check(lib().lsa_ret_steps(is_f32(dtype), ctypes.byref(a), n, longest, _stream()), "lsa_ret_steps")


def declare(L: ctypes.CDLL) -> None:
    """Signatures of these entry points (called by hip.load_library)."""
    vp, i = ctypes.c_void_p, ctypes.c_int
    ra = ctypes.POINTER(RetArgs)
    hip.set_signatures(L, {"lsa_ret_steps": [i, ra, i, i, vp], "lsa_ret_chunked": [ra, vp, i, i, i, vp, vp, i, vp]})

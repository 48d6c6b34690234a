"""Grouped-query attention over the paged cache as a layer mixer (:class:`..models.stack.AttentionSpec`):
weights and forward.

The projections of queries, keys, values and head gates ride in the block's input projection. One forward
of a row batch then is

    append      keys and values into the cache (not of a layer that reads another's); where they are normed or
                rotated first, queries and keys on the way; the means of finished blocks
    attention   runs of at least ``tile_min`` rows in query tiles, other rows one by one
    output      the block's output projection

A page holds keys token by token and values channel by channel (csrc/kernels/paged_attn.h). The CPU
engine keeps both token by token."""
from __future__ import annotations

import torch
import torch.nn.functional as F

from ..models.stack import HEAD, WHOLE, AttentionSpec
from .latent_mixer import _head_pad


def rotary_tables(rot, n: int, device) -> tuple:
    """cos, sin [n, dims / 2] fp32 of a RotarySpec's angles at positions 0 .. n - 1, times its amplitude."""
    ang = torch.outer(torch.arange(n, dtype=torch.float64), torch.tensor(rot.frequencies(), dtype=torch.float64))
    return tuple((f(ang) * rot.amplitude).float().to(device).contiguous() for f in (torch.cos, torch.sin))


def turned(eng, rot, x: torch.Tensor, pos) -> torch.Tensor:
    """x [n, heads, dim] rotated at positions ``pos`` (CPU engines)."""
    cos, sin = (t[pos][:, None] for t in eng.rotation(rot))
    half = rot.dims // 2
    u, v, rest = x[..., :half], x[..., half:2 * half], x[..., 2 * half:]
    return torch.cat([u * cos - v * sin, v * cos + u * sin, rest], -1)


class Attention:
    tile_min = 16  # rows from which a run of consecutive positions goes out in query tiles
    NORMS = {None: 0, HEAD: 1, WHOLE: 2}

    def __init__(self, spec: AttentionSpec, t: dict, gpu: bool, oscale: float = 1.0, alone: bool = True):
        """``oscale``: factor of the output; not ``alone``: ``out_weight`` goes into another's output projection."""
        self.spec, self.gpu, self.oscale, self.alone = spec, gpu, oscale, alone
        s = spec
        dev = t["q"].device
        temp = t["temp"].float() if s.head_temp else torch.ones(s.heads, device=dev)
        self.hscale = (temp * s.scale).contiguous()
        self.sig = torch.stack([t["r1"].float() if s.distance_bias else torch.zeros(s.heads, device=dev),
                                t["r2"].float() if s.distance_bias else torch.zeros(s.heads, device=dev),
                                t["pb"].float()]).contiguous() if s.sigmoid else None
        self.raw = None if gpu else t
        self.out_bias = t["o.b"].float().contiguous() if s.out_bias else None
        if not gpu:
            return
        from ..ops import paged_attn as A
        from ..ops import stream as L
        self.parts = []
        for name, heads, n, p in (("q", s.heads, s.dim, s.dkp), ("k", s.kv_heads, s.dim, s.dkp),
                                  ("v", s.kv_heads, s.vdim, s.dvp)):
            if name in t:
                bias = _head_pad(t[name + ".b"].float()[:, None], heads, [(n, p)])[:, 0] if s.bias else None
                self.parts.append((name, _head_pad(t[name], heads, [(n, p)]), bias, None))
        if s.head_gate:
            self.parts.append(("g", t["g"], None, None))
        if s.elem_gate:
            self.parts.append(("g", _head_pad(t["g"], s.heads, [(s.vdim, s.dvp)]), None, None))
        self.qk = None  # norm weights as the kernels read them
        if s.qk_norm is not None:
            self.qk = tuple(_head_pad(t[k + ".norm"].float()[:, None], n if s.qk_norm == WHOLE else 1, [(s.dim, s.dkp)])
                            .flatten().contiguous() for k, n in (("q", s.heads), ("k", s.kv_heads)))
        weight = _head_pad(t["o"].t().contiguous(), s.heads, [(s.vdim, s.dvp)]).t().contiguous()
        self.width, self.out_weight = weight.shape[1], None if alone else weight
        if alone:
            self.out = L.Linear(weight)
            if self.out_bias is not None:
                self.out_bias = F.pad(self.out_bias, (0, self.out.n - self.out_bias.numel()))
        self.tuned = A.tuned_size(s) and t["q"].dtype == torch.bfloat16

    def input_parts(self) -> list:
        return self.parts

    def tensors(self) -> list:
        if self.raw is not None:
            return list(self.raw.values())
        own = [self.hscale, self.sig, self.out_bias] + list(self.qk or ())
        return [t for t in own if t is not None] + (self.out.tensors() if self.alone else [])

    def scratch(self) -> dict:
        out = {"attn": self.out.k} if self.alone else {}
        if self.spec.prepared:
            out["q"] = self.spec.heads * self.spec.dkp
        return out

    def projections(self) -> list:
        return [self.out]

    # ------------------------------------------------------------------ GPU
    def forward(self, eng, inp, in32, col: dict, cache: tuple, state, slot, pos, rows: int, plan, ao=None) -> torch.Tensor:
        from ..ops import paged_attn as A
        s, table = self.spec, eng.pool.table
        ao = eng.scratch_view("attn", rows, self.out.k) if ao is None else ao

        def args(index=None):
            return A.make_args(s, cache, table, slot, pos, self.hscale, index=index, sig=self.sig, oscale=self.oscale,
                               ptable=eng.pools[s.pool].table if s.pool else None)
        a = args()
        gate = inp[:, col["g"]:] if s.head_gate or s.elem_gate else None
        idx, n, long = plan.split_rows(self.tile_min) if self.tuned else (None, rows, [])
        b = a if idx is None else args(idx)
        tiles = plan.memo(("tiles", self.tile_min), lambda: self._tiles(plan, long, rows, table)) if long else None
        if s.prepared:
            q = eng.scratch_view("q", rows, s.heads * s.dkp)
            cols = (col["q"], col["k"], col["k" if s.tied_values else "v"])
            rot = eng.rotation(s.rot) + (s.rot.dims,) if s.rot is not None else None
            how = (q, self.NORMS[s.qk_norm], self.qk, rot, eng.cfg.norm_eps)
            if n:
                A.prep(b, n, inp, cols, *how, values=True, pool=bool(s.pool) and plan.singles)
            if long:
                A.prep(a, tiles.shape[0], inp, cols, *how, tiles=tiles)
                A.append_tiles(a, tiles, inp, -1, cols[2])
        else:
            q = inp[:, col["q"]:]
            if s.kv_from is None and n:
                A.append(b, n, inp, col["k"], col["v"])
            if s.kv_from is None and long:
                A.append_tiles(a, tiles, inp, col["k"], col["v"])
        if s.pool and not (s.prepared and plan.singles):
            done, m = plan.finishing(s.pool)
            if m:
                A.pool(a if done is None else args(done), inp.dtype, m)
        if long:
            A.tiles(a, tiles, q, gate, ao, plan.longest)
        if n and self.tuned:
            A.rows(b, n, q, gate, ao, self.key_splits(eng, n, plan.longest), eng.part_o, eng.part_ml)
        elif n:
            A.plain(b, n, q, gate, ao, singles=plan.singles)
        return ao

    @staticmethod
    def _tiles(plan, long: list, rows: int, table) -> torch.Tensor:
        """Query tiles [row0, rows, slot, pos0] of the long runs, the ones with most keys first."""
        from ..ops import paged_attn as A
        t = [(r0 + c, min(A.TILE_ROWS, n - c), slot, p0 + c) for r0, n, slot, p0 in long for c in range(0, n, A.TILE_ROWS)]
        t.sort(key=lambda x: -x[3])
        host = torch.tensor(t, dtype=torch.int32)
        A.check_tiles(host, rows, *table.shape)
        from ..ops import hip
        return hip.to_device(host, plan.eng.device)

    def key_splits(self, eng, entries: int, longest: int) -> int:
        """Splits of a row's keys: about one workgroup per CU, four pages each at least, at most 16 (the merge
        reads one partial sum per split)."""
        from ..ops import hip
        from ..ops import paged_attn as A
        s = self.spec
        seen = longest if not s.window else min(longest, s.window + 64 + -(-s.keep_first // 64) * 64)
        seen += -(-longest // s.pool) if s.pool else 0
        want = hip.N_CU // max(1, entries * A.head_tiles(s))
        cap = eng.part_o.numel() // max(1, entries * s.heads * s.dvp)
        return int(max(1, min(16, want, cap, -(-seen // (4 * A.PAGE)))))

    # ------------------------------------------------------------------ CPU
    def forward_torch(self, eng, x, cache: tuple, state, slot, pos) -> torch.Tensor:
        """The same mixer on a CPU engine; cache (keys [pages, 64, kv_heads, dim], values [.., vdim], and those of the
        pooled blocks)."""
        s, w = self.spec, {k: v.float() for k, v in self.raw.items()}
        keys, values = cache[:2]
        n, dt, table = x.shape[0], eng.dtype, eng.pool.table

        def proj(name):
            return F.linear(x, w[name], w[name + ".b"] if s.bias else None)

        def ready(y, name, heads):  # normed and turned
            def rms(u, g):
                return u * torch.rsqrt(u.pow(2).mean(-1, keepdim=True) + eng.cfg.norm_eps) * g
            if s.qk_norm == WHOLE:
                y = rms(y, w[name + ".norm"])
            y = y.view(n, heads, s.dim)
            if s.qk_norm == HEAD:
                y = rms(y, w[name + ".norm"])
            return y if s.rot is None else turned(eng, s.rot, y, pos)

        def seen(kv, tab, i, at):
            pg = tab[slot[i], at // 64].long()
            return [c[pg, at % 64].float() for c in kv]       # [seen, kv_heads, .]
        if s.kv_from is None:
            page, k = table[slot, pos // 64].long(), proj("k")
            keys[page, pos % 64] = ready(k, "k", s.kv_heads).to(dt)
            values[page, pos % 64] = (k if s.tied_values else proj("v")).view(n, s.kv_heads, s.vdim).to(dt)
        if s.pool:
            ptable = eng.pools[s.pool].table
            for i in range(n):
                if (int(pos[i]) + 1) % s.pool == 0:
                    b = int(pos[i]) // s.pool
                    for c, x8 in zip(cache[2:], seen(cache[:2], table, i, torch.arange(b * s.pool, (b + 1) * s.pool))):
                        c[ptable[slot[i], b // 64].long(), b % 64] = x8.mean(0).to(dt)
        q = ready(proj("q"), "q", s.heads).view(n, s.kv_heads, s.group, s.dim)
        o = torch.empty(n, s.heads, s.vdim)
        for i in range(n):
            p = int(pos[i])
            at = torch.arange(p + 1)
            if s.window:
                at = at[(p - at < s.window) | (at < s.keep_first)]
            k, v = seen((keys, values), table, i, at)
            if s.pool and p >= s.window:
                pk, pv = seen(cache[2:], eng.pools[s.pool].table, i, torch.arange((p - s.window + 1) // s.pool))
                k, v = torch.cat([pk, k]), torch.cat([pv, v])
            sc = torch.einsum("ghd,ngd->ghn", q[i], k) * (self.hscale * s.temperature(p)).view(s.kv_heads, s.group, 1)
            if s.softcap:
                sc = s.softcap * torch.tanh(sc / s.softcap)
            if s.sigmoid:
                r1, r2, b = self.sig.view(3, s.kv_heads, s.group, 1)
                weight = torch.sigmoid(sc - r1 * torch.log1p(r2 * (p - at)) + b)
            elif s.sink:
                top = sc.amax(-1, keepdim=True).clamp(min=0)
                e = torch.exp(sc - top)
                weight = e / (torch.exp(-top) + e.sum(-1, keepdim=True))
            else:
                weight = torch.softmax(sc, -1)
            o[i] = torch.einsum("ghn,ngv->ghv", weight, v).reshape(s.heads, s.vdim)
        if s.head_gate:
            o = o * torch.sigmoid(F.linear(x, w["g"]))[..., None]
        o = o.reshape(n, -1)
        if s.elem_gate:
            o = o * torch.sigmoid(F.linear(x, w["g"]))
        return F.linear(o * self.oscale, w["o"], self.out_bias)


__all__ = ["Attention", "rotary_tables", "turned"]

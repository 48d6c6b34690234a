"""Dumizen on the HIP path: every kernel alone against the plain equations (tests/plain_dumizen.py), then the
engine: whole prompts, portions, decoding, mixed batches, reused pages and slots, generation through the
server's scheduler and captured decode graphs. fp32 engines are held to rounding; bf16 ones to what bf16
products leave."""
import dataclasses
import json
import math
import os
import subprocess
import sys

import pytest
import torch

import dumizen_models as M
import plain_dumizen as P
from llm_sharding_amd.models import dumizen as D
from llm_sharding_amd.models.stack import HEAD, WHOLE, AttentionSpec, MoeSpec, RetentionSpec, RotarySpec
from llm_sharding_amd.parallel.server import PipelineServer

pytestmark = pytest.mark.gpu
DEV = "cuda"
ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
BF, F32, F64 = torch.bfloat16, torch.float32, torch.float64
TOL = {BF: 3e-2, F32: 2e-5}   # engines
SHARP_TOL = 1e-4              # fp32 engines whose softmaxes pick single keys


def _gen(seed=0):
    return torch.Generator().manual_seed(seed)


def _rand(*shape, seed=0, scale=1.0, dtype=BF):
    return (torch.randn(*shape, generator=_gen(seed)) * scale).to(dtype)


def _ids(n, vocab=150, seed=0):
    return torch.randint(0, vocab, (n,), generator=_gen(seed)).tolist()


def close(got, want, tol, what=""):
    got, want = got.double().cpu(), want.double().cpu()
    assert torch.isfinite(got).all(), what
    err = float((got - want).norm() / (want.norm() + 1e-30))
    assert err < tol, f"{what}: rel err {err:.2e} (allowed {tol:.0e})"


def plain_rot(r):
    out = {"base": r.base, "dims": r.dims}
    if r.factor:
        out["scaling"] = {"factor": r.factor, "original": r.original, "fast": r.fast, "slow": r.slow}
    return out




def rows_close(got, want, tol, what=""):
    """As :func:`close` for every row by itself: a few wrong rows do not drown among right ones."""
    got, want = got.double().cpu().flatten(1), want.double().cpu().flatten(1)
    assert torch.isfinite(got).all(), what
    err = (got - want).norm(dim=1) / (want.norm(dim=1) + 1e-30)
    assert float(err.max()) < tol, f"{what}: row {int(err.argmax())} rel err {float(err.max()):.2e} (allowed {tol:.0e})"


# ------------------------------------------------------------------------------ projections and stream
@pytest.mark.parametrize("dtype", [BF, F32])
@pytest.mark.parametrize("rows", [1, 40, 128, 129, 300])
def test_projection_with_squared_relu(dtype, rows):
    from llm_sharding_amd.ops import hip
    from llm_sharding_amd.ops import stream as L
    N, K, at, col32 = 330, 200, 112, 256
    w, x, b = _rand(N, K, seed=N, scale=K ** -0.5), _rand(rows, K, seed=K), _rand(N, seed=1, dtype=F32)
    lin = L.Linear(w.to(DEV, dtype))
    xp = torch.zeros(rows, lin.k, dtype=dtype, device=DEV)
    xp[:, :K] = x.to(DEV, dtype)
    bias = torch.zeros(lin.n, device=DEV)
    bias[:N] = b.to(DEV)
    out = torch.full((rows, col32), 7.0, dtype=dtype, device=DEV)
    out32 = torch.full((rows, lin.n - col32), 7.0, device=DEV)
    lin(xp, rows, out, bias=bias, out32=out32, col32=col32, act_from=at, act=hip.ACT_RELU2)
    y = x.double() @ w.double().T + b.double()
    close(out, torch.cat([y[:, :at], P.relu2(y[:, at:col32])], 1), 5e-3 if dtype == BF else 1e-6, "engine's type")
    close(out32[:, :N - col32], y[:, col32:], 1e-5, "fp32 part")


@pytest.mark.parametrize("dtype", [BF, F32])
@pytest.mark.parametrize("W", [88, 250, 4096, 9001])
@pytest.mark.parametrize("rows", [5, 300])
def test_renorm(dtype, W, rows):
    from llm_sharding_amd.ops import stream as L
    top = 3
    x, y, ye = _rand(rows, W, seed=0, dtype=F32), _rand(rows, W, seed=1, dtype=F32), _rand(rows * top, W, seed=6)
    weight, place = torch.rand(rows * top, generator=_gen(7)), torch.randperm(rows * top, generator=_gen(8)).to(torch.int32)
    post, gain = _rand(W, seed=9, dtype=F32), _rand(W, seed=10, dtype=F32)
    mix = (ye.double()[place.long()] * weight.double()[:, None]).view(rows, top, W).sum(1)
    d = {k: v.to(DEV) for k, v in dict(x=x, y=y, weight=weight, place=place, post=post, gain=gain).items()}
    ex = (ye.to(DEV, dtype), d["weight"], d["place"], top)
    for y_, e_ in ((True, False), (False, True), (True, True)):
        v = (y.double() if y_ else 0) + (mix if e_ else 0)
        for post_ in (True, False):
            for add in (True, False):
                want = (x.double() if add else 0) + (P.norm(v, post.double(), 0.3) if post_ else v)
                for gain_ in (True, False, None):
                    got, out = d["x"].clone(), torch.zeros(rows, W, dtype=dtype, device=DEV)
                    L.stream_renorm(got, rows, y=d["y"] if y_ else None, experts=ex if e_ else None, eps=0.3, add=add,
                                    post=d["post"] if post_ else None, gain=d["gain"] if gain_ else None,
                                    out=None if gain_ is None else out)
                    close(got, want, 1e-6, "stream")
                    if gain_ is not None:
                        close(out, P.norm(want, gain.double(), 0.3) if gain_ else want, 5e-3 if dtype == BF else 1e-6, "copy")


# ------------------------------------------------------------------------------ attention
ROT = RotarySpec(300.0, 32, 2.0, 60, 6.0, 0.6)
SPECS = {
    # windows over pooled blocks: of sizes that do and do not divide a page, of one token, longer than a page
    "pool8": AttentionSpec(6, 3, 36, 24, 0.3, window=37, pool=8, qk_norm=HEAD, rot=ROT),
    "pool12": AttentionSpec(4, 4, 128, 128, 0.1, window=64, pool=12, qk_norm=HEAD, rot=RotarySpec(1e4, 128)),
    "pool1": AttentionSpec(5, 1, 64, 100, 0.2, window=9, pool=1, qk_norm=HEAD, rot=RotarySpec(1e4, 22)),
    "pool70": AttentionSpec(40, 2, 100, 128, 0.1, window=30, pool=70, qk_norm=HEAD, rot=RotarySpec(50.0, 64)),
    "pool_wide": AttentionSpec(2, 1, 300, 30, 0.1, window=65, pool=5, qk_norm=HEAD, rot=RotarySpec(1e4, 300)),
    "pool_bare": AttentionSpec(4, 2, 48, 48, 0.2, window=20, pool=3),
    # a sink, an element-wise gate, values that are the keys
    "sink": AttentionSpec(4, 2, 36, 36, 0.2, qk_norm=WHOLE, rot=RotarySpec(300.0, 36, 4.0, 100, 32.0, 1.0), sink=True,
                          elem_gate=True, tied_values=True),
    "sink_wide": AttentionSpec(24, 3, 128, 128, 0.1, qk_norm=WHOLE, rot=RotarySpec(1e4, 64), sink=True, elem_gate=True,
                               tied_values=True),
    "sink_one": AttentionSpec(3, 1, 200, 200, 0.1, qk_norm=WHOLE, rot=RotarySpec(1e4, 6), sink=True, elem_gate=True,
                              tied_values=True),
    # sigmoids
    "sigmoid": AttentionSpec(6, 2, 24, 40, 0.3, softcap=6.0, sigmoid=True, distance_bias=True, temp_coef=0.4, temp_every=7),
    "sigmoid_wide": AttentionSpec(34, 2, 128, 128, 0.1, softcap=30.0, sigmoid=True, distance_bias=True, temp_coef=0.1,
                                  temp_every=64),
    "sigmoid_bare": AttentionSpec(3, 3, 64, 256, 0.2, sigmoid=True),
    "sigmoid_plain": AttentionSpec(2, 2, 30, 270, 0.2, softcap=2.0, sigmoid=True, distance_bias=True),
}


class Case:
    """Projections of a few sequences on interleaved pages; whatever is not written is loud."""

    def __init__(self, s, lens, dtype, seed=0, eps=1e-5):
        from llm_sharding_amd.ops import paged_attn as A
        from llm_sharding_amd.runtime.attn_mixer import rotary_tables
        from llm_sharding_amd.runtime.latent_mixer import _head_pad
        self.s, self.lens, self.dtype, self.eps = s, lens, dtype, eps
        H, G = s.heads, s.kv_heads
        self.q = [_rand(n, H, s.dim, seed=seed + i, dtype=BF) for i, n in enumerate(lens)]
        self.k = [_rand(n, G, s.dim, seed=seed + 20 + i, dtype=BF) for i, n in enumerate(lens)]
        self.v = [self.k[i] if s.tied_values else _rand(n, G, s.vdim, seed=seed + 40 + i, dtype=BF) for i, n in enumerate(lens)]
        self.gate = [_rand(n, H, s.vdim if s.elem_gate else 1, seed=seed + 60 + i, dtype=BF) for i, n in enumerate(lens)]
        nq, nk = (s.dim * H, s.dim * G) if s.qk_norm == WHOLE else (s.dim, s.dim)
        self.wq, self.wk = torch.rand(nq, generator=_gen(seed + 1)) + 0.5, torch.rand(nk, generator=_gen(seed + 2)) + 0.5
        self.sig = torch.stack([torch.rand(H, generator=_gen(3)), torch.rand(H, generator=_gen(4)) * 0.5,
                                torch.randn(H, generator=_gen(5)) - 1])
        if not s.distance_bias:
            self.sig[:2] = 0
        pages, self.max_pages = sum(-(-n // 64) for n in lens), max(-(-n // 64) for n in lens) + 1

        def table(size, per, pages):
            order, t = torch.randperm(pages, generator=_gen(seed)).tolist(), torch.full((len(lens), size), -1, dtype=torch.int32)
            for i, n in enumerate(lens):
                for b in range(-(-n // per)):
                    t[i, b] = order.pop()
            return t.to(DEV)
        self.table = table(self.max_pages, 64, pages)
        self.cache, self.ptable = tuple(torch.full(x, 30.0, dtype=dtype, device=DEV) for x in A.cache_shapes(s, pages)), None
        if s.pool:
            pp = A.pooled_pages(pages, len(lens), s.pool)
            self.ptable = table(-(-self.max_pages * 64 // (64 * s.pool)) + 1, 64 * s.pool, pp)
            self.cache += tuple(torch.full(x, 30.0, dtype=dtype, device=DEV) for x in A.cache_shapes(s, pp))
        self.hscale = torch.full((H,), s.scale, device=DEV)
        self.oscale = 0.7
        self.sig_d = self.sig.to(DEV).contiguous() if s.sigmoid else None
        self.rot = rotary_tables(s.rot, self.max_pages * 64, DEV) + (s.rot.dims,) if s.rot else None
        self.norm = {None: 0, HEAD: 1, WHOLE: 2}[s.qk_norm]
        self.weights = tuple(_head_pad(w[:, None], n if s.qk_norm == WHOLE else 1, [(s.dim, s.dkp)]).flatten().contiguous().to(DEV)
                             for w, n in ((self.wq, H), (self.wk, G))) if self.norm else None
        self.at = [0] * len(lens)
        self.cols = (0, H * s.dkp, H * s.dkp + G * s.dkp, H * s.dkp + G * (s.dkp + s.dvp))

    def ready(self, i):
        """Queries and keys of a sequence as scored, float64."""
        s, n = self.s, self.lens[i]
        q, k = self.q[i].double(), self.k[i].double()
        if s.qk_norm == WHOLE:
            q = P.norm(q.flatten(1), self.wq.double(), self.eps).view_as(q)
            k = P.norm(k.flatten(1), self.wk.double(), self.eps).view_as(k)
        elif s.qk_norm == HEAD:
            q, k = P.norm(q, self.wq.double(), self.eps), P.norm(k, self.wk.double(), self.eps)
        if s.rot is not None:
            q, k = P.rotate(q, plain_rot(s.rot)), P.rotate(k, plain_rot(s.rot))
        if s.temp_coef:
            q = q * P.temperature(n, s.temp_coef, s.temp_every)[:, None, None]
        return q, k

    def want(self, i):
        s, n = self.s, self.lens[i]
        (q, k), v = self.ready(i), self.v[i].double()
        see = P.window(n, s.window or n)
        if s.pool:
            see = torch.cat([see, P.blocks_seen(n, s.window, s.pool)], 1)
            k, v = torch.cat([k, P.pooled(k, s.pool)]), torch.cat([v, P.pooled(v, s.pool)])
        out = torch.empty(n, s.heads, s.vdim, dtype=F64)
        for h in range(s.heads):
            g = h // s.group
            sc = q[:, h] @ k[:, g].T * s.scale
            if s.softcap:
                sc = P.capped(sc, s.softcap)
            if s.sigmoid:
                r1, r2, b = self.sig.double()[:, h]
                out[:, h] = torch.where(see, torch.sigmoid(sc - P.distance_bias(n, r1, r2) + b), torch.zeros_like(sc)) @ v[:, g]
            else:
                sc = sc.masked_fill(~see, -math.inf)
                out[:, h] = (P.sink_softmax(sc) if s.sink else torch.softmax(sc, -1)) @ v[:, g]
        if s.elem_gate:
            out = out * torch.sigmoid(self.gate[i].double())
        return out * self.oscale

    def step(self, parts, ns=1):
        """One batch over the next rows of some sequences, [(sequence, rows)], as the mixer launches it -> outputs
        by sequence."""
        from llm_sharding_amd.ops import paged_attn as A
        from llm_sharding_amd.runtime.attn_mixer import Attention
        from llm_sharding_amd.runtime.plan import Plan
        s, runs, at = self.s, [], []
        for i, n in parts:
            runs.append((len(at), n, i, self.at[i]))
            at += [(i, self.at[i] + t) for t in range(n)]
            self.at[i] += n
        rows = len(at)

        def pad(ts, n):
            x = torch.stack([ts[i][p] for i, p in at])
            return torch.nn.functional.pad(x, (0, n - x.shape[-1])).flatten(1)
        inp = torch.cat([pad(self.q, s.dkp), pad(self.k, s.dkp), pad(self.v, s.dvp),
                         pad(self.gate, s.dvp if s.elem_gate else 8)], 1).to(DEV, self.dtype)
        inp = torch.nn.functional.pad(inp, (0, -inp.shape[1] % 8))
        slot, pos = (torch.tensor(x, dtype=torch.int32, device=DEV) for x in zip(*at))

        class Eng:
            device = DEV
        plan = Plan(Eng, rows, runs)

        def args(index=None):
            return A.make_args(s, self.cache, self.table, slot, pos, self.hscale, index=index, ptable=self.ptable,
                               sig=self.sig_d, oscale=self.oscale)
        tuned = self.dtype == BF and A.tuned_size(s)
        idx, n, long = plan.split_rows(16) if tuned else (None, rows, [])
        tiles = Attention._tiles(plan, long, rows, self.table) if long else None
        oq, ok, ov, og = self.cols
        ov = ok if s.tied_values else ov
        out, q = torch.full((rows, s.heads * s.dvp), 9.0, dtype=self.dtype, device=DEV), inp[:, oq:]
        if s.prepared:
            q = torch.full((rows, s.heads * s.dkp), 9.0, dtype=self.dtype, device=DEV)
            how = (q, self.norm, self.weights, self.rot, self.eps)
            if n:
                A.prep(args(idx), n, inp, (oq, ok, ov), *how, values=True, pool=bool(s.pool) and plan.singles)
            if long:
                A.prep(args(), tiles.shape[0], inp, (oq, ok, ov), *how, tiles=tiles)
                A.append_tiles(args(), tiles, inp, -1, ov)
        else:
            if n:
                A.append(args(idx), n, inp, ok, ov)
            if long:
                A.append_tiles(args(), tiles, inp, ok, ov)
        if s.pool and not (s.prepared and plan.singles):
            done, m = plan.finishing(s.pool)
            if m:
                A.pool(args(done), self.dtype, m)
        gate = inp[:, og:] if s.elem_gate else None
        po, pm = torch.empty(rows * ns * s.heads * s.dvp, device=DEV), torch.empty(rows * ns * s.heads * 2, device=DEV)
        if long:
            A.tiles(args(), tiles, q, gate, out)
        if n and tuned:
            A.rows(args(idx), n, q, gate, out, ns, po, pm)
        elif n:
            A.plain(args(idx), n, q, gate, out)
        out = out.view(rows, s.heads, s.dvp)[..., :s.vdim].cpu()
        got = {}
        for (i, p), o in zip(at, out):
            got.setdefault(i, []).append(o)
        return {i: torch.stack(o) for i, o in got.items()}


@pytest.mark.parametrize("dtype", [BF, F32])
@pytest.mark.parametrize("name", list(SPECS))
def test_attention(name, dtype):
    """Two sequences in long and short portions and single rows, in several key splits, all over one cache; and the
    cache itself."""
    s = SPECS[name]
    case = Case(s, [330, 150], dtype)
    got = {0: [], 1: []}
    for parts, ns in (([(0, 1), (1, 2)], 1), ([(0, 93), (1, 60)], 1), ([(1, 1), (0, 1)], 3), ([(0, 6), (1, 2)], 2),
                      ([(1, 1), (0, 129)], 2)) + tuple(([(0, 1), (1, 1)], 1 + i % 3) for i in range(30)) \
            + (([(0, 70), (1, 54)], 1),):
        for i, o in case.step(parts, ns).items():
            got[i].append(o)
    assert case.at == [330, 150]
    for i in (0, 1):
        rows_close(torch.cat(got[i]), case.want(i), 1.5e-2 if dtype == BF else 1e-5, f"{name}: {i}")
    from llm_sharding_amd.ops import paged_attn as A
    order, tol = A.value_order(), 6e-3 if dtype == BF else 1e-6
    for i, n in enumerate(case.lens):
        (_, k), v = case.ready(i), case.v[i].double()
        kinds = [(0, case.table, k, v)] + ([(2, case.ptable, P.pooled(k, s.pool), P.pooled(v, s.pool))] if s.pool else [])
        for c, table, kk, vv in kinds:
            for b in range(-(-len(kk) // 64)):
                m, pg = min(64, len(kk) - b * 64), int(table[i, b])
                ck, cv = (t[pg].cpu() for t in case.cache[c:c + 2])
                close(ck[:, :m, :s.dim], kk[b * 64:b * 64 + m].transpose(0, 1), tol, f"{name}: keys")
                close(cv[:, :s.vdim, order[:m]], vv[b * 64:b * 64 + m].permute(1, 2, 0), tol, f"{name}: values")
                assert bool((ck[:, m:] == 30).all()) and bool((cv[..., order[m:]] == 30).all()), "behind the last one"


@pytest.mark.parametrize("dim", [64, 128, 256])
@pytest.mark.parametrize("vdim", [64, 128, 256])
def test_every_tuned_size(dim, vdim):
    """All kernels of query tiles and of single rows, row by row: portions that end inside a tile, at its end and
    behind it."""
    kinds = [dict(sigmoid=True, softcap=5.0, distance_bias=True), dict(sigmoid=True), dict(window=50, pool=6), dict(softcap=9.0)]
    if dim == vdim:
        kinds.append(dict(sink=True, elem_gate=True, tied_values=True))
    for kw in kinds:
        s = AttentionSpec(6, 2, dim, vdim, dim ** -0.5, **kw)
        case, got = Case(s, [230, 35], BF, seed=dim + vdim), {0: [], 1: []}
        for parts in ([(0, 64), (1, 35)], [(0, 150)], [(0, 1)], [(0, 15)]):
            for i, o in case.step(parts, 2).items():
                got[i].append(o)
        for i in (0, 1):
            rows_close(torch.cat(got[i]), case.want(i), 1.5e-2, f"{dim} {vdim} {kw}: {i}")


@pytest.mark.parametrize("dtype", [BF, F32])
@pytest.mark.parametrize("window,pool", [(40, 8), (64, 16), (1, 5), (100, 64), (65, 70), (30, 1)])
def test_a_token_leaves_the_window_and_comes_back_in_its_block(dtype, window, pool):
    """A key that outweighs all others: rows that see it return its value, rows that see its block the block's, rows
    between (behind the window, its block not yet seen) neither."""
    s = AttentionSpec(4, 2, 64, 64, 1.0, window=window, pool=pool)
    n = 400
    for far in sorted({0, 1, pool - 1, pool, 62, 63, 64, 65, 127, 128, 191}):
        case = Case(s, [n], dtype, seed=far)
        case.oscale = 1.0
        case.q[0][:] = 1.0
        case.k[0][:] *= 0.01
        case.k[0][far] = 0.3 * pool  # its block's mean outweighs the rest too
        case.step([(0, 300)])
        block_end = far // pool * pool + pool - 1
        single = {}
        for p in range(300, n):
            single[p] = case.step([(0, 1)])[0][0]
        want = case.want(0)
        edges = sorted({x for e in (far, far + window - 1, far + window, block_end + window - 1, block_end + window,
                                    block_end + window + 1) for x in (e, e + 63) if far <= x < n} | {299, 300, n - 1})
        again = Case(s, [n], dtype, seed=far)
        again.oscale, again.q, again.k, again.v = 1.0, case.q, case.k, case.v
        whole = again.step([(0, n)])[0]
        mean = case.v[0].double()[block_end + 1 - pool:block_end + 1].mean(0)
        for p in edges:
            outs = [whole[p]] + ([single[p]] if p in single else [])
            for o in outs:
                close(o, want[p], 2e-2 if dtype == BF else 1e-5, f"far {far} row {p}")
                alone = float((o.double() - case.v[0][far].double().repeat_interleave(2, 0)).norm())
                block = float((o.double() - mean.repeat_interleave(2, 0)).norm())
                assert (alone < 0.3) == (p - far < window or (pool == 1 and block_end <= p - window)), (far, p, alone)
                if pool > 1:
                    assert (block < 0.3) == (block_end <= p - window), (far, p, block)


def test_first_tokens_and_the_sink():
    """One token: a softmax returns its value whatever the score, with a sink its share of it; a sigmoid its weight."""
    for score in (-8.0, 0.0, 5.0):
        for name in ("sink", "sigmoid", "pool8"):
            s = dataclasses.replace(SPECS[name], rot=None, qk_norm=None, window=0 if name != "pool8" else 37, distance_bias=False)
            if name == "sink":
                s = dataclasses.replace(s, elem_gate=False)
            case = Case(s, [3], F32)
            case.oscale = 1.0
            case.q[0][:] = score / s.scale / s.dim
            case.k[0][:] = 1.0
            o = case.step([(0, 1)])[0][0]
            v = case.v[0][0].repeat_interleave(s.group, 0)
            x = torch.tensor(score, dtype=F64)
            t = (case.q[0][0, 0].double() @ case.k[0][0, 0].double()) * s.scale
            if name == "sink":
                w = torch.exp(t) / (1 + torch.exp(t)) * torch.ones(s.heads, dtype=F64)
            elif name == "sigmoid":
                w = torch.sigmoid(P.capped(t * P.temperature(1, s.temp_coef, s.temp_every)[0], s.softcap) + case.sig[2].double())
            else:
                w = torch.ones(s.heads, dtype=F64)
            close(o, v.double() * w[:, None], 1e-5, f"{name} {float(x)}")


def test_idle_rows_write_nothing():
    from llm_sharding_amd.ops import paged_attn as A
    s = SPECS["pool8"]
    case = Case(s, [8], BF)
    case.table[:] = -1
    before = [c.clone() for c in case.cache]
    out = case.step([(0, 1)])[0]
    assert not out.any() and all(torch.equal(a, b) for a, b in zip(before, case.cache))
    with pytest.raises(ValueError):
        A.make_args(s, case.cache, case.table, torch.zeros(1, dtype=torch.int32, device=DEV),
                    torch.zeros(1, dtype=torch.int32, device=DEV), case.hscale)  # no table of the blocks


# ------------------------------------------------------------------------------ retention
RET = {
    "square": RetentionSpec(4, 128, 128, (0.9, 0.99, 0.999, 0.9999), 128 ** -0.5, RotarySpec(1e4, 128)),
    "small": RetentionSpec(3, 20, 24, (0.5, 0.97, 1.0), 0.3, RotarySpec(100.0, 20)),
    "part": RetentionSpec(2, 64, 48, (0.95, 0.02), 0.125, RotarySpec(1e4, 32)),
    "wide_keys": RetentionSpec(1, 100, 32, (0.995,), 0.1, RotarySpec(1e4, 96)),
    "wide_values": RetentionSpec(2, 32, 70, (0.9, 0.998), 0.2, None),
    "one": RetentionSpec(1, 2, 1, (0.8,), 1.0, RotarySpec(1e4, 2)),
    "plain": RetentionSpec(2, 40, 200, (0.9, 0.999), 0.15, RotarySpec(1e4, 40)),
}


class RetCase:
    def __init__(self, s, lens, dtype, seed=0):
        from llm_sharding_amd.runtime.attn_mixer import rotary_tables
        self.s, self.dtype, self.lens = s, dtype, lens
        H = s.heads
        self.x = {c: [_rand(n, H, d, seed=seed + 10 * j + i) for i, n in enumerate(lens)]
                  for j, (c, d) in enumerate((("q", s.dim), ("k", s.dim), ("v", s.vdim), ("g", s.vdim)))}
        self.state = torch.full((len(lens), H) + s.state_dims, 3.0, device=DEV)  # stale
        self.table = torch.zeros((len(lens), 8), dtype=torch.int32, device=DEV)
        self.rot = rotary_tables(s.rot, 512, DEV) + (s.rot.dims,) if s.rot else None
        self.decay = torch.tensor(s.decay, dtype=F32, device=DEV)
        self.at, self.got = [0] * len(lens), [torch.zeros(n, H, s.vdim) for n in lens]

    def want(self, i):
        s = self.s
        q, k, v, g = (self.x[c][i].double() for c in "qkvg")
        if s.rot is not None:
            q, k = P.rotate(q, plain_rot(s.rot)), P.rotate(k, plain_rot(s.rot))
        out, states = torch.empty_like(v), []
        for h in range(s.heads):
            o, S = P.retain(q[:, h], k[:, h] * s.k_scale, v[:, h], float(self.decay[h].cpu().double()))
            out[:, h] = P.rms(o, 1e-5) * P.silu(g[:, h])
            states.append(S)
        return out * 0.7, torch.stack(states)

    def step(self, parts, how, wide=1):
        from llm_sharding_amd.ops import retention as X
        s, runs, pick = self.s, [], []
        for i, n in parts:
            runs.append((len(pick), n, i, self.at[i]))
            pick += [(i, self.at[i] + t) for t in range(n)]
            self.at[i] += n
        rows, (dk, dv), H = len(pick), s.state_dims, s.heads

        def col(c, n):
            x = torch.stack([self.x[c][i][p] for i, p in pick])
            return torch.nn.functional.pad(x, (0, n - x.shape[-1])).flatten(1)
        inp = torch.cat([torch.zeros(rows, 8, dtype=BF), col("q", dk), col("k", dk), col("v", dv), col("g", dv)], 1)
        inp = torch.nn.functional.pad(inp, (0, -inp.shape[1] % 8)).to(DEV, self.dtype)
        cols = (8, 8 + H * dk, 8 + 2 * H * dk, 8 + 2 * H * dk + H * dv)
        out = torch.zeros(rows, H * dv + -H * dv % 8, dtype=self.dtype, device=DEV)
        X.check_runs(torch.tensor(runs, dtype=torch.int32), rows, len(self.lens))

        def args(**kw):
            return X.make_args(s, self.decay, self.state, inp, cols, out, self.rot, 1e-5, self.table, 8, oscale=0.7, **kw)
        if how == "rows":
            slot, pos = (torch.tensor([r[j] for r in runs], dtype=torch.int32, device=DEV) for j in (2, 3))
            X.steps(args(slot=slot, pos=pos), self.dtype, rows)
        elif how in ("steps", "known"):  # (how long the longest run is decides between kernels)
            X.steps(args(runs=torch.tensor(runs, dtype=torch.int32, device=DEV)), self.dtype, len(runs),
                    max(n for _, n, *_ in runs) if how == "known" else 0)
        else:
            items, entries, longest, several = X.segments(s, runs, wide, least=64)
            ws = torch.full((entries, H, dk, dv), float("nan"), device=DEV)
            o32 = torch.full((rows, H * dv), float("nan"), device=DEV)
            items = items.to(DEV)
            X.chunked(args(runs=items), s, items, longest, several, ws, o32)
        for (i, p), o in zip(pick, out[:, :H * dv].reshape(rows, H, dv)[..., :s.vdim].cpu().float()):
            self.got[i][p] = o


@pytest.mark.parametrize("wide", [1, 1000])
@pytest.mark.parametrize("dtype", [BF, F32])
@pytest.mark.parametrize("name", list(RET))
def test_retention(name, dtype, wide):
    """Two sequences, in step-by-step runs, single rows and (bf16) chunks and segments, all carrying the state on."""
    from llm_sharding_amd.ops import retention as X
    s = RET[name]
    long = "chunks" if dtype == BF and X.chunk_size(s) and name not in ("small", "one") else "steps"
    assert X.chunk_size(s) == (name not in ("plain", "small", "one"))
    case = RetCase(s, [420, 190], dtype)
    case.step([(1, 1), (0, 1)], "rows")
    case.step([(0, 70), (1, 33)], long, wide)
    case.step([(1, 2), (0, 3)], "steps")
    for _ in range(5):
        case.step([(0, 1), (1, 1)], "rows")
    case.step([(1, 149), (0, 300)], long, wide)
    case.step([(0, 1)], "rows")
    case.step([(0, 40)], long, wide)
    assert case.at == [420, 190]
    for i in (0, 1):
        out, S = case.want(i)
        close(case.got[i], out, 6e-3 if dtype == BF else 2e-5, f"{name}: outputs of {i}")
        rows_close(case.got[i], out, 5e-2 if dtype == BF else 1e-2, f"{name}: outputs of {i}")
        close(case.state[i, :, :s.dim, :s.vdim], S, 3e-5, f"{name}: state of {i}")
    rest = case.state.clone()
    rest[:, :, :s.dim, :s.vdim] = 0
    assert not rest.any()


@pytest.mark.parametrize("name,count", [(n, 2) for n in RET] + [("square", 32), ("square", 33), ("part", 130)])
def test_retention_with_several_workgroups_a_head(name, count):
    """Runs around batches of 16 rows, from a start and from a state; as many as the form takes, and one more. The state is that
    of the other form."""
    lens = [12 + 33 + 1 + i % 18 for i in range(count)]
    case, other = RetCase(RET[name], lens, F32), RetCase(RET[name], lens, F32)
    case.step([(i, 12 - i % 3) for i in reversed(range(count))], "known")
    case.step([(i, 33 if i % 2 else 16) for i in range(count)], "known")
    case.step([(i, 1) for i in range(count)], "known")
    case.step([(i, lens[i] - case.at[i]) for i in range(count)], "known")
    other.step([(i, lens[i]) for i in range(count)], "steps")
    for i in range(count):
        close(case.got[i], other.got[i], 2e-5, f"{name} {i}")
    for i in {0, 1, count // 2, count - 1}:
        out, S = case.want(i)
        close(case.got[i], out, 2e-5, f"{name}: outputs of {i}")
        close(case.state[i, :, :RET[name].dim, :RET[name].vdim], S, 3e-5, f"{name}: state of {i}")
    close(case.state, other.state, 1e-5, name)


@pytest.mark.parametrize("name", ["square", "part", "wide_keys"])
def test_retention_with_several_workgroups_a_head_rounds_no_more(name):
    """States and outputs of both forms against float64. A step rounds the state once; where its product with the decay were
    rounded too, the state's errors would be up to 2 ** 0.5 times those of the other form."""
    cases = {how: RetCase(RET[name], [190, 150, 170], F32) for how in ("steps", "known")}
    off = {}
    for how, case in cases.items():
        case.step([(i, n) for i, n in enumerate(case.lens)], how)
        pairs = [(case.got[i], case.state[i, :, :RET[name].dim, :RET[name].vdim].cpu(), *case.want(i)) for i in range(3)]
        off[how] = [sum(float((a.double() - b).norm() / b.norm()) for a, b in p)
                    for p in (((g, o) for g, _, o, _ in pairs), ((s, S) for _, s, _, S in pairs))]
    print(name, off)
    for a, b in zip(off["known"], off["steps"]):
        assert a < 1.1 * b, (name, off)


def test_a_portion_from_the_start_ignores_what_the_slot_held():
    for how, wide in (("steps", 1), ("chunks", 1), ("chunks", 1000), ("rows", 1)):
        case = RetCase(RET["square"], [200], BF)
        case.state.fill_(1e4)
        case.step([(0, 1 if how == "rows" else 200)], how, wide)
        out, _ = case.want(0)
        n = case.at[0]
        close(case.got[0][:n], out[:n], 6e-3, how)


def test_retention_forgets_and_remembers():
    """One loud write: the read-out three hundred rows later shows whether the head keeps it."""
    for wide in (1, 1000):
        s = RetentionSpec(2, 32, 32, (0.9999, 0.5), 1.0, None)
        case = RetCase(s, [330], BF)
        for c in "qk":
            case.x[c][0][:] = 1.0
        case.x["v"][0][:] *= 0.01
        case.x["v"][0][5] = torch.arange(32) - 15.0
        case.x["g"][0][:] = 3.0
        case.step([(0, 330)], "chunks", wide)
        out, _ = case.want(0)
        close(case.got[0], out, 6e-3, "outputs")
        loud = (torch.arange(32) - 15.0) / (torch.arange(32) - 15.0).norm()
        for h, kept in ((0, True), (1, False)):
            o = case.got[0][329, h]
            assert (float(o @ loud / o.norm()) > 0.9) == kept


def test_idle_rows_leave_state_alone():
    from llm_sharding_amd.ops import retention as X
    case = RetCase(RET["small"], [4, 4], BF)
    case.table[1] = -1
    before = case.state.clone()
    case.step([(1, 1)], "rows")
    assert not case.got[1].any() and torch.equal(before, case.state)
    with pytest.raises(ValueError):
        X.check_runs(torch.tensor([[0, 2, 0, 0], [2, 2, 0, 9]]), 4, 2)  # two runs of one slot


# ------------------------------------------------------------------------------ experts
@pytest.mark.parametrize("dtype", [BF, F32])
@pytest.mark.parametrize("rows,experts,top,groups,keep,ff,width", [
    (1, 8, 2, 4, 1, 40, 72), (5, 5, 3, 1, 1, 130, 200), (16, 6, 1, 6, 2, 30, 64), (64, 12, 4, 3, 2, 64, 256),
    (65, 300, 5, 10, 3, 20, 130), (130, 4, 4, 2, 2, 90, 88), (300, 4, 2, 2, 1, 100, 140), (1200, 4, 2, 1, 1, 256, 384)])
def test_experts_by_groups(dtype, rows, experts, top, groups, keep, ff, width):
    """Choices within the best groups, negative choice scores among them, weights without the correction, squared
    relu; few and many pairs per expert."""
    from llm_sharding_amd.ops import moe as X
    s = MoeSpec(experts, top, ff, "relu2", True, True, groups, keep, 1.7)
    up = [_rand(ff, width, seed=e, scale=width ** -0.5) for e in range(experts)]
    down = [_rand(width, ff, seed=e + 300, scale=ff ** -0.5) for e in range(experts)]
    x = X.Experts(None, *([w.to(DEV, dtype) for w in ws] for ws in (up, down)))
    h, logits = _rand(rows, width, seed=4), _rand(rows, experts + 5, seed=5, dtype=F32)
    corr = _rand(experts, seed=6, dtype=F32) * 0.5 - 1.0  # most choice scores are negative
    pairs = rows * top
    hp = torch.zeros(rows, x.width, dtype=dtype, device=DEV)
    hp[:, :width] = h.to(DEV, dtype)
    expert, order, place = torch.full((3, pairs), -7, dtype=torch.int32, device=DEV)
    weight = torch.zeros(pairs, device=DEV)
    tr = X.tile_rows(pairs, experts, dtype == F32)
    tiles = torch.full((X.max_tiles(pairs, experts, tr), 4), -9, dtype=torch.int32, device=DEV)
    corr_d = corr.to(DEV)
    nt = X.route_group(logits.to(DEV), rows, experts, top, tr, expert, weight, order, place, tiles, X.route_args(s, corr_d))
    at, g = P.route(logits[:, :experts].double(), corr.double(), {"top": top, "scale": 1.7,
                                                                 "groups": {"count": groups, "keep": keep}})
    assert torch.equal(expert.cpu().view(rows, top).long(), at)
    close(weight.view(rows, top), g, 1e-6, "weights")
    act, ye = (torch.zeros(pairs, n, dtype=dtype, device=DEV) for n in (x.ff, x.width))
    X.gemm(tiles, nt, tr, order, top, hp, x.up, x.up_n, x.width, act, pairs, x.kind)
    X.gemm(tiles, nt, tr, order, top, act, x.down, x.width, x.ff, ye, pairs, X.DOWN)
    got = (ye.cpu().double()[place.cpu().long()] * weight.cpu().double()[:, None]).view(rows, top, -1).sum(1)
    want = torch.zeros(rows, width, dtype=F64)
    for e in range(experts):
        r, k = (at == e).nonzero(as_tuple=True)
        want.index_add_(0, r, P.expert(h[r].double(), up[e].double(), down[e].double()) * g[r, k, None])
    close(got[:, :width], want, 1e-2 if dtype == BF else 1e-5, "experts")
    assert not got[:, width:].any()


def test_groups_decide_before_experts():
    """The best single expert stays out when its group's two best sum lower."""
    from llm_sharding_amd.ops import moe as X
    s = MoeSpec(6, 2, 8, "relu2", True, False, 3, 1)
    z = torch.tensor([[5.0, -5.0, 1.0, 1.2, -1.0, 0.0]])
    out = [torch.zeros(2, dtype=t, device=DEV) for t in (torch.int32, F32)]
    X.route(z.to(DEV), 1, 6, 2, *out, X.route_args(s))
    assert out[0].tolist() == [3, 2] and P.choose(torch.sigmoid(z), 2, 3, 1).tolist() == [[3, 2]]


# ------------------------------------------------------------------------------ engine
@pytest.fixture(scope="module")
def ordinary():
    """A model and its tensors by compute type."""
    cfg = M.stack()
    return cfg, {F32: M.tensors(cfg), BF: M.decided(cfg)}


@pytest.mark.parametrize("dtype", [BF, F32])
@pytest.mark.parametrize("sizes", [[300], [64, 1, 63, 66, 128], [2, 3, 2], [100, 65, 1, 1, 1], [1]])
def test_portions(ordinary, dtype, sizes):
    cfg, t = ordinary
    ids = _ids(300 if sizes[0] > 3 else 140)
    want = P.run(cfg.to_dict(), t[dtype], ids)
    eng = M.engine(cfg, DEV, dtype, t=t[dtype])
    got = torch.cat([M.feed(eng, [(1, p)]) for p in M.cut(ids, sizes)])
    assert M.rel(got, want) < TOL[dtype]


def test_stream_after_every_layer(ordinary):
    """Stages of one layer run each: the stream between them is the oracle's."""
    cfg, t = ordinary
    ids, trail = _ids(90, seed=7), []
    P.run(cfg.to_dict(), t[F32], ids, trail=trail)
    for end in range(1, cfg.num_hidden_layers + 1):
        eng = M.engine(cfg, DEV, F32, end=end)
        slot, pos = eng.prefill_rows([0], [90])
        h = eng.forward(eng.embed(torch.tensor(ids)), slot, pos)
        close(h, trail[end - 1], 1e-5, f"run {end - 1}")


def test_portions_whose_softmax_picks_single_keys():
    cfg = M.stack(sharp=3.0)
    ids = _ids(330, seed=2)
    want = P.run(cfg.to_dict(), M.tensors(cfg), ids)
    for sizes in ([330], [190, 1, 2, 63], [37, 37, 3]):
        eng = M.engine(cfg, DEV, F32)
        got = torch.cat([M.feed(eng, [(0, p)]) for p in M.cut(ids, sizes)])
        assert M.rel(got, want) < SHARP_TOL, sizes


@pytest.mark.parametrize("dtype", [BF, F32])
def test_long_decoding(ordinary, dtype):
    """A two-token prompt, then 330 single tokens across pages, windows and blocks."""
    cfg, t = ordinary
    ids = _ids(332, seed=5)
    want = P.run(cfg.to_dict(), t[dtype], ids)
    eng = M.engine(cfg, DEV, dtype, t=t[dtype])
    got = [M.feed(eng, [(3, ids[:2])])] + [M.feed(eng, [(3, [x])]) for x in ids[2:]]
    assert M.rel(torch.cat(got), want) < TOL[dtype]


@pytest.mark.parametrize("dtype", [BF, F32])
def test_unequal_batches_on_reused_pages_and_slots(ordinary, dtype):
    cfg, t = ordinary
    eng = M.engine(cfg, DEV, dtype, t=t[dtype], cache_tokens=64 * 10)
    seqs = {k: _ids(n, seed=k) for k, n in ((0, 260), (1, 75), (2, 200), (3, 140), (4, 3))}
    want = {k: P.run(cfg.to_dict(), t[dtype], v) for k, v in seqs.items()}
    slot, at, got = {0: 2, 1: 0, 2: 1, 3: 0, 4: 3}, {k: 0 for k in seqs}, {k: [] for k in seqs}

    def step(parts):
        lg = M.feed(eng, [(slot[k], seqs[k][at[k]:at[k] + n]) for k, n in parts])
        for k, n in parts:
            got[k].append(lg[:n])
            lg, at[k] = lg[n:], at[k] + n

    step([(0, 200), (1, 1)])
    step([(1, 70), (0, 1), (2, 3)])
    step([(0, 1), (2, 130), (1, 1)])
    step([(1, 3), (0, 1), (2, 1)])
    eng.reset([slot[1]])
    step([(0, 57), (2, 66), (4, 1)])
    eng.reset([slot[0], slot[2]])
    step([(3, 65), (4, 2)])
    step([(3, 75)])
    for k in seqs:
        assert at[k] == len(seqs[k]) and M.rel(torch.cat(got[k]), want[k]) < TOL[dtype], k


def test_rows_do_not_depend_on_the_batch(ordinary):
    cfg, _ = ordinary
    ids = _ids(90, seed=8)
    alone = M.engine(cfg, DEV, F32)
    M.feed(alone, [(0, ids[:89])])
    a = M.feed(alone, [(0, ids[89:])])
    other = M.engine(cfg, DEV, F32)
    M.feed(other, [(1, _ids(130, seed=3))])
    M.feed(other, [(3, ids[:50]), (0, _ids(7, seed=1))])
    M.feed(other, [(1, [4]), (3, ids[50:89])])
    b = M.feed(other, [(0, [9]), (1, [8, 7]), (3, ids[89:])])
    assert M.rel(b[-1:], a) < TOL[F32]


def test_other_sizes_and_values_that_often_coincide():
    """Sizes beyond the tuned kernels, ones, one expert, a window of one key, blocks of one token and of more than a
    page, scale 1, decays of 1, a whole model in the loop, a loop of one pass, none."""
    r = D.rot
    for width, loop in ((130, (0, 6, 2)), (144, (2, 3, 1)), (129, None)):
        cfg = D.make_config(width, 129, [
            D.attention_entry(2, 1, 300, 270, 1, 1, r(300), D.moe(1, 1, 1, 1), scale=1.0),
            D.sigmoid_entry(1, 1, 1, 1, None, scale=1.0, softcap=1.0, coef=0.0, every=1),
            D.parallel_entry(D.left_entry(3, 3, 2, r(2)), D.right_entry(1, 2, 1, r(2), [1.0]), D.moe(9, 9, 17, 130, 9, 9, 1.0)),
            D.attention_entry(34, 1, 16, 16, 100, 70, r(10, 50.0, 1.0, 30), D.moe(8, 1, 129, 3, 8, 1)),
            D.parallel_entry(D.left_entry(2, 1, 270, r(8)), D.right_entry(2, 140, 130, r(140), [0.9, 0.99]), None, 2.0, -0.5),
            D.sigmoid_entry(2, 2, 300, 30, D.moe(4, 2, 16, 16, 2, 2, 0.3), softcap=50.0, coef=3.0, every=1000)], loop, eps=0.5)
        t = M.decided(cfg)
        ids = _ids(170, vocab=129)
        want = P.run(cfg.to_dict(), t, ids)
        for dtype, tol in ((F32, SHARP_TOL), (BF, 5e-2)):
            eng = M.engine(cfg, DEV, dtype, t=t)
            got = torch.cat([M.feed(eng, [(0, p)]) for p in M.cut(ids, [120, 1, 49])])
            assert M.rel(got, want) < tol, (width, dtype)


def test_layers_of_a_real_width():
    """Wide heads and states, enough pairs for every expert kernel, portions on every projection kernel."""
    cfg = D.make_config(512, 260, [
        D.attention_entry(16, 4, 128, 128, 200, 16, D.rot(64, 1e4, 2.0, 400), D.moe(2, 1, 256, 384)),
        D.parallel_entry(D.left_entry(16, 4, 128, D.rot(128)), D.right_entry(4, 128, 128, D.rot(128)), D.moe(6, 2, 200, 100, 3, 2)),
        D.sigmoid_entry(16, 4, 128, 128, D.moe(4, 2, 300, 128), coef=0.2, every=100)], (0, 2, 2))
    t = M.decided(cfg)
    ids = _ids(850, vocab=260)
    want = P.run(cfg.to_dict(), t, ids, dtype=F32)
    eng = M.engine(cfg, DEV, BF, t=t, max_seq=1024, max_prefill_rows=1024)
    got = torch.cat([M.feed(eng, [(0, p)]) for p in M.cut(ids, [600, 1, 20, 64, 129, 2, 34])])
    assert M.rel(got, want) < TOL[BF]


# ------------------------------------------------------------------------------ generation
@pytest.mark.parametrize("dtype", [F32, BF])
@pytest.mark.parametrize("graph", [True, False])
def test_greedy_generation_through_the_server(ordinary, dtype, graph):
    """More requests than slots over a small page pool, prompts cut at the prefill budget, decode graphs
    replayed while slots (and their states and blocks) come and go."""
    cfg, t = ordinary
    prompts = [_ids(n, seed=20 + n) for n in (4, 130, 1, 65, 33, 90, 7)]
    t = t[dtype]
    srv = PipelineServer(cfg, M.NamedSource(cfg, t=t), device=DEV, batch=2, microbatches=2, max_seq=192, prefill_budget=100,
                         dtype=dtype, use_graph=graph, cache_tokens=64 * 7)
    outs = srv.generate(prompts, 8, eos_ids=())
    for p, o in zip(prompts, outs):
        want, gaps = P.greedy(cfg.to_dict(), t, p, 8)
        clear = next((i for i, gp in enumerate(gaps) if gp < (0.1 if dtype == BF else 1e-3)), 8)
        assert o[:clear] == want[:clear], (len(p), o, want, gaps)
    assert all(len(p.free) == p.pages for p in (srv.eng.pool, *srv.eng.pools.values()))


def test_concurrent_streams_generate_the_same(ordinary):
    cfg, _ = ordinary
    prompts = [_ids(n, seed=40 + n) for n in (70, 12, 100, 5, 30, 66)]
    outs = []
    for streams in (1, 2):
        srv = PipelineServer(cfg, M.NamedSource(cfg, 0), device=DEV, batch=2, microbatches=2, max_seq=192,
                             prefill_budget=128, dtype=F32, streams=streams)
        outs.append(srv.generate(prompts, 12, eos_ids=()))
    assert outs[0] == outs[1]


@pytest.mark.parametrize("dtype", [F32, BF])
def test_graph_replays_equal_eager_steps(ordinary, dtype):
    """The capture of a graph over live sequences moves no state; replays move it as eager steps do."""
    from llm_sharding_amd.runtime.engine import DecodeGraph
    cfg, t = ordinary
    prompts = [_ids(60, seed=1), _ids(62, seed=2), _ids(3, seed=3)]
    a, b = (M.engine(cfg, DEV, dtype, t=t[dtype]) for _ in range(2))
    for eng in (a, b):
        M.feed(eng, [(i, p) for i, p in enumerate(prompts)])
    g = DecodeGraph(a, 3, "full", history_len=14)
    tok = torch.tensor([5, 6, 7], dtype=torch.int32)
    g.tokens.copy_(tok)
    g.capture()
    for i in range(14):  # crosses page and block borders
        g.replay()
        M.feed(b, [(3, [i + 1])])  # the eager engine's own work in between
        torch.cuda.synchronize()
        slot, pos = b.prefill_rows([0, 1, 2], [1, 1, 1])
        h = b.forward(b.embed(tok), slot, pos)
        b.advance([0, 1, 2], [1, 1, 1])
        assert M.rel(g.out_hidden.cpu(), h.cpu()) < (2e-2 if dtype == BF else 1e-5), i
        lg, tok = b.logits(h).cpu(), b.head(h).to(torch.int32).cpu()
        got = g.history[i].cpu()
        best = lg.max(-1).values - lg.gather(1, got.long()[:, None])[:, 0]
        assert float(best.max()) <= 2e-2 * float(lg.abs().max()), i
        g.tokens.copy_(tok)
    for s, r in zip(a.states, b.states):
        if s is not None:
            close(s[0][:3], r[0][:3], 2e-2 if dtype == BF else 1e-5, "state")


def test_stages_on_one_gpu():
    """Pipeline stages (split head, captured graphs, fp32 stream between them) give the single engine's tokens."""
    from llm_sharding_amd.config import get_preset
    from llm_sharding_amd.parallel.pipeline import drive_local_pipeline, run_pipeline_generate
    cfg = get_preset("tiny-dumizen")
    src = M.NamedSource(cfg, 3)
    prompts = torch.randint(3, cfg.vocab_size, (2, 2, 70), generator=_gen(4))
    kw = dict(batch=2, microbatches=2, max_seq=128, dtype=F32)
    one = run_pipeline_generate(cfg, src, prompts, 6, 0, 1, device=DEV, **kw)
    want, _ = P.greedy(cfg.to_dict(), M.tensors(cfg, 3), prompts[1, 0].tolist(), 6)
    assert one[:, 1, 0].tolist() == want
    for n in (2, 3):
        assert torch.equal(drive_local_pipeline(cfg, src, prompts, 6, n, DEV, **kw), one), n


def test_stage_costs_are_measured(ordinary):
    from llm_sharding_amd.utils.node_profiler import profile_stage_costs
    cfg, _ = ordinary
    r = profile_stage_costs(cfg, M.NamedSource(cfg, 0), DEV, batch=2, context=70, n_layers=3, prefill_len=80, replays=4)
    assert r["layer_decode_ms"] > 0 and r["layer_prefill_ms"] > 0


def test_trace_replay(ordinary, tmp_path):
    cfg, t = ordinary
    folder = D.write_random_checkpoint(cfg, str(tmp_path / "m"), seed=0)
    ids = _ids(70)
    want = P.run(cfg.to_dict(), t[F32], ids)
    steps = [{"step": 0, "entries": [{"id": "a", "tokens": ids[:66], "want": [0, 65]}], "end": []},
             {"step": 1, "entries": [{"id": "b", "tokens": ids[:2], "want": []}, {"id": "a", "tokens": ids[66:67], "want": []}],
              "end": ["b"]},
             {"step": 2, "entries": [{"id": "c", "tokens": ids[:1], "want": [0]}, {"id": "a", "tokens": ids[67:], "want": [2]}],
              "end": ["a", "c"]}]
    r = subprocess.run([sys.executable, os.path.join(ROOT, "bin", "trace_run"), "--model", folder, "--dtype", "float32",
                        "--out", str(tmp_path), "--max-tokens", "200"], input="\n".join(map(json.dumps, steps)),
                       capture_output=True, text=True, timeout=100)
    assert r.returncode == 0, r.stderr[-2000:]
    assert [x for x in r.stdout.splitlines() if x.startswith("done")] == ["done 0", "done 1", "done 2"]

    def read(n):
        return torch.frombuffer(bytearray((tmp_path / f"{n}.f32").read_bytes()), dtype=torch.float32).view(-1, cfg.vocab_size)

    assert not (tmp_path / "1.f32").exists()
    assert M.rel(read(0), want[[0, 65]]) < TOL[F32] and M.rel(read(2), want[[0, 69]]) < TOL[F32]

"""Gupuvik on the HIP path: every kernel alone against the plain equations (tests/plain_gupuvik.py), then the
engine: whole prompts, portions, decoding, mixed batches, reused pages and slots, generation through the
server's scheduler and captured decode graphs. fp32 engines are held to rounding; bf16 ones to what bf16
products leave."""
import json
import os
import subprocess
import sys

import pytest
import torch

import gupuvik_models as M
import plain_gupuvik as P
from llm_sharding_amd.models import gupuvik as G
from llm_sharding_amd.models.stack import AttentionSpec, DeltaSpec
from llm_sharding_amd.parallel.server import PipelineServer

pytestmark = pytest.mark.gpu
DEV = "cuda"
ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
BF, F32, F64 = torch.bfloat16, torch.float32, torch.float64
TOL = {BF: 2e-2, F32: 2e-5}   # engines
SHARP_TOL = 1e-4              # fp32 engines whose softmaxes pick single keys


def _gen(seed=0):
    return torch.Generator().manual_seed(seed)


def _rand(*shape, seed=0, scale=1.0, dtype=BF):
    return (torch.randn(*shape, generator=_gen(seed)) * scale).to(dtype)


def _ids(n, vocab=150, seed=0):
    return torch.randint(0, vocab, (n,), generator=_gen(seed)).tolist()


def off(got, want, dtype):
    return M.rel(got, want) if dtype == F32 else M.rel_most(got, want)


def close(got, want, tol, what=""):
    got, want = got.double().cpu(), want.double().cpu()
    assert torch.isfinite(got).all(), what
    err = float((got - want).norm() / (want.norm() + 1e-30))
    assert err < tol, f"{what}: rel err {err:.2e} (allowed {tol:.0e})"


# ------------------------------------------------------------------------------ projections and stream
@pytest.mark.parametrize("dtype", [BF, F32])
@pytest.mark.parametrize("rows", [1, 16, 17, 40, 128, 129, 300])
def test_one_projection_of_several_parts(dtype, rows):
    """Columns in the engine's type, gelu'd ones, fp32 ones, biases; and products that join a gated stream."""
    from llm_sharding_amd.ops import stream as L
    for N, K, gelu, col32 in ((330, 200, 112, 256), (96, 72, 0, 48)):
        w, x, b = _rand(N, K, seed=N, scale=K ** -0.5), _rand(rows, K, seed=K), _rand(N, seed=1, dtype=F32)
        lin = L.Linear(w.to(DEV, dtype))
        xp = torch.zeros(rows, lin.k, dtype=dtype, device=DEV)
        xp[:, :K] = x.to(DEV, dtype)
        bias = torch.zeros(lin.n, device=DEV)
        bias[:N] = b.to(DEV)
        out = torch.full((rows, col32), 7.0, dtype=dtype, device=DEV)
        out32 = torch.full((rows, lin.n - col32), 7.0, device=DEV)
        lin(xp, rows, out, bias=bias, out32=out32, col32=col32, act_from=gelu)
        y = x.double() @ w.double().T + b.double()
        want = torch.cat([y[:, :gelu], P.gelu(y[:, gelu:col32])], 1)
        close(out, want, 5e-3 if dtype == BF else 1e-6, "engine's type")
        close(out32[:, :N - col32], y[:, col32:], 1e-5, "fp32 part")
        cols = N // 16 * 16
        stream, gate = _rand(rows, cols, seed=3, dtype=F32), _rand(rows, cols + 24, seed=4)
        acc = stream.to(DEV)
        lin(xp, rows, None, out32=acc, gate=gate.to(DEV, dtype), cols=cols)
        close(acc, stream.double() + torch.sigmoid(gate[:, :cols].double()) * (y - b.double())[:, :cols], 1e-5, "gated")


@pytest.mark.parametrize("dtype", [BF, F32])
@pytest.mark.parametrize("W", [88, 250, 4096, 9001])
def test_join(dtype, W):
    from llm_sharding_amd.ops import stream as L
    rows, top = 5, 6
    x, y1, y2 = (_rand(rows, W, seed=i, dtype=F32) for i in range(3))
    g1, g2, ye = _rand(rows, W, seed=4), _rand(rows, W, seed=5), _rand(rows * top, W, seed=6)
    weight = torch.rand(rows * top, generator=_gen(7))
    place = torch.randperm(rows * top, generator=_gen(8)).to(torch.int32)
    gain = _rand(W, seed=9, dtype=F32)
    first = x.double() + torch.sigmoid(g1.double()) * y1.double()
    mix = (ye.double()[place.long()] * weight.double()[:, None]).view(rows, top, W).sum(1)
    dev = {k: v.to(DEV) for k, v in dict(x=x, y1=y1, y2=y2, weight=weight, place=place, gain=gain).items()}
    g1, g2, ye = (t.to(DEV, dtype) for t in (g1, g2, ye))
    for kw, want in ((dict(first=(dev["y1"], g1)), first),
                     (dict(first=(dev["y1"], g1), second=dev["y2"], gate2=g2),
                      first + torch.sigmoid(g2.double().cpu()) * y2.double()),
                     (dict(experts=(ye, dev["weight"], dev["place"], top), gate2=g2),
                      x.double() + torch.sigmoid(g2.double().cpu()) * mix)):
        for normed in (False, True):
            got, out = dev["x"].clone(), torch.zeros(rows, W, dtype=dtype, device=DEV)
            L.stream_join(got, rows, **kw, gain=dev["gain"] if normed else None, eps=0.3, out=out if normed else None)
            close(got, want, 1e-6, "stream")
            if normed:
                close(out, P.rms(want, 0.3) * gain.double(), 5e-3 if dtype == BF else 1e-6, "norm")


# ------------------------------------------------------------------------------ attention
# heads, kv_heads, dim, vdim, scale, softcap, window, keep_first
SIZES = {
    "small": AttentionSpec(6, 3, 20, 24, 0.3, 4.0, 37, 3),
    "one_group": AttentionSpec(5, 1, 64, 64, 0.2, 0.0, 0, 0),
    "many_heads": AttentionSpec(40, 2, 100, 128, 0.1, 20.0, 100, 70),
    "wide_keys": AttentionSpec(4, 4, 200, 40, 0.1, 30.0, 1, 0),
    "wide_values": AttentionSpec(8, 8, 128, 256, 0.1, 30.0, 130, 1),
    "plain_wide": AttentionSpec(2, 1, 300, 30, 0.1, 8.0, 65, 64),
}


class Case:
    """Keys and values of a few sequences on interleaved pages; whatever is not written is loud."""

    def __init__(self, s, lens, dtype, seed=0):
        from llm_sharding_amd.ops import paged_attn as A
        self.s, self.lens, self.dtype = s, lens, dtype
        self.k = [_rand(n, s.kv_heads, s.dim, seed=seed + i, dtype=dtype) for i, n in enumerate(lens)]
        self.v = [_rand(n, s.kv_heads, s.vdim, seed=seed + 20 + i, dtype=dtype) for i, n in enumerate(lens)]
        pages = sum(-(-n // 64) for n in lens)
        self.max_pages = max(-(-n // 64) for n in lens) + 1
        order = torch.randperm(pages, generator=_gen(seed)).tolist()
        self.table = torch.full((len(lens), self.max_pages), -1, dtype=torch.int32)
        for i, n in enumerate(lens):
            for b in range(-(-n // 64)):
                self.table[i, b] = order.pop()
        self.table = self.table.to(DEV)
        self.cache = tuple(torch.full(x, 30.0, dtype=dtype, device=DEV) for x in A.cache_shapes(s, pages))
        self.temp = torch.rand(s.heads, generator=_gen(seed + 5)) + 0.5
        self.hscale = (self.temp * s.scale).to(DEV)

    def args(self, slot, pos, index=None):
        from llm_sharding_amd.ops import paged_attn as A
        self.hold = [torch.tensor(x, dtype=torch.int32, device=DEV) for x in (slot, pos)]
        return A.make_args(self.s, self.cache, self.table, *self.hold, self.hscale, index=index)

    def padded(self, x, n):
        return torch.nn.functional.pad(x, (0, n - x.shape[-1])).flatten(1)

    def fill(self):
        """Appends everything, rows in an order of their own (decoded tokens)."""
        from llm_sharding_amd.ops import paged_attn as A
        s = self.s
        at = [(i, p) for i, n in enumerate(self.lens) for p in range(n)]
        at = [at[j] for j in torch.randperm(len(at), generator=_gen(3)).tolist()]
        rows = torch.cat([torch.cat([self.padded(self.k[i][p:p + 1], s.dkp), self.padded(self.v[i][p:p + 1], s.dvp)], 1)
                          for i, p in at]).to(DEV)
        A.append(self.args(*zip(*at)), len(at), rows, 0, s.kv_heads * s.dkp)
        return self

    def want(self, q, slot, pos, gate=None):
        s, out = self.s, []
        for i in range(len(pos)):
            k, v = self.k[slot[i]][:pos[i] + 1].double(), self.v[slot[i]][:pos[i] + 1].double()
            see = P.visible(pos[i] + 1, s.window or 1 << 30, s.keep_first)[-1]
            k, v = (t[see].repeat_interleave(s.group, 1) for t in (k, v))
            sc = torch.einsum("hd,nhd->hn", q[i].double(), k) * s.scale * self.temp.double()[:, None]
            if s.softcap:
                sc = P.capped(sc, s.softcap)
            out.append(torch.einsum("hn,nhv->hv", torch.softmax(sc, -1), v))
        o = torch.stack(out)
        return o if gate is None else o * torch.sigmoid(gate.double())[..., None]

    def unpad(self, out):
        return out[:, :self.s.heads * self.s.dvp].view(-1, self.s.heads, self.s.dvp)[..., :self.s.vdim]


@pytest.mark.parametrize("dtype", [BF, F32])
@pytest.mark.parametrize("name", list(SIZES))
def test_attention_of_single_rows(name, dtype):
    """Rows of two sequences at page borders, in several splits, by index, and idle ones."""
    from llm_sharding_amd.ops import paged_attn as A
    s = SIZES[name]
    case = Case(s, [200, 130], dtype).fill()
    slot, pos = [0, 0, 1, 0, 1, 0, 0, 1, 0], [0, 1, 129, 63, 64, 65, 199, 127, 128]
    q, gate = _rand(9, s.heads, s.dim, seed=7, dtype=dtype), _rand(9, s.heads, seed=8, dtype=dtype)
    qp, gp = case.padded(q, s.dkp).to(DEV), gate.to(DEV)
    tuned = dtype == BF and A.tuned_size(s)
    assert tuned == (dtype == BF and name != "plain_wide")
    tol = 1.5e-2 if dtype == BF else 3e-6
    po, pm = torch.empty(9 * 7 * s.heads * s.dvp, device=DEV), torch.empty(9 * 7 * s.heads * 2, device=DEV)

    def run(a, n, out, ns, g):
        A.rows(a, n, qp, g, out, ns, po, pm) if tuned else A.plain(a, n, qp, g, out)
        return out
    for ns in (1, 3, 7):
        out = torch.full((9, s.heads * s.dvp), 9.0, dtype=dtype, device=DEV)
        run(case.args(slot, pos), 9, out, ns, gp)
        close(case.unpad(out), case.want(q, slot, pos, gate), tol, f"{name} ns={ns}")
    idx = torch.tensor([8, 2, 5], dtype=torch.int32, device=DEV)
    out = run(case.args(slot, pos, idx), 3, torch.zeros(9, s.heads * s.dvp, dtype=dtype, device=DEV), 2, None)
    close(case.unpad(out)[idx.long()], case.want(q, slot, pos)[idx.cpu().long()], tol, "indexed rows")
    rest = torch.ones(9, dtype=torch.bool)
    rest[idx.cpu().long()] = False
    assert not out.cpu()[rest].any()
    idle = run(case.args([0, 1, 0], [-1, 64 * case.max_pages - 1, 5]), 3, torch.ones(9, s.heads * s.dvp, dtype=dtype, device=DEV), 1, None)
    assert not idle[:2].any() and torch.isfinite(idle[2].float()).all()


@pytest.mark.parametrize("name", [n for n in SIZES if n != "plain_wide"])
def test_attention_of_query_tiles(name):
    """Portions that start at 0, inside a page and inside a tile of 32, appended and attended as tiles."""
    from llm_sharding_amd.ops import paged_attn as A
    from llm_sharding_amd.runtime.attn_mixer import Attention
    s = SIZES[name]
    case = Case(s, [400, 150], BF, seed=2)
    runs = [(0, 307, 0, 93), (307, 150, 1, 0)]
    first = [(0, p) for p in range(93)]
    head = torch.cat([case.padded(case.k[0][:93], s.dkp), case.padded(case.v[0][:93], s.dvp)], 1).to(DEV)
    A.append(case.args(*zip(*first)), 93, head, 0, s.kv_heads * s.dkp)
    slot = [r[2] for r in runs for _ in range(r[1])]
    pos = [r[3] + i for r in runs for i in range(r[1])]
    rows = len(pos)
    q, gate = _rand(rows, s.heads, s.dim, seed=7), _rand(rows, s.heads, seed=8)
    inp = torch.cat([case.padded(q, s.dkp), case.padded(torch.cat([case.k[0][93:], case.k[1]]), s.dkp),
                     case.padded(torch.cat([case.v[0][93:], case.v[1]]), s.dvp)], 1)
    inp = torch.nn.functional.pad(inp, (0, -inp.shape[1] % 8)).to(DEV)
    ok = s.heads * s.dkp

    class Eng:
        device = DEV
    plan = type("Plan", (), {"eng": Eng})
    tiles = Attention._tiles(plan, runs, rows, case.table)
    assert tiles.shape == (5, 4)
    a = case.args(slot, pos)
    A.append_tiles(a, tiles, inp, ok, ok + s.kv_heads * s.dkp)
    order = A.value_order()
    for i, n in enumerate(case.lens):
        for b in range(-(-n // 64)):
            m, pg = min(64, n - b * 64), int(case.table[i, b])
            k, v = (c[pg].cpu() for c in case.cache)
            assert torch.equal(k[:, :m, :s.dim], case.k[i][b * 64:b * 64 + m].transpose(0, 1))
            assert torch.equal(v[:, :s.vdim, order[:m]], case.v[i][b * 64:b * 64 + m].permute(1, 2, 0))
            assert bool((k[:, m:] == 30).all()) and bool((v[..., order[m:]] == 30).all())
    out = torch.zeros(rows, s.heads * s.dvp, dtype=BF, device=DEV)
    A.tiles(a, tiles, inp, gate.to(DEV), out)
    pick = list(range(0, rows, 7)) + [1, rows - 1]
    close(case.unpad(out).cpu()[pick], case.want(q[pick], [slot[i] for i in pick], [pos[i] for i in pick], gate[pick]),
          1.5e-2, name)
    with pytest.raises(ValueError):
        A.check_tiles(torch.tensor([[0, 129, 0, 0]]), 200, 2, 4)
    with pytest.raises(ValueError):
        A.check_tiles(torch.tensor([[0, 10, 0, 250]]), 200, 2, 4)


@pytest.mark.parametrize("rows", [768, 769, 1537])
def test_attention_of_query_tiles_in_two_rows(rows):
    """40 heads: 30, 35 and 65 tiles an XCD, of which 32 have a CU each and the rest the second place. Limit as above."""
    from llm_sharding_amd.ops import paged_attn as A
    from llm_sharding_amd.runtime.attn_mixer import Attention
    s = SIZES["many_heads"]
    case = Case(s, [rows], BF, seed=4).fill()
    q = _rand(rows, s.heads, s.dim, seed=9)
    eng = type("Eng", (), {"device": DEV})
    tiles = Attention._tiles(type("Plan", (), {"eng": eng}), [(0, rows, 0, 0)], rows, case.table)
    out = torch.full((rows, s.heads * s.dvp), float("nan"), dtype=BF, device=DEV)
    A.tiles(case.args([0] * rows, list(range(rows))), tiles, case.padded(q, s.dkp).to(DEV), None, out)
    pick = list(range(5, rows, 61)) + [rows - 1]
    assert not out.isnan().any()
    close(case.unpad(out).cpu()[pick], case.want(q[pick], [0] * len(pick), pick), 1.5e-2, "rows")


@pytest.mark.parametrize("dtype", [BF, F32])
@pytest.mark.parametrize("window,keep", [(40, 5), (64, 0), (1, 64), (100, 1), (65, 130)])
def test_one_key_stands_out(dtype, window, keep):
    """A key that outweighs all others: rows that see it return its value, rows just outside its window do not,
    wherever it lies, unless it is one of the first."""
    from llm_sharding_amd.ops import paged_attn as A
    s = AttentionSpec(6, 2, 48, 56, 1.0, 30.0, window, keep)
    for far in sorted({0, 1, keep - 1, keep, keep + 1, 62, 63, 64, 65, 127, 128} - {-1}):
        case = Case(s, [330], dtype, seed=far)
        case.temp.fill_(1.0)
        case.hscale.fill_(1.0)
        case.k[0][:] *= 0.05
        case.k[0][far] = 5.0 / 48 ** 0.5
        case.fill()
        pos = sorted({p for p in (far, far + window - 1, far + window, far + window + 1, far + 63, 329) if far <= p < 330})
        n = len(pos)
        q = torch.full((n, 6, 48), 5.0 / 48 ** 0.5).to(dtype)
        qp = case.padded(q, s.dkp).to(DEV)
        out = torch.zeros(n, s.heads * s.dvp, dtype=dtype, device=DEV)
        if dtype == F32:
            A.plain(case.args([0] * n, pos), n, qp, None, out)
        else:
            po, pm = torch.empty(n * 3 * 6 * s.dvp, device=DEV), torch.empty(n * 3 * 12, device=DEV)
            A.rows(case.args([0] * n, pos), n, qp, None, out, 3, po, pm)
        got, want = case.unpad(out), case.want(q, [0] * n, pos)
        close(got, want, 1.5e-2 if dtype == BF else 1e-5, f"far={far}")
        outs = [got]
        if dtype == BF:  # the same rows as one-row tiles
            tiles = torch.tensor([[i, 1, 0, p] for i, p in enumerate(pos)], dtype=torch.int32)
            A.check_tiles(tiles, n, *case.table.shape)
            out2 = torch.zeros_like(out)
            A.tiles(case.args([0] * n, pos), tiles.to(DEV), qp, None, out2)
            close(case.unpad(out2), want, 1.5e-2, f"tiles far={far}")
            outs.append(case.unpad(out2))
        alone = case.v[0][far].double().repeat_interleave(3, 0)
        for o in outs:
            for i, p in enumerate(pos):
                d = float((o[i].double().cpu() - alone).norm() / alone.norm())
                assert (d < 0.05) == (p - far < window or far < keep), (far, p, d)


# ------------------------------------------------------------------------------ gated delta rule
DELTA = {
    "square": DeltaSpec(4, 2, 128, 128, 4, 8, 8, 128 ** -0.5, 1e-6),
    "small": DeltaSpec(3, 1, 20, 24, 3, 8, 8, 0.3, 1e-6),
    "long_conv": DeltaSpec(2, 2, 64, 48, 6, 8, 8, 64 ** -0.5, 1e-2),
    "no_history": DeltaSpec(6, 3, 33, 128, 1, 8, 8, 1.0, 1e-6),
    "narrow": DeltaSpec(2, 1, 128, 33, 2, 8, 8, 0.1, 1e-6),
    "plain": DeltaSpec(2, 1, 40, 200, 4, 8, 8, 0.15, 1e-6),
}


class DeltaCase:
    def __init__(self, s, lens, dtype, seed=0, fast=1.0):
        """``fast`` scales the decays (50: whole chunks forget everything, some channels at once)."""
        from llm_sharding_amd.ops import delta as D
        self.s, self.dtype, self.lens = s, dtype, lens
        kc, vc = s.kv_heads * s.dim, s.heads * s.vdim
        self.cols = (8, 8 + kc, 8 + 2 * kc)
        self.w = {"conv": _rand(s.channels, s.taps, seed=seed, dtype=F32), "decay": torch.rand(s.heads, generator=_gen(1)) * fast + 0.02,
                  "dt_bias": _rand(s.heads * s.dim, seed=2, dtype=F32) - 1, "norm": torch.rand(s.vdim, generator=_gen(3)) + 0.5}
        self.x = [_rand(n, 8 + 2 * kc + vc, seed=seed + 10 + i, dtype=dtype) for i, n in enumerate(lens)]
        self.in32 = [_rand(n, s.heads + 3, seed=seed + 30 + i, dtype=F32) for i, n in enumerate(lens)]
        self.z = [_rand(n, s.heads * s.dim, seed=seed + 50 + i, dtype=F32) * 2 for i, n in enumerate(lens)]
        self.gate = [_rand(n, vc, seed=seed + 70 + i, dtype=dtype) for i, n in enumerate(lens)]
        self.state = tuple(torch.full(n, 3.0, device=DEV) for n in D.state_shapes(s, len(lens)))  # stale
        self.table = torch.zeros((len(lens), 8), dtype=torch.int32, device=DEV)
        self.wd = {k: v.to(DEV).contiguous() for k, v in self.w.items()}
        self.got = [torch.zeros(n, vc) for n in lens]
        self.at = [0] * len(lens)

    def want(self, i):
        s, w = self.s, {k: v.double() for k, v in self.w.items()}
        x, n = self.x[i].double(), self.lens[i]
        kc, H = s.kv_heads * s.dim, s.heads
        y = P.silu(P.short_conv(x[:, 8:], w["conv"]))
        q, k = P.unit_eps(y[:, :kc].view(n, -1, s.dim), s.unit_eps) * s.q_scale, P.unit_eps(y[:, kc:2 * kc].view(n, -1, s.dim), s.unit_eps)
        v = y[:, 2 * kc:].view(n, H, s.vdim)
        soft = torch.nn.functional.softplus(self.z[i].double() + w["dt_bias"]).view(n, H, s.dim)
        decay, beta = torch.exp(-w["decay"][:, None] * soft), torch.sigmoid(self.in32[i].double()[:, 3:])
        out, states = torch.empty(n, H, s.vdim, dtype=F64), []
        for h in range(H):
            o, S = P.delta_rule(q[:, h // s.group], k[:, h // s.group], v[:, h], decay[:, h], beta[:, h])
            out[:, h] = P.rms(o, 1e-5) * w["norm"]
            states.append(S)
        return out.reshape(n, -1) * torch.sigmoid(self.gate[i].double()), torch.stack(states)

    def step(self, parts, how):
        """One launch over the next rows of some sequences: [(sequence, rows)]."""
        from llm_sharding_amd.ops import delta as D
        s, runs, pick, row = self.s, [], [], 0
        for i, n in parts:
            runs.append((row, n, i, self.at[i]))
            pick += [(i, self.at[i] + t) for t in range(n)]
            row += n
            self.at[i] += n

        def rows(ts):
            return torch.stack([ts[i][p] for i, p in pick]).to(DEV)
        x, in32, z, gate = rows(self.x), rows(self.in32), rows(self.z), rows(self.gate)
        out = torch.zeros(row, s.heads * s.vdim, dtype=self.dtype, device=DEV)
        table = torch.tensor(runs, dtype=torch.int32)
        D.check_runs(table, row, len(self.lens))
        table = table.to(DEV)
        slot, pos = (torch.tensor(v, dtype=torch.int32, device=DEV) for v in ([r[2] for r in runs], [r[3] for r in runs]))
        kw = dict(slot=slot, pos=pos) if how == "rows" else dict(runs=table)
        a = D.make_args(s, self.wd, self.state, x, self.cols, in32, 3, z, gate, out, 1e-5, self.table, 8, **kw)
        if how in ("rows", "single"):
            D.steps(a, self.dtype, len(runs), keep=True)
        elif how == "steps":
            D.steps(a, self.dtype, len(runs), keep=False)
            D.ring(a, self.dtype, len(runs))
        else:
            nb = D.chunk_bytes(s)
            ws = torch.full((5 * s.heads * nb,), 255, dtype=torch.uint8, device=DEV)
            held = [(c.to(DEV), p.to(DEV)) for c, p in D.chunk_groups(runs, 5)]
            o32 = torch.full((row, s.heads * s.vdim), float("nan"), device=DEV)
            for c, p in held:
                D.chunked(a, c, p, ws, nb, o32)
            D.ring(a, self.dtype, len(runs))
        out = out.cpu().float()
        for (i, p), o in zip(pick, out):
            self.got[i][p] = o


@pytest.mark.parametrize("fast", [0.3, 50.0])
@pytest.mark.parametrize("dtype", [BF, F32])
@pytest.mark.parametrize("name", list(DELTA))
def test_delta_rule(name, dtype, fast):
    """Two sequences, in step-by-step runs, single rows and (bf16) chunks, all carrying the state on."""
    from llm_sharding_amd.ops import delta as D
    s = DELTA[name]
    nb = D.chunk_bytes(s)
    assert (nb > 0) == (name != "plain")
    long = "chunks" if dtype == BF and nb else "steps"
    case = DeltaCase(s, [180, 90], dtype, fast=fast)
    case.step([(1, 1), (0, 1)], "rows")
    case.step([(0, 70), (1, 33)], long)
    case.step([(1, 2), (0, 3)], "steps")
    for _ in range(5):
        case.step([(0, 1), (1, 1)], "single")
    case.step([(1, 49), (0, 100)], long)
    case.step([(0, 1)], "rows")
    assert case.at == [180, 90]
    for i in (0, 1):
        out, S = case.want(i)
        close(case.got[i], out, 6e-3 if dtype == BF else 2e-5, f"{name}: outputs of {i}")
        close(case.state[0][i, :, :s.dim, :s.vdim], S, 3e-5, f"{name}: state of {i}")
    rest = case.state[0].clone()
    rest[:, :, :s.dim, :s.vdim] = 0
    assert not rest.any()


def test_delta_forgets_and_remembers():
    """One loud write, then a decay that keeps (or drops) it: the read-out a hundred rows later shows which."""
    s = DeltaSpec(1, 1, 32, 32, 2, 8, 8, 1.0, 1e-6)
    for z, kept in ((-30.0, True), (3.0, False)):
        case = DeltaCase(s, [140], BF)
        case.w["conv"][:] = 0
        case.w["conv"][:, -1] = 1
        case.wd["conv"] = case.w["conv"].to(DEV)
        case.z[0][:] = z
        case.in32[0][:] = -30.0   # no writes ..
        case.in32[0][3] = 30.0    # .. but one
        case.x[0][:, 8:72] = case.x[0][3, 8:72].abs()  # the same query and key throughout
        case.step([(0, 140)], "chunks")
        out, _ = case.want(0)
        close(case.got[0], out, 6e-3, "outputs")
        assert (case.got[0][139].abs().max() > 0.3) == kept


@pytest.mark.parametrize("heads,dim,vdim", [(64, 128, 128), (65, 128, 128), (128, 64, 40), (129, 64, 40), (3, 64, 128)])
def test_delta_scan_of_few_and_many_heads(heads, dim, vdim):
    """Value channels to 256 workgroups or fewer, and past that; a ragged last chunk and a state carried on. Limits as above."""
    case = DeltaCase(DeltaSpec(heads, 1, dim, vdim, 4, 8, 8, dim ** -0.5, 1e-6), [103], BF, fast=0.3)
    case.step([(0, 97)], "chunks")
    case.step([(0, 6)], "chunks")
    out, S = case.want(0)
    close(case.got[0], out, 6e-3, "outputs")
    close(case.state[0][0, :, :dim, :vdim], S, 3e-5, "state")


def test_idle_rows_leave_state_alone():
    from llm_sharding_amd.ops import delta as D
    s = DELTA["small"]
    case = DeltaCase(s, [4, 4], BF)
    case.table[1] = -1
    before = [t.clone() for t in case.state]
    case.step([(1, 1)], "rows")
    assert not case.got[1].any() and all(torch.equal(a, b) for a, b in zip(before, case.state))
    case.table[1] = 0
    with pytest.raises(ValueError):
        D.check_runs(torch.tensor([[0, 2, 0, 0], [2, 2, 0, 9]]), 4, 2)  # two runs of one slot
    with pytest.raises(ValueError):
        D.check_runs(torch.tensor([[0, 5, 0, 0]]), 4, 2)


# ------------------------------------------------------------------------------ experts
@pytest.mark.parametrize("dtype", [BF, F32])
@pytest.mark.parametrize("rows,experts,top,ff,width", [
    (1, 8, 8, 40, 72), (5, 5, 1, 130, 200), (64, 7, 3, 64, 256), (65, 300, 2, 20, 130), (130, 4, 4, 90, 88),
    (300, 3, 2, 100, 140), (700, 2, 1, 257, 384), (2000, 5, 2, 128, 256)])
def test_experts(dtype, rows, experts, top, ff, width):
    """Few and many pairs per expert, experts nobody chose, one expert for all rows, ties."""
    from llm_sharding_amd.ops import moe as X
    gate, up = ([_rand(ff, width, seed=e + 100 * i, scale=width ** -0.5) for e in range(experts)] for i in (1, 2))
    down = [_rand(width, ff, seed=e + 300, scale=ff ** -0.5) for e in range(experts)]
    x = X.Experts(*([w.to(DEV, dtype) for w in ws] for ws in (gate, up, down)))
    h, logits = _rand(rows, width, seed=4), _rand(rows, experts + 5, seed=5, dtype=F32)
    logits[:, 2 % experts] += 3           # a favourite
    logits[::3, :experts] = logits[::3, :1]  # ties: the first ones
    pairs = rows * top
    hp = torch.zeros(rows, x.width, dtype=dtype, device=DEV)
    hp[:, :width] = h.to(DEV, dtype)
    expert, order, place = torch.full((3, pairs), -7, dtype=torch.int32, device=DEV)
    weight = torch.zeros(pairs, device=DEV)
    tr = X.tile_rows(pairs, experts, dtype == F32)
    tiles = torch.full((X.max_tiles(pairs, experts, tr), 4), -9, dtype=torch.int32, device=DEV)
    nt = X.route_group(logits.to(DEV), rows, experts, top, tr, expert, weight, order, place, tiles)
    best = logits[:, :experts].double().sort(dim=-1, descending=True, stable=True)
    at = best.indices[:, :top]
    assert torch.equal(expert.cpu().view(rows, top).long(), at)
    close(weight.view(rows, top), torch.softmax(best.values[:, :top], -1), 1e-6, "weights")
    assert torch.equal(order.cpu().long()[place.cpu().long()], torch.arange(pairs))
    seen = 0
    for e, start, count, _ in tiles.cpu().tolist():
        if e >= 0:
            assert 1 <= count <= tr and bool((expert.cpu()[order.cpu()[start:start + count].long()] == e).all())
            seen += count
    assert seen == pairs and nt == tiles.shape[0]
    act, ye = (torch.zeros(pairs, n, dtype=dtype, device=DEV) for n in (x.ff, x.width))
    X.gemm(tiles, nt, tr, order, top, hp, x.up, 2 * x.ff, x.width, act, pairs, X.GLU)
    X.gemm(tiles, nt, tr, order, top, act, x.down, x.width, x.ff, ye, pairs, X.DOWN)
    got = (ye.cpu().double()[place.cpu().long()] * weight.cpu().double()[:, None]).view(rows, top, -1).sum(1)
    want = torch.zeros(rows, width, dtype=F64)
    wts = torch.softmax(best.values[:, :top], -1)
    for e in range(experts):
        r, k = (at == e).nonzero(as_tuple=True)
        a = P.silu(h[r].double() @ gate[e].double().T) * (h[r].double() @ up[e].double().T)
        want.index_add_(0, r, a @ down[e].double().T * wts[r, k, None])
    close(got[:, :width], want, 1e-2 if dtype == BF else 1e-5, "experts")
    assert not got[:, width:].any()


# ------------------------------------------------------------------------------ engine
@pytest.fixture(scope="module")
def ordinary():
    cfg = M.stack()
    return cfg, M.tensors(cfg)


@pytest.mark.parametrize("dtype", [BF, F32])
@pytest.mark.parametrize("sizes", [[300], [64, 1, 63, 66, 128], [2, 3, 2], [100, 65, 1, 1, 1], [1]])
def test_portions(ordinary, dtype, sizes):
    cfg, t = ordinary
    ids = _ids(300 if sizes[0] > 3 else 140)
    want = P.run(cfg.to_dict(), t, ids)
    eng = M.engine(cfg, DEV, dtype)
    got = torch.cat([M.feed(eng, [(1, p)]) for p in M.cut(ids, sizes)])
    assert off(got, want, dtype) < TOL[dtype]


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
    """A two-token prompt, then 330 single tokens across pages and windows."""
    cfg, t = ordinary
    ids = _ids(332, seed=5)
    want = P.run(cfg.to_dict(), t, ids)
    eng = M.engine(cfg, DEV, dtype)
    got = [M.feed(eng, [(3, ids[:2])])] + [M.feed(eng, [(3, [x])]) for x in ids[2:]]
    assert off(torch.cat(got), want, dtype) < TOL[dtype]


@pytest.mark.parametrize("dtype", [BF, F32])
def test_unequal_batches_on_reused_pages_and_slots(ordinary, dtype):
    cfg, t = ordinary
    eng = M.engine(cfg, DEV, dtype, cache_tokens=64 * 10)
    seqs = {k: _ids(n, seed=k) for k, n in ((0, 260), (1, 75), (2, 200), (3, 140), (4, 3))}
    want = {k: P.run(cfg.to_dict(), t, v) for k, v in seqs.items()}
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
        assert at[k] == len(seqs[k]) and off(torch.cat(got[k]), want[k], dtype) < TOL[dtype], k
    with pytest.raises(ValueError):
        eng.forward(torch.zeros(3, cfg.hidden_size, device=DEV), [0, 1, 0], [140, 0, 143])


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
    """Sizes beyond the tuned kernels, ones, one expert, a window of one key, scale 1, a tight cap, a width the
    fused joins take and one they do not."""
    for width in (130, 144):
        cfg = G.make_config(width, 129, [
            G.attention_entry(2, 1, 300, 270, 1, 1, G.moe(1, 1, 1), scale=1.0, softcap=1.0),
            G.delta_entry(1, 1, 1, 1, 1, G.dense(1)),
            G.attention_entry(3, 3, 1, 1, 64, 64, None, softcap=0.5),
            G.delta_entry(4, 1, 130, 140, 7, G.moe(9, 9, 17)),
            G.attention_entry(34, 1, 16, 16, 100, 0, G.dense(129), kv_from=None),
            G.attention_entry(2, 1, 300, 270, 77, 2, G.dense(30), kv_from=0)], eps=0.5, embed_scale=1.0, rank=1)
        t = M.tensors(cfg)
        ids = _ids(150, vocab=129)
        want = P.run(cfg.to_dict(), t, ids)
        for dtype, tol in ((F32, SHARP_TOL), (BF, 5e-2)):
            eng = M.engine(cfg, DEV, dtype)
            got = torch.cat([M.feed(eng, [(0, p)]) for p in M.cut(ids, [100, 1, 49])])
            assert off(got, want, dtype) < tol, (width, dtype)


def test_layers_of_a_real_width():
    """Wide heads and states, enough pairs for every expert kernel, portions on every projection kernel."""
    cfg = G.make_config(512, 260, [
        G.attention_entry(16, 4, 128, 128, 200, 4, G.dense(600)),
        G.delta_entry(4, 2, 128, 128, 4, G.moe(2, 1, 256)),
        G.attention_entry(16, 4, 128, 128, 90, 4, G.moe(6, 2, 200), kv_from=0)], rank=64)
    t = M.tensors(cfg)
    ids = _ids(850, vocab=260)
    want = P.run(cfg.to_dict(), t, ids, dtype=F32)
    eng = M.engine(cfg, DEV, BF, max_seq=1024, max_prefill_rows=1024)
    got = torch.cat([M.feed(eng, [(0, p)]) for p in M.cut(ids, [600, 1, 20, 64, 129, 2, 34])])
    assert off(got, want, BF) < TOL[BF]


# ------------------------------------------------------------------------------ generation
@pytest.mark.parametrize("dtype", [F32, BF])
@pytest.mark.parametrize("graph", [True, False])
def test_greedy_generation_through_the_server(ordinary, dtype, graph):
    """More requests than slots over a small page pool, prompts cut at the prefill budget, decode graphs
    replayed while slots (and their states) come and go."""
    cfg, t = ordinary
    prompts = [_ids(n, seed=20 + n) for n in (4, 130, 1, 65, 33, 90, 7)]
    srv = PipelineServer(cfg, M.NamedSource(cfg, 0), device=DEV, batch=2, microbatches=2, max_seq=192, prefill_budget=100,
                         dtype=dtype, use_graph=graph, cache_tokens=64 * 7)
    outs = srv.generate(prompts, 8, eos_ids=())
    for p, o in zip(prompts, outs):
        want, gaps = P.greedy(cfg.to_dict(), t, p, 8)
        clear = next((i for i, gp in enumerate(gaps) if gp < (0.1 if dtype == BF else 1e-3)), 8)
        assert o[:clear] == want[:clear], (len(p), o, want, gaps)
    assert len(srv.eng.pool.free) == srv.eng.pool.pages


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
    cfg, _ = ordinary
    prompts = [_ids(60, seed=1), _ids(62, seed=2), _ids(3, seed=3)]
    a, b = M.engine(cfg, DEV, dtype), M.engine(cfg, DEV, dtype)
    for eng in (a, b):
        M.feed(eng, [(i, p) for i, p in enumerate(prompts)])
    g = DecodeGraph(a, 3, "full", history_len=8)
    tok = torch.tensor([5, 6, 7], dtype=torch.int32)
    g.tokens.copy_(tok)
    g.capture()
    for i in range(8):  # crosses a page border
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
    cfg = get_preset("tiny-gupuvik")
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
    folder = G.write_random_checkpoint(cfg, str(tmp_path / "m"), seed=0)
    ids = _ids(70)
    want = P.run(cfg.to_dict(), t, ids)
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


@pytest.mark.parametrize("pairs,experts", [(700, 1), (2500, 5), (4100, 12)])
@pytest.mark.parametrize("rows", [64, 128, 256])  # (64: fp32)
def test_experts_share_out_the_tiles_there_are(pairs, experts, rows):
    """Every entry tells how many tiles the table has; a table that does not tell gives the same."""
    from llm_sharding_amd.ops import moe as X
    from llm_sharding_amd.ops.packing import pack_b, pack_f32
    dtype, pack = (F32, pack_f32) if rows == 64 else (BF, pack_b)
    g = torch.Generator().manual_seed(pairs)
    expert = (torch.rand(pairs, generator=g).square() * experts).int().to(DEV)
    n, k = 256, 128
    w = torch.stack([pack(torch.randn(n, k, generator=g).to(DEV, dtype)) for _ in range(experts)]).contiguous()
    a = torch.randn(pairs, k, generator=g).to(DEV, dtype)
    order, place = (torch.empty(pairs, dtype=torch.int32, device=DEV) for _ in range(2))
    tiles = torch.full((X.max_tiles(pairs, experts, rows), 4), -7, dtype=torch.int32, device=DEV)
    nt = X.group(expert, pairs, experts, rows, order, place, tiles)
    count = torch.bincount(expert.long().cpu(), minlength=experts)
    used = int(((count + rows - 1) // rows).sum())
    assert nt == tiles.shape[0] and bool((tiles[:, 3] == used).all())
    assert bool((tiles[:used, 0] >= 0).all()) and bool((tiles[used:, 0] == -1).all())
    outs = []
    for table in (tiles, tiles * torch.tensor([1, 1, 1, 0], dtype=torch.int32, device=DEV)):
        out = torch.zeros(pairs, n, dtype=dtype, device=DEV)
        X.gemm(table, nt, rows, order, 1, a, w, n, k, out, pairs, X.DOWN)
        outs.append(out)
    assert torch.equal(*outs) and bool((outs[0].abs().sum(1) > 0).all())


# pairs of each expert; on which tiles have the fewest rounds: a few rows over a tile's, one below, none, one expert for all
DEALS = [[129] * 8, [193] * 40 + [0, 1], [257, 256, 255, 0, 1], [321, 320, 319] * 20, [640] * 16, [5000], [1] * 7 + [700], [797] * 32]


@pytest.mark.parametrize("deal", range(len(DEALS)))
@pytest.mark.parametrize("up", ["glu", "relu2"])
def test_experts_tiles_of_the_height_that_the_pairs_make_best(deal, up):
    """The height is the cheapest by the costs given, the table that of this height, and both products give what tiles of 128 and 256
    rows give, bit for bit (a pair's sums run in the same order)."""
    from llm_sharding_amd.ops import moe as X
    from llm_sharding_amd.ops.packing import pack_b
    counts = torch.tensor(DEALS[deal])
    experts, pairs = len(counts), int(counts.sum())
    g = torch.Generator().manual_seed(deal)
    e = torch.repeat_interleave(torch.arange(experts), counts)[torch.randperm(pairs, generator=g)].int()
    kind, n, k = (X.GLU, 512, 192) if up == "glu" else (X.RELU2, 256, 192)
    width, ff = 256, n // 2 if up == "glu" else n
    assert X.pick((n + 128, k), (width, ff)) is None
    heights = X.pick((n, k), (width, ff))

    def us(i):
        total = 0.0
        for p in range(2):
            tiles = int(((counts + X.HEIGHTS[i] - 1) // X.HEIGHTS[i]).sum()) * heights.nt[p]
            full, rem = divmod(tiles, 256)
            last = heights.step[i][p] * (1 - 0.47 * (1 - rem / 256)) + heights.own[i] if rem else 0.0
            total += full * (heights.step[i][p] + heights.own[i]) + last
        return total
    cost = [us(i) for i in range(4)]
    wu = torch.stack([pack_b(_rand(n, k, seed=i, scale=k ** -0.5).to(DEV)) for i in range(experts)])
    wd = torch.stack([pack_b(_rand(width, ff, seed=i + 99, scale=ff ** -0.5).to(DEV)) for i in range(experts)])
    h = _rand(pairs, k, seed=7).to(DEV)
    for spare in (None, torch.zeros(pairs + 1024, dtype=torch.int32, device=DEV)):
        order, place = (torch.empty(pairs, dtype=torch.int32, device=DEV) for _ in range(2))
        outs = []
        for rows in (0, 128, 256):
            tiles = torch.full((X.max_tiles(pairs, experts, rows or 128), 4), -7, dtype=torch.int32, device=DEV)
            nt = X.group(e.to(DEV), pairs, experts, rows or 128, order, place, tiles, spare, None if rows else heights)
            if not rows:
                i, used = divmod(int(tiles[0, 3]), 1 << 24)
                assert cost[i] <= min(cost) * (1 + 1e-5), (i, cost)
                assert used == int(((counts + X.HEIGHTS[i] - 1) // X.HEIGHTS[i]).sum()) and bool((tiles[used:, 0] == -1).all())
                assert int(tiles[:used, 2].max()) <= X.HEIGHTS[i] and int(tiles[:used, 2].sum()) == pairs
            act, ye = (torch.full((pairs, c), float("nan"), dtype=BF, device=DEV) for c in (ff, width))
            X.gemm(tiles, nt, rows, order, 1, h, wu, n, k, act, pairs, kind)
            X.gemm(tiles, nt, rows, order, 1, act, wd, width, ff, ye, pairs, X.DOWN)
            outs.append((act[place.long()], ye[place.long()]))  # (the order within an expert is not the same every time)
        for a, y in outs[1:]:
            assert torch.equal(a, outs[0][0]) and torch.equal(y, outs[0][1])


@pytest.mark.parametrize("pairs", [10239, 10240, 12287, 12288, 12289, 40961])
@pytest.mark.parametrize("experts", [1, 7, 32, 1024])
def test_many_pairs_are_sorted_by_several_workgroups(pairs, experts):
    """With scratch the order is a sort by expert, ``place`` its inverse, and the tiles are those of one workgroup; one expert
    has none. Too little scratch is none."""
    from llm_sharding_amd.ops import moe as X
    g = torch.Generator().manual_seed(pairs + experts)
    e = (torch.rand(pairs, generator=g).square() * experts).int()
    if experts > 1:
        e[e == 3] = 1
    expert, tables = e.to(DEV), []
    for spare in (None, torch.full((pairs,), -9, dtype=torch.int32, device=DEV), torch.zeros(3, dtype=torch.int32, device=DEV)):
        order, place = (torch.full((pairs,), -5, dtype=torch.int32, device=DEV) for _ in range(2))
        tiles = torch.full((X.max_tiles(pairs, experts, 64), 4), -7, dtype=torch.int32, device=DEV)
        X.group(expert, pairs, experts, 64, order, place, tiles, spare)
        o = order.cpu().long()
        assert torch.equal(o.sort().values, torch.arange(pairs)) and torch.equal(e[o], e.sort().values)
        assert torch.equal(place.cpu().long()[o], torch.arange(pairs))
        tables.append(tiles)
    assert torch.equal(tables[0], tables[1]) and torch.equal(tables[0], tables[2])


@pytest.mark.parametrize("kind", ["down", "glu", "relu2"])
@pytest.mark.parametrize("n,k", [(32, 32), (96, 160), (160, 64), (256, 96)])
@pytest.mark.parametrize("narrow", [False, True])
def test_fp32_tiles_of_both_widths(kind, n, k, narrow, monkeypatch):
    """64 pairs by 64 and by 128 columns: columns and pairs that fill no tile, experts with one pair, none, and a tile and two more;
    nothing written beside the result."""
    from llm_sharding_amd.ops import moe as X
    from llm_sharding_amd.ops.packing import pack_f32
    up = {"down": X.DOWN, "glu": X.GLU, "relu2": X.RELU2}[kind]
    monkeypatch.setattr(X, "narrow_tiles", lambda *a: narrow)
    e = torch.tensor([0] * 66 + [2] + [3] * 64).int()[torch.randperm(131, generator=torch.Generator().manual_seed(1))]
    pairs, experts, cols = 131, 4, n // 2 if up == X.GLU else n
    w, a = _rand(experts, n, k, seed=2, scale=k ** -0.5, dtype=F32), _rand(pairs, k, seed=3, dtype=F32)
    order, place = (torch.zeros(pairs, dtype=torch.int32, device=DEV) for _ in range(2))
    tiles = torch.zeros((X.max_tiles(pairs, experts, 64), 4), dtype=torch.int32, device=DEV)
    nt = X.group(e.to(DEV), pairs, experts, 64, order, place, tiles)
    at = order.cpu().long()
    rows = a if up else a[at]  # down reads the sorted pairs
    out = torch.full((pairs + 1, cols + 4), 7.0, device=DEV)
    X.gemm(tiles, nt, 64, order, 1, rows.to(DEV), torch.stack([pack_f32(x) for x in w]).to(DEV), n, k, out, pairs, up)
    y = torch.einsum("pnk,pk->pn", w.double()[e[at].long()], a.double()[at])
    if up == X.GLU:
        y = y.view(pairs, -1, 2, 16)
        y = (torch.nn.functional.silu(y[:, :, 0]) * y[:, :, 1]).flatten(1)
    elif up == X.RELU2:
        y = y.relu().square()
    close(out[:pairs, :cols], y, 2e-6, kind)
    assert bool((out[pairs:] == 7).all()) and bool((out[:, cols:] == 7).all())

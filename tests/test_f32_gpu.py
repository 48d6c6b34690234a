"""Products and attention of the fp32 engine on the GPU against float64, at the edges of their tiles and of the rules that
choose between their forms."""
import pytest
import torch

from llm_sharding_amd.models.stack import GluSpec
from llm_sharding_amd.ops import hip
from llm_sharding_amd.ops.packing import pack_f32
from llm_sharding_amd.ops.stream import Linear, linear_f32_form

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _rand(*shape, seed=0, scale=1.0):
    return torch.randn(*shape, generator=torch.Generator().manual_seed(seed)) * scale


def rows_close(got, want, tol, what):
    """Every row by itself."""
    got = got.double().cpu()
    assert torch.isfinite(got).all(), what
    off = (got - want).norm(dim=-1) / want.norm(dim=-1)
    assert off.max() < tol, f"{what}: row {int(off.argmax())} is {float(off.max()):.2e} off"


def sum_tol(k):
    """k products and sums, each rounded or cut to 2^-23 of a partial sum that grows as the root of their number."""
    return 2.0 ** -23 * k ** 0.5 + 2.0 ** -22


@pytest.mark.parametrize("rows", [1, 8, 16, 17, 33, 64, 65, 128, 129, 200, 520])
@pytest.mark.parametrize("n,k", [(48, 16), (144, 48), (1024, 128), (4112, 160)])
def test_linear_store(rows, n, k):
    """Few and many rows, columns and k that fill no tile; a stride; nothing written beside the result."""
    x, w, b = _rand(rows, k + 4, seed=1), _rand(n, k, seed=2, scale=k ** -0.5), _rand(n, seed=3)
    xd, wd, bd = x.to(DEV), pack_f32(w).to(DEV), b.to(DEV)
    out = torch.full((rows + 1, n + 16 - n % 8), 7.0, device=DEV)
    ep = hip.make_epi(out=out, ldo=out.stride(0), bias=bd)
    st = hip.lib().lsa_linear_f32(xd.data_ptr(), xd.stride(0), wd.data_ptr(), rows, n, k, hip.EPI_STORE, ep, None, 0, None, 0,
                                  torch.cuda.current_stream().cuda_stream)
    assert st == 0
    rows_close(out[:rows, :n], x[:, :k].double() @ w.double().T + b.double(), sum_tol(k), "store")
    assert bool((out[rows:] == 7).all()) and bool((out[:, n:] == 7).all())


@pytest.mark.parametrize("rows,n,k", [(33, 1456, 4096), (64, 2048, 64), (64, 2048, 992), (90, 1040, 2080), (170, 4112, 160),
                                      (700, 2048, 2048), (1030, 1024, 4096)])
@pytest.mark.parametrize("slab", [0, 70000, 768 * 4096])
def test_linear_in_parts(rows, n, k, slab):
    """Products of short and long K around the border between streamed weights and tiles, with scratch and without: the same bits
    each time, the counters left at zero, and nothing written past the scratch."""
    in_parts(rows, n, k, slab)


SLAB = 256 * 128 * 256  # an engine's


@pytest.mark.parametrize("rows,n,k,slab,form", [
    (70, 2080, 2144, SLAB, (64, 64, 0, 3)), (70, 2080, 2144, 600000, (64, 64, 0, 2)), (283, 4096, 8192, 1000000, (64, 64, 256, 3)),
    (283, 4096, 8192, 768 * 4096, (64, 64, 256, 4)), (283, 4096, 8192, 0, (64, 128, 160, 1)), (283, 4096, 8192, SLAB, (64, 128, 0, 3)),
    (70, 4128, 2080, SLAB, (64, 128, 0, 3)), (505, 4128, 2144, SLAB, (64, 128, 256, 8)), (505, 2080, 2144, SLAB, (128, 128, 0, 3)),
    (505, 8224, 2080, SLAB, (128, 128, 256, 8)), (505, 4416, 4064, SLAB, (128, 256, 0, 3)), (900, 8224, 2080, SLAB, (128, 256, 256, 6))])
@pytest.mark.parametrize("gated", [False, True])
def test_linear_in_parts_of_every_form(rows, n, k, slab, form, gated):
    """K in parts of each size of tiles: of all tiles and of those past the ones that fill the CUs, uneven, fewer where the
    scratch is small, none without it; rows and columns that fill no tile."""
    n -= 16 if n % 64 and not gated else 0
    assert linear_f32_form(rows, n, k, gated, slab) == form
    in_parts(rows, n, k, slab, gated)


def in_parts(rows, n, k, slab, gated=False):
    x, w, b = _rand(rows, k, seed=1).to(DEV), _rand(n, k, seed=2, scale=k ** -0.5).to(DEV), _rand(n, seed=3).to(DEV)
    wd = pack_f32(w)
    part, cnt = torch.full((slab + 64,), 7.0, device=DEV), torch.zeros(256, dtype=torch.int32, device=DEV)
    outs = []
    for _ in range(3):
        out = torch.full((rows, n + 16 - n % 8), 7.0, device=DEV)
        ep = hip.make_epi(**{"out32" if gated else "out": out}, ldo=out.stride(0), bias=b)
        st = hip.lib().lsa_linear_f32(x.data_ptr(), k, wd.data_ptr(), rows, n, k, hip.EPI_GEGLU if gated else hip.EPI_STORE, ep,
                                      part.data_ptr() if slab else None, slab, cnt.data_ptr(), 256,
                                      torch.cuda.current_stream().cuda_stream)
        assert st == 0
        outs.append(out)
    want = (x.double() @ w.double().T + b.double()).cpu()
    if gated:  # 16 columns of gates, 16 of what they open
        want = want.view(rows, -1, 2, 16)
        want = (torch.nn.functional.gelu(want[:, :, 0], approximate="tanh") * want[:, :, 1]).flatten(1)
    rows_close(outs[0][:, :want.shape[1]], want, 2 * sum_tol(k) + 1e-6 if gated else sum_tol(k), "parts")
    assert all(torch.equal(outs[0], o) for o in outs[1:]) and bool((outs[0][:, want.shape[1]:] == 7).all())
    assert not cnt.any() and bool((part[slab:] == 7).all())


def product(x, w):
    """x w^T by the kernel itself (Linear fills k up), 16 columns of 7 beside it."""
    (rows, k), n, xd, wd = x.shape, w.shape[0], x.to(DEV), pack_f32(w).to(DEV)
    out, part = torch.full((rows, n + 16), 7.0, device=DEV), torch.empty(256 * 128 * 256, device=DEV)
    cnt = torch.zeros(256, dtype=torch.int32, device=DEV)
    assert hip.lib().lsa_linear_f32(xd.data_ptr(), k, wd.data_ptr(), rows, n, k, hip.EPI_STORE, hip.make_epi(out=out, ldo=n + 16),
                                    part.data_ptr(), part.numel(), cnt.data_ptr(), 256,
                                    torch.cuda.current_stream().cuda_stream) == 0
    assert bool((out[:, n:] == 7).all())
    return out[:, :n].double().cpu()


@pytest.mark.parametrize("rows", [4, 33, 64])
@pytest.mark.parametrize("k", [2048, 4096])
def test_streamed_products_are_sums_of_sixteenths(rows, k):
    """Of random operands. k / 16 roundings in each of 16 sums, of partial sums that grow as the root of their number: each off by
    2^-24 / 3^0.5 of its value on average, together by the root of k / 32 times that."""
    assert linear_f32_form(rows, 2048, k) == (16, 0, 0, 1)
    x, w = _rand(rows, k, seed=1), _rand(2048, k, seed=2, scale=k ** -0.5)
    want = x.double() @ w.double().T
    assert (product(x, w) - want).norm() / want.norm() < 2.0 ** -24 / 3 ** 0.5 * (k / 32) ** 0.5


@pytest.mark.parametrize("rows,n,k", [(33, 8464, 64), (65, 16400, 32), (100, 4112, 96), (129, 16400, 224), (257, 4368, 544),
                                      (960, 8208, 128), (2100, 2064, 160)])
def test_linear_tiles(rows, n, k):
    """Every size of tiles, with rows, columns and groups' parts of k that fill none; values of very different sizes, which a
    product of only the leading pieces would miss."""
    x, w = _rand(rows, k, seed=1), _rand(n, k, seed=2, scale=k ** -0.5)
    x *= torch.exp2(torch.randint(-90, 60, (rows, 1), generator=torch.Generator().manual_seed(3)).float())
    w *= torch.exp2(torch.randint(-30, 30, (n, 1), generator=torch.Generator().manual_seed(4)).float())
    want = x.double() @ w.double().T
    scale = x.double().norm(dim=1)[:, None] * w.double().norm(dim=1)[None]
    off = ((product(x, w) - want).abs() / scale).max()  # of every value by itself
    assert off < sum_tol(k)


@pytest.mark.parametrize("rows,n,k", [(40, 4112, 64), (200, 2064, 2048), (600, 8464, 96)])
def test_linear_values_that_are_no_numbers(rows, n, k):
    """Infinities, NaN and values that round to an infinity in bf16 give what fp32 products of them give, and leave all other
    results as they are without them; zeros meet infinities, and values at the lower end keep all their bits."""
    x, w = _rand(rows, k, seed=1), _rand(n, k, seed=2, scale=k ** -0.5)
    w[::7, 5] = 0
    w[3::16] = w[3::16].bfloat16().float()  # second and third pieces that are zero
    clean = x.double() @ w.double().T
    x[1, 5], x[rows - 1, 5], x[2, 7], x[17, 5], x[17, 6], x[30, 9] = [float(v) for v in ("inf", "-inf", "nan", "inf", "-inf", 3.4e38)]
    x[33] = torch.rand(k) * 1e-38
    x[34] = 1e-41
    want = x.double() @ w.double().T
    got = product(x, w)
    fine = torch.ones(rows, dtype=torch.bool)
    fine[[1, 2, 17, 30, 33, 34, rows - 1]] = False
    rows_close(got[fine], clean[fine], sum_tol(k), "rows beside")
    for r in (1, 2, 17, rows - 1):
        assert torch.equal(got[r].isnan(), want[r].isnan()) and torch.equal(got[r][got[r].isinf()], want[r][want[r].isinf()]), r
        assert not got[r].isfinite().any()
    over = want[30].abs() > 3.402823e38
    assert torch.equal(got[30].isinf(), over) or (got[30].isinf() ^ over).sum() <= 1
    assert ((got[30] - want[30]).abs()[~over & got[30].isfinite()] < 1e-5 * 3.4e38).all()
    rows_close(got[33:34], want[33:34], sum_tol(k) + 2.0 ** -20, "small values")  # (results down to 2^-130, of 19 bits)
    assert (got[34] - want[34]).abs().max() < sum_tol(k) * want[34].abs().max() + 2.0 ** -145  # up to 20 sums' last bits of 2^-149


@pytest.mark.parametrize("rows,n,k", [(33, 8464, 64), (100, 4112, 96), (200, 2064, 2048), (257, 4368, 544), (960, 8208, 128)])
def test_linear_tiles_at_the_ends_of_the_range(rows, n, k):
    """Rows of values from fp32's last bit to 2^120, as exact as any; and values of both kinds in one row, where the small ones'
    weights are as much larger."""
    x, w = _rand(rows, k, seed=1), _rand(n, k, seed=2, scale=k ** -0.5)
    e = torch.arange(rows)[:, None].remainder(270).double() - 150
    lo = (x.double() * torch.exp2(e)).float()
    a, b = (e < -50)[:, 0], (e >= -50)[:, 0]
    for r, f in ((a, 2.0 ** 40), (b, 2.0 ** -40)):
        if r.any():
            some = lo[r].any(1)
            rows_close(product(lo[r], w * f)[some], (lo[r].double() @ (w * f).double().T)[some], sum_tol(k), "rows")
    x[:, ::2] *= 2.0 ** -125
    w[:, ::2] *= 2.0 ** 95
    w[:, 1::2] *= 2.0 ** -30
    rows_close(product(x, w), x.double() @ w.double().T, sum_tol(k), "in one row")


@pytest.mark.parametrize("kind", ["store", "silu", "gelu"])
@pytest.mark.parametrize("rows,n,k", [(20, 8448, 2048), (64, 8448, 2048), (700, 8448, 2048), (283, 4096, 8192), (2500, 4352, 2048)])
def test_parts_beside_each_other_on_a_cu(kind, rows, n, k):
    """More parts than CUs, or whole tiles for all CUs and parts (the two largest products; the others have one for a CU at most): one
    writes its sums while another of the same CU keeps the memory pipe busy."""
    bm, bn, whole, parts = linear_f32_form(rows, n, k, kind != "store")
    if n < 8448:
        assert parts > 1 and whole + (-(-rows // bm) * -(-n // bn) - whole) * parts > 256
    x, w = _rand(rows, k, seed=1).to(DEV), _rand(n, k, seed=2, scale=k ** -0.5).to(DEV)
    if kind == "store":
        lin, glu, want = Linear(w), None, x.double() @ w.double().T
    else:
        g, u = w[:n // 2], w[n // 2:]
        lin, glu = Linear.glu(g, u), GluSpec(ff=n // 2, gelu=kind == "gelu")
        a = x.double() @ g.double().T
        a = torch.nn.functional.gelu(a, approximate="tanh") if glu.gelu else torch.nn.functional.silu(a)
        want = a * (x.double() @ u.double().T)
    for _ in range(5):
        out = torch.zeros(rows, want.shape[1], device=DEV)
        lin(x, rows, out, glu=glu)
        rows_close(out, want.cpu(), 2 * sum_tol(k) + 1e-6, kind)


@pytest.mark.parametrize("rows", [1, 16, 31, 100, 300, 2100])
@pytest.mark.parametrize("gelu", [False, True])
def test_linear_gated(rows, gelu):
    ff, k = 1040, 256
    x, g, u = _rand(rows, k, seed=1), _rand(ff, k, seed=2, scale=k ** -0.5), _rand(ff, k, seed=3, scale=k ** -0.5)
    lin = Linear.glu(g.to(DEV), u.to(DEV))
    out = torch.zeros(rows, lin.n // 2, device=DEV)
    lin(x.to(DEV), rows, out, glu=GluSpec(ff=ff, gelu=True) if gelu else GluSpec(ff=ff))
    a, b = x.double() @ g.double().T, x.double() @ u.double().T
    act = torch.nn.functional.gelu(a, approximate="tanh") if gelu else torch.nn.functional.silu(a)
    rows_close(out[:, :ff], act * b, 2 * sum_tol(k) + 1e-6, "gated")
    assert not out[:, ff:].any()


@pytest.mark.parametrize("rows", [5, 40, 700])
def test_linear_two_outputs_and_join(rows):
    """Columns beside each other in two tensors with an activation on some; a result that joins a stream through a gate."""
    n, k = 640, 128
    x, w, gate, s = _rand(rows, k, seed=1), _rand(n, k, seed=2, scale=k ** -0.5), _rand(rows, n, seed=3), _rand(rows, n, seed=4)
    lin, y = Linear(w.to(DEV)), x.double() @ w.double().T
    out, out32 = torch.zeros(rows, 512, device=DEV), torch.zeros(rows, 128, device=DEV)
    lin(x.to(DEV), rows, out, out32=out32, col32=512, act_from=256)
    act = torch.nn.functional.gelu(y[:, 256:512], approximate="tanh")
    rows_close(out, torch.cat([y[:, :256], act], 1), sum_tol(k) + 1e-6, "store")
    rows_close(out32, y[:, 512:], sum_tol(k), "fp32 columns")
    sd = s.to(DEV)
    lin(x.to(DEV), rows, None, out32=sd, gate=gate.to(DEV), cols=624)
    want = s.double()
    want[:, :624] += torch.sigmoid(gate.double()[:, :624]) * y[:, :624]
    rows_close(sd, want, sum_tol(k) + 1e-6, "join")


@pytest.mark.parametrize("name,rows", [("r512_many", 340), ("small", 40)])
def test_latent_attention_of_many_rows(name, rows):
    """Enough rows for the wide form of the absorbed queries; rows at both ends of a page, and idle ones between."""
    from test_deretar_gpu import SIZES, Case, _absorbed
    case = Case(SIZES[name], [200, 130], torch.float32)
    slot = [i % 2 for i in range(rows)]
    pos = [(i * 29) % (200, 130)[i % 2] for i in range(rows)]
    q, qp = case.queries(rows)
    got = case.unpad(_absorbed(case, slot, pos, qp, 2))
    rows_close(got, case.want(q, slot, pos), 1e-5, name)
    pos[3] = -1  # an idle row's output is nothing
    got = case.unpad(_absorbed(case, slot, pos, qp, 2))
    assert not got[3].any() and torch.isfinite(got).all()


@pytest.mark.parametrize("name", ["pool8", "pool12", "sink_wide", "sigmoid", "sigmoid_bare"])
def test_paged_attention_of_many_rows(name):
    """Rows of a sequence that share a workgroup, workgroups in which one sequence ends and another begins, groups that do
    not divide a tile's columns."""
    from test_dumizen_gpu import SPECS, Case
    case = Case(SPECS[name], [401, 301, 31], torch.float32)
    got = {0: [], 1: [], 2: []}
    for parts in ([(0, 399), (1, 300), (2, 29)], [(2, 1), (0, 1)], [(0, 1), (1, 1), (2, 1)]):
        for i, o in case.step(parts).items():
            got[i].append(o)
    for i in range(3):
        rows_close(torch.cat(got[i]).flatten(1), case.want(i).flatten(1), 1e-5, f"{name}: {i}")


@pytest.mark.parametrize("name", ["sink", "sigmoid"])
def test_paged_attention_behind_the_first_64_pages(name):
    """Single rows of a sequence whose page table is longer than what a wave reads of it at once, beside a short one."""
    from test_dumizen_gpu import SPECS, Case
    case = Case(SPECS[name], [4163, 70], torch.float32)
    case.step([(0, 4094), (1, 60)])
    got = {0: [], 1: []}
    for parts in ([(0, 1), (1, 1)], [(1, 1), (0, 1)], [(0, 1)], [(0, 64), (1, 6)], [(0, 1), (1, 1)], [(0, 1)]):
        for i, o in case.step(parts).items():
            got[i].append(o)
    for i, first in ((0, 4094), (1, 60)):
        o = torch.cat(got[i]).flatten(1)
        rows_close(o, case.want(i).flatten(1)[first:first + len(o)], 1e-5, f"{name}: {i}")


def _engine_with_a_parted_head(slots):
    """One layer of a real width; 40 rows of its head are 64 tiles, whose K is shared out."""
    assert linear_f32_form(40, 4096, 2048) == (64, 64, 0, 4)
    import dataclasses
    from llm_sharding_amd.config import get_preset
    from llm_sharding_amd.runtime.registry import make_engine, random_source
    cfg = get_preset("deretar-2k")
    cfg = dataclasses.replace(cfg, layers=cfg.layers[:1], vocab_size=4096)
    return make_engine(cfg, 0, 1, torch.device(DEV, 0), torch.float32, has_embed=True, has_head=True, source=random_source(cfg, 3),
                       max_slots=slots, max_seq=16, max_prefill_rows=slots)


@torch.inference_mode()
def test_captured_heads_share_no_workspace(monkeypatch):
    """Two graphs with scratch sets of their own, side by side: the tokens and sums of each by itself, and those of an eager
    step; no workspace but the sets'."""
    from llm_sharding_amd.runtime.engine import DecodeGraph
    n, steps = 40, 6
    monkeypatch.setattr(hip, "_WS", {})
    eng = _engine_with_a_parted_head(2 * n)
    graphs = [DecodeGraph(eng, n, "full", slots=list(range(i * n, i * n + n)), scratch=i).capture() for i in range(2)]
    ids = torch.randint(3, 2048, (2, n), generator=torch.Generator().manual_seed(1), dtype=torch.int32).to(DEV)
    streams = [torch.cuda.Stream(), torch.cuda.Stream()]

    def run(together):
        eng.reset()
        got = [[], []]
        for i, g in enumerate(graphs):
            g.set_positions()
            g.tokens.copy_(ids[i])
        torch.cuda.synchronize()
        for _ in range(steps):
            for i, g in enumerate(graphs):
                with torch.cuda.stream(streams[i if together else 0]):
                    g.replay()
                    got[i].append((g.out_hidden.clone(), g.tokens.clone()))
        torch.cuda.synchronize()
        return got
    alone, both = run(False), run(True)
    for a, b in zip(alone[0] + alone[1], both[0] + both[1]):
        assert torch.equal(a[0], b[0]) and torch.equal(a[1], b[1])
    for i in range(2):
        for h, t in alone[i]:
            assert torch.equal(eng.head(h, list(range(n))).to(torch.int32), t)
    assert not hip._WS


@torch.inference_mode()
def test_positions_arrive_before_replays_of_other_streams():
    """Positions that a busy stream is yet to bring: a replay and a read of another stream come behind them."""
    from llm_sharding_amd.runtime.engine import DecodeGraph
    eng = _engine_with_a_parted_head(4)
    g = DecodeGraph(eng, 4, "full").capture()
    ids, busy, other = torch.tensor([5, 9, 11, 300], dtype=torch.int32, device=DEV), torch.cuda.Stream(), torch.cuda.Stream()
    outs = []
    for late in (False, True):
        eng.reset()
        g.set_positions()
        for _ in range(2):
            g.tokens.copy_(ids)
            g.replay()
        eng.advance([0, 1, 2, 3], [1] * 4)  # back by a token: the next replay is the second one again
        g.tokens.copy_(ids)
        torch.cuda.synchronize()
        with torch.cuda.stream(busy):
            if late:
                torch.cuda._sleep(20_000_000)
            g.set_positions()
        with torch.cuda.stream(other):
            g.replay()
            g.sync_positions()
        assert [eng.seq_len[i] for i in range(4)] == [2] * 4
        torch.cuda.synchronize()
        outs.append((g.out_hidden.clone(), g.tokens.clone()))
    assert torch.equal(outs[0][0], outs[1][0]) and torch.equal(outs[0][1], outs[1][1])


@pytest.mark.parametrize("n", [2048, 4096])  # streamed; in parts of K where there is a workspace
@torch.inference_mode()
def test_captured_product_without_a_workspace(n):
    """In a graph, a product that is given no workspace takes none: its replays may run beside others of any stream."""
    k, rows = 2048, 40
    assert linear_f32_form(rows, n, k)[3] == (4 if n == 4096 else 1)
    x, lin = _rand(rows, k, seed=1).to(DEV), Linear(_rand(n, k, seed=2, scale=k ** -0.5).to(DEV))
    out, want = torch.zeros(rows, n, device=DEV), torch.zeros(rows, n, device=DEV)
    lin(x, rows, want)
    before, s, g = set(hip._WS), torch.cuda.Stream(), torch.cuda.CUDAGraph()
    torch.cuda.synchronize()
    with torch.cuda.graph(g, stream=s):
        lin(x, rows, out)
    for _ in range(3):
        out.zero_()
        g.replay()
        rows_close(out, want.double().cpu(), 2 * sum_tol(k), "replay")
    assert set(hip._WS) == before


@pytest.mark.parametrize("name", ["one_group", "small", "wide_values"])
@pytest.mark.parametrize("loud", [False, True])
@pytest.mark.parametrize("n", [1030, 120])
def test_paged_attention_of_values_that_are_no_numbers(name, loud, n):
    """An infinity and a NaN among the values reach the rows that give their tokens a weight, and no other, also where rows
    share a workgroup: not those before, not those whose window has passed, and (``loud``) not those whose scores leave the
    tokens' weights at 0."""
    from test_gupuvik_gpu import SIZES, Case
    from llm_sharding_amd.ops import paged_attn as A
    s, bad = SIZES[name], [n // 5, n // 5 + 1]
    case = Case(s, [n], torch.float32)
    case.v[0][bad[0]], case.v[0][bad[1]] = float("inf"), float("nan")
    if loud:
        case.k[0][bad] *= 2000
    case.fill()
    q = _rand(n, s.heads, s.dim, seed=7)
    out = torch.full((n, s.heads * s.dvp), 9.0, device=DEV)
    A.plain(case.args([0] * n, list(range(n))), n, case.padded(q, s.dkp).to(DEV), None, out)
    got = case.unpad(out).double().cpu()
    i, j = torch.arange(n)[:, None], torch.arange(n)[None]
    see = (j <= i) & ((i - j < (s.window or n)) | (j < s.keep_first))
    k, v = (x.double().repeat_interleave(s.group, 1) for x in (case.k[0], case.v[0].nan_to_num(0, 0, 0)))
    sc = torch.einsum("ihd,jhd->hij", q.double(), k) * s.scale * case.temp.double()[:, None, None]
    if s.softcap:
        sc = s.softcap * torch.tanh(sc / s.softcap)
    sc = sc.masked_fill(~see, -float("inf"))
    far = (sc[..., bad] - sc.amax(-1, keepdim=True)).amax(-1).T  # the louder one's distance below the top
    none, some = far < -120, far > -80  # weights below 2^-150 are 0 in fp32, above 2^-126 they are not
    assert none.any() and some.any()
    want = torch.einsum("hij,jhd->ihd", torch.softmax(sc, -1), v)
    off = (got - want).norm(dim=-1) / want.norm(dim=-1)
    assert off[none].max() < 1e-5, f"{name}: {off[none].max():.2e}"
    assert not torch.isfinite(got[some]).any()


@pytest.mark.parametrize("name", ["one_group", "small", "wide_values"])
@pytest.mark.parametrize("bad", [5, 40, 70, 100])
def test_paged_attention_of_a_value_far_below_the_top(name, bad):
    """A token that outweighs all others leaves an infinity's weight at 0, also where another wave has it: its rows' sums are
    those without the infinity."""
    import dataclasses
    from test_gupuvik_gpu import SIZES, Case
    from llm_sharding_amd.ops import paged_attn as A
    s, n, top = dataclasses.replace(SIZES[name], softcap=0.0, window=0, keep_first=0), 128, 20
    case = Case(s, [n], torch.float32)
    q = torch.ones(n, s.heads, s.dim)
    case.k[0][top] = 2000 / s.scale / s.dim  # a score of 2000 times a head's factor
    case.k[0][bad] = 0
    case.fill()
    want = case.want(q, [0] * n, list(range(n)))
    case.v[0][bad] = float("inf")
    case.fill()
    out = torch.full((n, s.heads * s.dvp), 9.0, device=DEV)
    A.plain(case.args([0] * n, list(range(n))), n, case.padded(q, s.dkp).to(DEV), None, out)
    got = case.unpad(out).double().cpu()
    rows_close(got[max(top, bad):].flatten(1), want[max(top, bad):].flatten(1), 1e-5, f"{name}: {bad}")


@pytest.mark.parametrize("name", ["one_group", "small", "wide_values"])
def test_paged_attention_rounds_no_more_than_four_sums_a_score(name):
    """Large scores, whose rounding the softmax passes on: against float64 no further off than scores that are added up in fp32
    as four sums of every fourth value (what the plain kernel does), everything behind them in float64, and an eighth for
    that; a single sum is about twice as far."""
    import dataclasses
    from test_gupuvik_gpu import SIZES, Case
    from llm_sharding_amd.ops import paged_attn as A
    s, n = dataclasses.replace(SIZES[name], scale=10 * SIZES[name].scale, softcap=0.0), 400
    case = Case(s, [n], torch.float32).fill()
    q = _rand(n, s.heads, s.dim, seed=7)
    out = torch.full((n, s.heads * s.dvp), 9.0, device=DEV)
    A.plain(case.args([0] * n, list(range(n))), n, case.padded(q, s.dkp).to(DEV), None, out)
    got, want = case.unpad(out).double().cpu(), case.want(q, [0] * n, list(range(n)))
    i, j = torch.arange(n)[:, None], torch.arange(n)[None]
    see = (j <= i) & ((i - j < (s.window or n)) | (j < s.keep_first))
    k, v = (x.repeat_interleave(s.group, 1) for x in (case.k[0], case.v[0]))
    parts = torch.zeros(4, s.heads, n, n)
    for d in range(s.dim):
        parts[d % 4] += q[:, None, :, d].permute(2, 0, 1) * k[None, :, :, d].permute(2, 0, 1)
    sc = ((parts[0] + parts[1]) + (parts[2] + parts[3])) * case.hscale.cpu()[:, None, None]
    four = torch.einsum("hij,jhd->ihd", torch.softmax(sc.double().masked_fill(~see, -float("inf")), -1), v.double())
    ours, theirs = (float((x - want).norm() / want.norm()) for x in (got, four))
    print(f"{name}: {ours:.2e}, four sums a score {theirs:.2e}")
    assert ours < 1.125 * theirs


@torch.inference_mode()
def test_paged_attention_of_many_single_rows(monkeypatch):
    """One row of each of 130 sequences: the same from workgroups of a row each and from shared ones; a decode step asks for
    the former, a prompt's rows share."""
    from test_gupuvik_gpu import SIZES, Case
    from llm_sharding_amd.ops import paged_attn as A
    s, n = SIZES["wide_values"], 130
    case = Case(s, [1 + (37 * i) % 150 for i in range(n)], torch.float32).fill()
    slot, pos = list(range(n)), [x - 1 for x in case.lens]
    pos[5] = -1  # idle
    q = _rand(n, s.heads, s.dim, seed=7)
    live = [i for i in range(n) if pos[i] >= 0]
    want = case.want(q[live], live, [pos[i] for i in live])
    for singles in (False, True):
        out = torch.full((n, s.heads * s.dvp), 9.0, device=DEV)
        A.plain(case.args(slot, pos), n, case.padded(q, s.dkp).to(DEV), None, out, singles=singles)
        rows_close(case.unpad(out)[live].flatten(1), want.flatten(1), 1e-5, f"singles {singles}")
        assert not out[5].any()
    import dumizen_models as M
    from llm_sharding_amd.runtime.engine import DecodeGraph
    asked, plain = [], A.plain
    monkeypatch.setattr(A, "plain", lambda *a, singles=False: (asked.append(singles), plain(*a, singles=singles)))
    eng = M.engine(M.stack(), DEV, torch.float32)
    sl, po = eng.prefill_rows([0, 1], [9, 4])
    eng.forward(eng.embed(torch.arange(13, dtype=torch.int32, device=DEV)), sl, po)
    eng.advance([0, 1], [9, 4])
    assert asked and not any(asked)
    asked.clear()
    DecodeGraph(eng, 2, "first").capture()
    assert asked and all(asked)

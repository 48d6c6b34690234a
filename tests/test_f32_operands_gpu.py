"""What fp32 products of an engine do with their operands, on the GPU against float64: they keep all 24 bits of every value, whatever stands
beside it in its row or column, and take weights as they are when they are called."""
import pytest
import torch

from llm_sharding_amd.models.stack import RELU2, MoeSpec
from llm_sharding_amd.ops import moe as X
from llm_sharding_amd.ops.packing import pack_f32
from llm_sharding_amd.ops.stream import Linear

pytestmark = pytest.mark.gpu
DEV = "cuda"
# Streamed weights, tiles of every size, in parts of K and whole
PRODUCTS = [(8, 2048, 2048), (64, 2048, 2048), (100, 4096, 1024), (300, 4224, 2048), (505, 2176, 2176), (963, 8192, 2048), (257, 4096, 8704)]


def _rand(*shape, seed=0, scale=1.0):
    return (torch.randn(*shape, generator=torch.Generator().manual_seed(seed)) * scale).to(DEV)


def linear(x, w, factor=1.0):
    """x w^T as an engine makes it; ``factor``: what the weights are multiplied by in place, once a first product is made."""
    lin, out = Linear(w), torch.zeros(x.shape[0], -(-w.shape[0] // 128) * 128, device=DEV)
    lin(x, x.shape[0], out)
    if factor != 1.0:
        lin.w.mul_(factor)
        lin(x, x.shape[0], out.zero_())
    return out[:, :w.shape[0]]


def off(got, want):
    return float((got.double() - want).norm() / want.norm())


def off_tol(k):
    """A sum is rounded at most once for 16 k, partial sums grow as the root of their number: each rounding is off by 2^-24 / 3^0.5 of its
    value on average, together by the root of k / 32 times that."""
    return 2.0 ** -24 / 3 ** 0.5 * (k / 32) ** 0.5


@pytest.mark.parametrize("rows,n,k", PRODUCTS)
@pytest.mark.parametrize("place", ["weights", "rows"])
def test_single_values_keep_all_their_bits(rows, n, k, place):
    """Rows of one power of two give weights bit for bit; columns of one give the rows' values."""
    x, w = _rand(rows, k, seed=1), _rand(n, k, seed=2, scale=k ** -0.5)
    m, one = (rows, x) if place == "weights" else (n, w)
    at = (torch.arange(m, device=DEV) * 997 + 5) % k
    size = torch.exp2((torch.arange(m, device=DEV) % 40 - 20).float())
    one.zero_()
    one[torch.arange(m, device=DEV), at] = size
    want = (w[:, at] * size).T if place == "weights" else x[:, at] * size
    assert torch.equal(linear(x, w), want)


@pytest.mark.parametrize("rows,n,k", PRODUCTS)
@pytest.mark.parametrize("depth", [0, 20, 24, 30, 41, 60])
@pytest.mark.parametrize("place", ["row", "column"])
def test_small_values_that_alone_count(rows, n, k, depth, place):
    """A sixteenth of a row, 2^-depth as large as the rest of it, which meets zeros."""
    x, w = _rand(rows, k, seed=1), _rand(n, k, seed=2, scale=k ** -0.5)
    few = k // 16 - 8
    of, other = (x, w) if place == "row" else (w, x)
    of[:, :few] *= 2.0 ** -depth
    other[:, few:] = 0
    want = x[:, :few].double() @ w[:, :few].double().T
    assert off(linear(x, w), want) < off_tol(k)


@pytest.mark.parametrize("place", ["row", "column"])
@pytest.mark.parametrize("rows", [8, 300])
def test_one_value_far_above_the_others(rows, place):
    """One value 2^30 times as large as the others, which are all that counts."""
    x, w = _rand(rows, 2048, seed=1), _rand(4112, 2048, seed=2, scale=2048 ** -0.5)
    (x if place == "row" else w)[7, 9] = 2.0 ** 30
    (w if place == "row" else x)[:, 9] = 0
    want = x.double() @ w.double().T
    got = linear(x, w)
    at = (7, slice(None)) if place == "row" else (slice(None), 7)
    assert off(got, want) < off_tol(2048) and off(got[at], want[at]) < 2 * off_tol(2048)


def test_rows_and_columns_of_very_different_sizes():
    x, w = _rand(300, 2048, seed=1), _rand(4112, 2048, seed=2, scale=2048 ** -0.5)
    g = torch.Generator().manual_seed(3)
    x *= torch.exp2(torch.randint(-90, 60, (300, 1), generator=g).float()).to(DEV)
    w *= torch.exp2(torch.randint(-30, 30, (4112, 1), generator=g).float()).to(DEV)
    want = x.double() @ w.double().T
    got = (linear(x, w).double() - want).abs() / (x.double().norm(dim=1)[:, None] * w.double().norm(dim=1)[None])
    assert got.max() < 2.0 ** -22  # of every value by itself: some six times the root mean square


@pytest.mark.parametrize("rows,n,k", PRODUCTS)
@pytest.mark.parametrize("factor", [8.0, 2.0 ** -7, 2.0 ** -20, 2.0 ** -30, 2.0 ** -60])
def test_weights_changed_in_place(rows, n, k, factor):
    """Weights times a power of two give results times a power of two, bit for bit, also where a product was made of the former ones."""
    x, w = _rand(rows, k, seed=1), _rand(n, k, seed=2, scale=k ** -0.5)
    assert torch.equal(linear(x, w, factor), linear(x, w) * factor)


@pytest.mark.parametrize("rows,experts,ff,width", [(400, 16, 1024, 1024), (2400, 8, 512, 1024), (900, 32, 1024, 2048)])
def test_experts_weights_changed_in_place(rows, experts, ff, width):
    """The same of experts' products, as an engine's feed-forward makes them: up and down times a power of two."""
    from llm_sharding_amd.runtime.feed_forward import Moe
    spec, e = MoeSpec(experts, 2, ff, act=RELU2), range(experts)
    t = {"router": _rand(experts, width, seed=3)}
    t.update({f"e{i}.up": _rand(ff, width, seed=10 + i, scale=width ** -0.5) for i in e})
    t.update({f"e{i}.down": _rand(width, ff, seed=100 + i, scale=ff ** -0.5) for i in e})
    moe = Moe(spec, t, True)
    h, logits, flat = _rand(rows, width, seed=1), _rand(rows, experts, seed=2), {}

    class Eng:
        def scratch_view(self, name, n, k):
            m, kind = sizes[name] if isinstance(sizes[name], tuple) else (sizes[name], torch.float32)
            return flat.setdefault(name, torch.zeros(rows * m, dtype=kind, device=DEV))[:n * k].view(n, k)
    sizes, eng = moe.scratch(), Eng()

    def results():
        ye, weight, place, top = moe.forward(eng, h, None, logits, {"router": 0}, None, rows)["experts"]
        return ye[place.long()].view(rows, top, -1), weight.view(rows, top).clone()
    before, weight = results()
    score, at = logits[:8].double().topk(2)
    assert torch.allclose(weight[:8].double(), torch.softmax(score, -1), atol=1e-6)
    for r in range(8):
        for j in range(2):
            up = h[r].double() @ t[f"e{at[r, j]}.up"].double().T
            want = up.relu().square() @ t[f"e{at[r, j]}.down"].double().T
            assert off(before[r, j], want) < 4 * off_tol(width)
    moe.experts.up.mul_(2.0 ** -20)
    moe.experts.down.mul_(2.0 ** -10)
    assert torch.equal(results()[0], before * 2.0 ** -50)


@pytest.mark.parametrize("rows,each", [(64, 100), (128, 260), (128, 18)])
@pytest.mark.parametrize("up", [X.GLU, X.RELU2, X.DOWN])
@pytest.mark.parametrize("wide", [False, True])
def test_experts(rows, each, up, wide):
    """Experts' tiles, counts that fill none; a row of which a part is much smaller: against float64."""
    E, top, k, n = 5, 2, 2048, 2080
    pairs = E * each
    g = torch.Generator().manual_seed(5)
    expert = torch.randint(0, E, (pairs,), generator=g, dtype=torch.int32)
    a, w = _rand(pairs // top if up else pairs, k, seed=1), _rand(E, n, k, seed=2, scale=k ** -0.5)
    if wide:
        a[11, :300] *= 2.0 ** -20
    wd = torch.stack([pack_f32(v) for v in w])
    order, place = (torch.zeros(pairs, dtype=torch.int32, device=DEV) for _ in range(2))
    tiles = torch.zeros(8 * pairs, dtype=torch.int32, device=DEV)
    nt = X.group(expert.to(DEV), pairs, E, rows, order, place, tiles)
    at, of = order.long().cpu(), expert[order.long().cpu()]
    want = torch.stack([w[int(e)].double() @ a[int(i) // top if up else j].double() for j, (i, e) in enumerate(zip(at, of))])
    if up == X.GLU:
        v = want.view(pairs, -1, 2, 16)
        want = (torch.nn.functional.silu(v[:, :, 0]) * v[:, :, 1]).flatten(1)
    elif up == X.RELU2:
        want = want.relu().square()
    out = torch.full((pairs, want.shape[1]), 7.0, device=DEV)
    X.gemm(tiles, nt, rows, order, top, a, wd, n, k, out, pairs, up)
    assert off(out, want) < 2 * off_tol(k)

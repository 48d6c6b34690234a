"""Row tables of a forward pass: how host numbers are read and sent, and prefill's query tiles against a plain walk."""
import random

import numpy as np
import pytest
import torch

from llm_sharding_amd.ops import hip, packing


def plain_tiles(slot, pos, kv_len, tile_rows):
    tiles, r, n = [], 0, len(slot)
    while r < n:
        e = r + 1
        while (e < n and slot[e] == slot[r] and pos[e] == pos[e - 1] + 1 and e - r < tile_rows
               and (kv_len is None or kv_len[e] == kv_len[r])):
            e += 1
        tiles.append([r, e - r, slot[r], pos[r], pos[e - 1] + 1 if kv_len is None else kv_len[r], 0, 0, 0])
        r = e
    return torch.tensor(sorted(tiles, key=lambda t: -t[4]), dtype=torch.int32)


@pytest.mark.parametrize("kind", [list, tuple, torch.tensor, np.array])
def test_prefill_tiles(kind):
    rng = random.Random(5)
    for case in range(40):
        slot, pos, kv = [], [], []
        for _ in range(rng.randint(1, 6)):  # runs, some joining the one before, some of the same slot elsewhere
            s, p, n, k = rng.randint(0, 2), rng.choice([0, 3, pos[-1] + 1 if pos else 0]), rng.randint(1, 50), rng.choice([60, 70])
            slot, pos, kv = slot + [s] * n, pos + list(range(p, p + n)), kv + [k] * n
        for tile_rows in (1, 16, 128):
            for kvl in (None, kv):
                got = hip.build_prefill_tiles(kind(slot), kind(pos), None if kvl is None else kind(kvl), tile_rows=tile_rows)
                assert torch.equal(got, plain_tiles(slot, pos, kvl, tile_rows)), (case, tile_rows)
    assert hip.build_prefill_tiles([], []).numel() == 0


def test_host_numbers_are_read_as_before():
    for x in ([], [3, 1, 2], (4, 5), [True, False], [torch.tensor(7), 8], [2.0, 3.9], np.array([1, 2], dtype=np.int16),
              torch.tensor([5, 6]), range(4)):
        want = torch.tensor([int(v) for v in x], dtype=torch.int32)
        got = hip.to_device(x, "cpu")
        assert torch.equal(got, want) and got.dtype == torch.int32
        assert hip.host_ints(x).tolist() == want.tolist()
    rows = [(0, 3, 1, 5), (3, 1, 0, 0)]
    assert torch.equal(hip.to_device(rows, "cpu"), torch.tensor(rows, dtype=torch.int32))
    assert hip.host_ints(rows).tolist() == [list(r) for r in rows]
    with pytest.raises(TypeError):
        hip.host_ints(3)


@pytest.mark.parametrize("x", [2 ** 31, 2 ** 32 + 1, -2 ** 31 - 1, 2 ** 70])
def test_numbers_past_32_bits_are_refused(x):
    """A position that int32 does not hold is an error as it is for torch, not another position."""
    with pytest.raises((RuntimeError, OverflowError, ValueError)):
        torch.tensor([x], dtype=torch.int32)
    for rows in ([x], [3, x, 5]):
        with pytest.raises((RuntimeError, OverflowError, ValueError)):
            hip.to_device(rows, "cpu")
        with pytest.raises((RuntimeError, OverflowError, ValueError)):
            hip.to_device(hip.host_ints(rows), "cpu")
        with pytest.raises((RuntimeError, OverflowError, ValueError)):
            hip.build_prefill_tiles([0] * len(rows), rows)
    for bad in (float("nan"), float("inf")):
        for rows in ([bad], np.array([1.0, bad]), torch.tensor([bad])):
            with pytest.raises((RuntimeError, OverflowError, ValueError)):
                hip.host_ints(rows)
    assert hip.to_device(np.array([2 ** 31 - 1, -2 ** 31]), "cpu").tolist() == [2 ** 31 - 1, -2 ** 31]


def test_remembered_candidates_are_not_shared():
    a = packing.coop_candidates(768, 4096, 64)
    a.append("more")
    assert "more" not in packing.coop_candidates(768, 4096, 64)
    assert all(packing.coop_allowed(c, 768, 4096, 64) for c in a[:-1]) and not packing.coop_allowed(a[0], 768, 4096, 16)
    b = packing.gemv_candidates(768, 4096, 8)
    b.clear()
    assert packing.gemv_candidates(768, 4096, 8)


def test_sent_numbers_fill_their_places():
    """As many int32 as there are places, on the way that takes no launch as on the others."""
    out = torch.full((2, 3), -5, dtype=torch.int32)
    hip.send([4, 5, 6], out[0])
    hip.send(np.array([7]), out[1, 2:])
    hip.send([], out[1, :0])
    assert out.tolist() == [[4, 5, 6], [-5, -5, 7]]
    hip.send(list(range(6)), out.t())  # places in the order of the shape
    assert out.t().flatten().tolist() == list(range(6))
    for x, to in (([1], out[0]), ([1, 2], out[0]), ([1, 2, 3], torch.zeros(3, dtype=torch.int64)), ([1.0], torch.zeros(1))):
        with pytest.raises(ValueError):
            hip.send(x, to)


@pytest.mark.parametrize("slot,pos", [([0, 0, 0], [0, 1, 2]), ([[0], [0], [0]], torch.tensor([[0], [1], [2]])),
                                      (torch.zeros(1, 3), np.array([[0, 1, 2]])), (range(0, 1), 0), (torch.tensor(0), (0,))])
def test_rows_of_a_stack_in_any_shape(slot, pos):
    """Slots and positions come as lists, arrays or tensors, flat or not, one row also as a number."""
    from deretar_models import engine, stack
    eng = engine(stack(), "cpu", torch.float32)
    n = torch.as_tensor(pos).numel()
    h = eng.embed(torch.tensor([3, 4, 5][:n], dtype=torch.int32))
    got = eng.forward(h.clone(), slot, pos)
    eng.reset()
    assert torch.equal(got, eng.forward(h.clone(), [0] * n, list(range(n))))


@pytest.mark.gpu
def test_copies_are_not_overtaken():
    """Many copies in a row behind a busy stream, each from memory that the next ones may be given again, and on two streams."""
    a = torch.randn(4096, 4096, device="cuda")
    streams = [torch.cuda.current_stream(), torch.cuda.Stream()]
    got = []
    for i in range(300):
        with torch.cuda.stream(streams[i % 2]):
            if i % 10 < 2:
                a @ a
            got.append(hip.to_device([i] * (1 + i % 70), "cuda"))
    torch.cuda.synchronize()
    for i, t in enumerate(got):
        assert t.tolist() == [i] * (1 + i % 70)


@pytest.mark.gpu
def test_no_copy_from_the_host_inside_a_capture():
    """A graph would keep the address of pinned memory that the next tables are written to: refused, and the capture goes on."""
    x, g = torch.zeros(4, device="cuda"), torch.cuda.CUDAGraph()
    x += 0
    torch.cuda.synchronize()
    with torch.cuda.graph(g, stream=torch.cuda.Stream()):
        with pytest.raises(RuntimeError):
            hip.to_device([1, 2, 3], "cuda")
        with pytest.raises(RuntimeError):
            hip.to_device(torch.tensor([1, 2, 3]), "cuda")
        x += 1
    assert hip.to_device([1, 2, 3], "cuda").tolist() == [1, 2, 3]
    for _ in range(3):
        g.replay()
    assert x.tolist() == [3.0] * 4


@pytest.mark.parametrize("even", [False, True])
def test_coop_choice_without_a_table_entry(even, monkeypatch):
    """Every choice is a candidate, the same for all rows of a block (the workspace is sized at 32, 64 and 128 rows), and no
    dearer by the model than the smallest split that fills the chip."""
    monkeypatch.setattr(packing, "_TUNED", {})
    for n in (256, 512, 1040, 3072, 5120, 16384, 50688):
        for k in (512, 1024, 3072, 8192, 11008):
            for lo, hi in ((17, 32), (33, 64), (65, 128)):
                cands = packing.coop_candidates(n // 16, k, lo, even)
                if not any(c[3] >= 1 for c in cands):
                    continue
                algo, cfg = packing.proj_config(n // 16, lo, need_even=even, k=k)
                assert algo == "coop" and packing.coop_allowed(cfg, n // 16, k, hi, even)
                assert packing.proj_config(n // 16, hi, need_even=even, k=k) == (algo, cfg)
                floats, groups = packing.coop_workspace_need([(n, k)], hi, [(n, k)] if even else ())
                assert floats >= packing.coop_slab_floats(n, lo, *cfg[:4]) and groups >= n // 16 // (cfg[0] * cfg[1])
                full = [c for c in cands if c[0] == 1 and c[2] == cfg[2] and c[3] >= 1 and c[4] <= 2 and c[5] == 3]
                mb = packing.row_blocks(lo)
                assert all(packing.coop_cost(n // 16, k, mb, cfg) <= packing.coop_cost(n // 16, k, mb, c)
                           for c in full if c[3] <= 8)


def test_fp32_head_takes_the_workspace_of_its_scratch_set(monkeypatch):
    """A captured head is replayed beside other graphs: scratch of its own set, not what belongs to the capturing stream."""
    from types import SimpleNamespace
    from llm_sharding_amd.ops import stream
    from llm_sharding_amd.runtime.stack_engine import StackEngine
    got = {}

    class Head:
        n = 128

        def __call__(self, x, rows, out, **kw):
            got.update(kw)
    eng = SimpleNamespace(dtype=torch.float32, device="cpu", lm_head=Head(), head_vocab=100, head_v0=0, coop_ws=object(),
                          _normed=lambda h, rows, a_rows: h)
    monkeypatch.setattr(stream, "logits_argmax", lambda *a, **kw: None)
    StackEngine.head_gemv(eng, torch.zeros(4, 128), 4, torch.zeros(4, dtype=torch.int64))
    assert got.get("ws") is eng.coop_ws


@pytest.mark.parametrize("n,k", [(1152, 3072), (2304, 2048), (6144, 3072), (8192, 8192)])
def test_workspace_of_a_size_with_and_without_gates(n, k):
    """Two projections of one size, one of them gated: scratch for what either takes, by the table and by the cost model."""
    floats, groups = packing.coop_workspace_need([(n, k), (n, k)], 128, [(n, k)])
    for rows in (17, 32, 33, 64, 65, 128):
        for even in (False, True):
            algo, cfg = packing.proj_config(n // 16, rows, need_even=even, k=k)
            if algo == "coop":
                assert floats >= packing.coop_slab_floats(n, rows, *cfg[:4]) and groups >= n // 16 // (cfg[0] * cfg[1])


# us of products whose weights are 360 to 940 MB on MI355X, each read from memory: what the cost model chose before it knew
# that such weights push the activations out of L2, the smallest split that fills the chip, and the fastest that it may choose
LARGE = {
    (8192, 22016, 64): {(1, 2, 4, 1, 2, 3): 82.3, (1, 8, 8, 4, 1, 3): 70.3, (1, 4, 4, 2, 1, 3): 73.2, (1, 8, 4, 4, 1, 3): 66.4},
    (8192, 22016, 128): {(1, 4, 2, 2, 1, 3): 103.3, (1, 8, 4, 4, 1, 3): 80.3, (1, 8, 2, 4, 1, 3): 79.2},
    (8192, 28672, 64): {(1, 2, 4, 1, 2, 3): 101.7, (1, 8, 8, 4, 1, 3): 82.2, (1, 4, 4, 2, 1, 3): 86.1, (1, 8, 4, 4, 1, 3): 78.8},
    (8192, 28672, 128): {(1, 4, 2, 2, 1, 3): 129.6, (1, 8, 4, 4, 1, 3): 96.0, (1, 8, 2, 4, 1, 3): 98.7},
    (16384, 28672, 64): {(1, 2, 4, 1, 1, 3): 223.2, (1, 8, 8, 2, 1, 3): 147.5, (1, 4, 4, 1, 1, 3): 168.5, (1, 8, 4, 2, 1, 3): 145.7},
}


@pytest.mark.parametrize("n,k,rows", list(LARGE))
def test_coop_choice_of_large_products(n, k, rows, monkeypatch):
    """No slower than the smallest split that fills the chip by more than a box's products differ between runs (5 %)."""
    monkeypatch.setattr(packing, "_TUNED", {})
    us, cfg = LARGE[n, k, rows], packing.proj_config(n // 16, rows, k=k)[1]
    fills = next(c for c in packing.coop_candidates(n // 16, k, rows)
                 if c[:3] == (1, 8, 4 if rows > 64 else 8) and c[3] >= 1 and c[4:] == (1, 3) and n // 128 * c[3] >= 256)
    assert us[cfg] <= 1.05 * us[fills], (cfg, fills)


@pytest.mark.parametrize("experts,mean,cols,rows", [
    (8, 136, 1024, 64), (8, 208, 768, 64), (8, 250, 2048, 64), (8, 256, 2048, 128), (8, 640, 4096, 128), (32, 112, 4096, 64),
    (32, 113, 2048, 128), (32, 136, 1024, 128), (32, 400, 256, 64), (1, 5000, 1024, 64), (1, 5000, 1024 + 4096, 128), (64, 20, 4096, 32)])
def test_fp32_experts_have_large_tiles_where_these_fill_the_chip(experts, mean, cols, rows):
    from llm_sharding_amd.ops import moe
    assert moe.tile_rows(mean * experts, experts, True, cols) == rows
    assert moe.tile_rows(mean * experts, experts, True) == (128 if mean > 112 else rows)


@pytest.mark.parametrize("pairs,experts,rows,cols,narrow", [
    (320, 8, 64, 1024, True), (640, 8, 64, 1024, True), (896, 8, 64, 1024, False), (1400, 8, 64, 768, False), (328, 8, 64, 2048, False),
    (40, 1000, 64, 384, True), (40, 1000, 64, 448, False), (320, 8, 32, 1024, False), (5120, 8, 128, 1024, False)])
def test_fp32_experts_have_narrow_tiles_where_these_leave_cus(pairs, experts, rows, cols, narrow):
    from llm_sharding_amd.ops import moe
    assert moe.narrow_tiles(pairs, experts, rows, cols) == narrow


def test_stream_handle_with_and_without_the_raw_call(monkeypatch):
    """The raw handle of the current device's stream where torch has the call, the Stream object's elsewhere."""
    from types import SimpleNamespace
    monkeypatch.setattr(torch.cuda, "current_device", lambda: 3)
    monkeypatch.setattr(torch.cuda, "current_stream", lambda: SimpleNamespace(cuda_stream=7))
    monkeypatch.setattr(torch._C, "_cuda_getCurrentRawStream", lambda d: 100 + d, raising=False)
    assert hip._stream().value == 103
    monkeypatch.delattr(torch._C, "_cuda_getCurrentRawStream")
    assert hip._stream().value == 7


@pytest.mark.gpu
@pytest.mark.parametrize("n", [1, 63, 64, 895, 896, 897, 1792, 1793, 5000])
def test_small_tables_are_kernel_arguments(n):
    """As lists, arrays and tensors, into tensors of their own and into part of another; numbers past 32 bits are refused."""
    x = np.random.default_rng(n).integers(-2 ** 31, 2 ** 31, n)
    for kind in (list, lambda v: v, torch.from_numpy, lambda v: torch.from_numpy(v).to(torch.int32)):
        got = hip.to_device(kind(x), "cuda")
        assert got.dtype == torch.int32 and got.is_cuda and got.tolist() == x.tolist()
    table = torch.full((3, n + 7), -5, dtype=torch.int32, device="cuda")
    hip.send(x.tolist(), table[1, 4:n + 4])
    assert table[1, 4:n + 4].tolist() == x.tolist()
    table[1, 4:n + 4] = -5
    assert bool((table == -5).all())
    with pytest.raises(RuntimeError):
        hip.send([2 ** 31] + [0] * (n - 1), table[1, 4:n + 4])


@pytest.mark.gpu
@pytest.mark.parametrize("runs", [1, 2, 3, 64, 255, 256, 257, 297, 298, 299, 700])
def test_row_tables_from_runs(runs):
    """Rows in as many runs of a slot's consecutive positions as one launch takes, and more; neighbouring runs of one slot."""
    g = np.random.default_rng(runs)
    slot, pos = [], []
    for i in range(runs):
        n, p = int(g.integers(1, 9 if runs > 3 else 900)), int(g.integers(0, 5000))
        slot += [i // 2] * n
        pos += range(p, p + n)
    s, p = hip.row_tables(np.array(slot), np.array(pos), "cuda")
    assert s.dtype == p.dtype == torch.int32 and s.is_contiguous() and p.is_contiguous()
    assert s.tolist() == slot and p.tolist() == pos
    with pytest.raises(RuntimeError):
        hip.row_tables(np.array([0, 0]), np.array([5, 2 ** 31]), "cuda")


def test_expert_tables_too_long_for_a_picked_height():
    """The sorting kernel takes 2^19 - 1 tiles with heights; longer tables have tiles of 256 rows, as without them."""
    from llm_sharding_amd.ops import moe as X
    products = (512, 256), (256, 256)
    most = ((1 << 19) - 1 - 32) * 128
    assert X.heights(most, 32, 256, False, *products) is not None and X.heights(most + 128, 32, 256, False, *products) is None
    assert X.max_tiles(most + 128, 32, 256) <= 1 << 20  # (of the experts' products)
    for rows, f32, cols in ((64, False, 512), (256, True, 512), (256, False, 640)):
        assert X.heights(4096, 32, rows, f32, (cols, 256), (256, 256)) is None

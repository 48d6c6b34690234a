"""gemm_sk's work-decomposition planner (ops/hip.py gemm_sk_plan): measured winners from
ops/gemm_sk_tuning.json (scripts/tune_gemm_sk.py) for tuned shapes, the cost model elsewhere;
every plan is one the kernel accepts (N tiles by bn, one workgroup per CU)."""
from llm_sharding_amd.ops import hip


def test_tuned_shapes_use_the_table():
    tab = hip._sk_tuned()
    assert tab, "ops/gemm_sk_tuning.json missing or empty"
    for (N, K), rows in tab.items():
        for M, cfg in rows:
            assert hip.gemm_sk_plan(M, N, K) == (cfg[0], hip.N_CU, cfg[2], cfg[3], cfg[4] if len(cfg) > 4 else 256)


def test_nearest_measured_m_with_same_row_tiles():
    tab = hip._sk_tuned()
    rows = dict(tab[(4096, 4096)])
    # 500 rows -> four 128-row tiles: the M=512 entry, never the M=384 or M=640 one
    got = hip.gemm_sk_plan(500, 4096, 4096)
    want = rows[512]
    assert got == (want[0], hip.N_CU, want[2], want[3], want[4] if len(want) > 4 else 256)


def test_cost_model_for_untuned_shapes():
    for M, N, K in [(65536, 12288, 4096), (300, 5120, 3072), (4096, 128, 64)]:
        bn, grid, dp, split, bm = hip.gemm_sk_plan(M, N, K)
        assert bn in (128, 192, 256) and N % (16 if bn == 192 else bn) == 0 and grid == hip.N_CU and split >= 0
        assert bm in (128, 256)
        assert hip.gemm_sk_plan(M, N, K, tuned=False) == (bn, grid, dp, split, bm) or (N, K) in hip._sk_tuned()


def test_gemm_wr_route(monkeypatch):
    """hip.gemm sends a qkv projection to gemm_wr.hip only inside its measured row ranges
    (hip.WR_ROUTES); everything else, and LSA_GEMM_WR=0, stays on gemm_sk."""
    monkeypatch.delenv("LSA_GEMM_WR", raising=False)
    ep = hip.EpiArgs()
    assert hip.gemm_wr_plan(512, 12288, 4096, hip.EPI_QKV, ep) == 192
    assert hip.gemm_wr_plan(448, 12288, 4096, hip.EPI_STORE, ep) == 192
    assert hip.gemm_wr_plan(384, 12288, 4096, hip.EPI_QKV, ep) == 192
    assert hip.gemm_wr_plan(384, 15360, 5120, hip.EPI_QKV, ep) == 192   # 13B
    assert hip.gemm_wr_plan(512, 15360, 5120, hip.EPI_QKV, ep) == 256
    assert hip.gemm_wr_plan(512, 5120, 3072, hip.EPI_QKV, ep) == 128    # 3B
    assert hip.gemm_wr_plan(512, 16384, 3072, hip.EPI_SWIGLU, ep) == 256  # 3B gate_up
    assert hip.gemm_wr_plan(447, 12288, 4096, hip.EPI_STORE, ep) is None  # last row tile < half full
    assert hip.gemm_wr_plan(319, 12288, 4096, hip.EPI_STORE, ep) is None
    assert hip.gemm_wr_plan(256, 12288, 4096, hip.EPI_QKV, ep) == 128   # 2 row tiles
    assert hip.gemm_wr_plan(256, 16384, 3072, hip.EPI_SWIGLU, ep) == 128
    for M, N, K, epi in [(192, 12288, 4096, hip.EPI_QKV),   # below the measured range
                         (513, 12288, 4096, hip.EPI_QKV),   # above it
                         (512, 12288, 4096, hip.EPI_SWIGLU),
                         (512, 4096, 4096, hip.EPI_RESID),
                         (384, 10240, 8192, hip.EPI_QKV),   # 70B qkv: measured a tie, not routed
                         (1024, 6144, 4096, hip.EPI_QKV),   # never measured
                         (512, 22016, 4096, hip.EPI_SWIGLU),
                         (128, 5120, 3072, hip.EPI_QKV),    # 3B below its range
                         (512, 12288, 4160, hip.EPI_QKV)]:  # another K
        assert hip.gemm_wr_plan(M, N, K, epi, ep) is None, (M, N, K, epi)
    monkeypatch.setenv("LSA_GEMM_WR", "0")
    assert hip.gemm_wr_plan(512, 12288, 4096, hip.EPI_QKV, ep) is None


def test_cost_model_takes_the_cheapest_of_what_the_kernel_accepts():
    """Odd sizes: tiles that divide the columns, splits that fit the grid and the K steps, no 192-wide tiles where a wave's
    64 columns are reduced."""
    for M in (129, 257, 300, 1256, 7970):
        for N, K in ((128, 64), (384, 128), (5120, 3072), (16384, 3072), (6208, 4096)):
            for whole64 in (False, True):
                if N % 128 and whole64:
                    continue
                bn, grid, dp, split, bm = hip.gemm_sk_plan(M, N, K, tuned=False, whole64=whole64)
                rem = -(-M // bm) * -(-N // bn) % hip.N_CU
                assert (bm, bn) in hip.SK_COST and N % (16 if bn == 192 else bn) == 0 and not (whole64 and bn == 192)
                assert grid == hip.N_CU and dp == 1 and 0 <= split <= min(8, max(1, K // 64))
                assert rem * split <= hip.N_CU and (rem or split == 0)
                cost = hip.gemm_sk_cost(M, N, K, bm, bn, split)
                for b in (x for x in hip.SK_COST if N % (16 if x[1] == 192 else x[1]) == 0 and not (whole64 and x[1] == 192)):
                    assert cost <= hip.gemm_sk_cost(M, N, K, *b, 1) + 1e-6


def test_choice_is_no_slower_than_the_one_of_two_heights():
    """Every product that the model was fitted to and the planner is asked for (gemm_wr has some), by its measured times
    (profiles/cost_gemm_sk.csv): against the choice of the model before, of tiles of 128 and 256 rows, none takes more than 1.05 times
    as long, and all 378 together take 0.984 of it at most."""
    import csv
    import math
    import os
    tiles = {(256, 256): (1.39, 6.3), (256, 192): (1.12, 4.7), (256, 128): (0.83, 2.9),
             (128, 256): (0.85, 2.9), (128, 192): (0.72, 2.4), (128, 128): (0.55, 1.5)}

    def before(M, N, K, bm, bn, split):
        (step, own), nkt, slab = tiles[(bm, bn)], K // 64, bm * bn * 4 / 1e5
        rounds, rem = divmod(-(-M // bm) * -(-N // bn), 256)
        us = 5.5 + rounds * (nkt * step + own)
        if rem and split:
            us += -(-nkt // split) * step * (1 - 0.36 * (1 - min(256, rem * split) / 256)) + own
            us += 2.1 + 1.5 * slab * (split if split > 2 else 1) if split > 1 else 0
        elif rem:
            us += rem * nkt / 256 * step * 1.6 + own * max(1.0, rem / 256) + 2.1 + 1.5 * slab * min(max(256 / rem, 1.0), 8.0)
        return max(us, 5.5 + N * K * 2 / 5e6)
    times = {}
    with open(os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "profiles", "cost_gemm_sk.csv")) as fh:
        for r in csv.DictReader(fh):
            times.setdefault(tuple(int(r[c]) for c in "mnk"), {})[int(r["bm"]), int(r["bn"]), int(r["split"])] = float(r["us"])
    ratio = {}
    for (M, N, K), t in times.items():
        bn, _, _, split, bm = hip.gemm_sk_plan(M, N, K, tuned=False)
        if -(-M // bm) * -(-N // bn) % hip.N_CU == 0:
            split = 1
        old = min((c for c in t if c[:2] in tiles), key=lambda c: before(M, N, K, *c))
        ratio[M, N, K] = t[bm, bn, split] / t[old]
    assert len(ratio) == 378
    asked = {k: r for k, r in ratio.items() if hip.gemm_wr_plan(*k, hip.EPI_STORE, hip.EpiArgs()) is None}
    assert max(asked.values()) <= 1.05, sorted(asked.items(), key=lambda x: -x[1])[:5]
    assert math.exp(sum(map(math.log, ratio.values())) / len(ratio)) <= 0.984


def test_an_entry_is_taken_where_it_is_the_nearest_measured(monkeypatch):
    """Of the rows with as many tiles of 128: entries at both ends, one of which says that the model's choice stands."""
    hip.gemm_sk_plan.cache_clear()
    monkeypatch.setattr(hip, "_SK_TUNED", {(4096, 11008): [(256, (128, 256, 1, 6, 256))]})
    monkeypatch.setattr(hip, "_SK_MODELLED", {(4096, 11008): [160, 384]})
    try:
        for M in (129, 160, 207):
            assert hip.gemm_sk_plan(M, 4096, 11008) == hip.gemm_sk_plan(M, 4096, 11008, tuned=False) != (128, 256, 1, 6, 256), M
        for M in (208, 256):
            assert hip.gemm_sk_plan(M, 4096, 11008) == (128, 256, 1, 6, 256), M
        for M in (128, 257):  # other numbers of tiles
            assert hip.gemm_sk_plan(M, 4096, 11008) == hip.gemm_sk_plan(M, 4096, 11008, tuned=False)
    finally:
        hip.gemm_sk_plan.cache_clear()


def test_residual_projections_of_few_row_tiles_at_both_ends():
    """Rows whose plan was another entry's, measured at its other end: 7B's and 70B's residual projections."""
    for M, N, K in [(129, 4096, 11008), (160, 4096, 11008), (257, 4096, 4096), (288, 4096, 4096), (513, 8192, 8192), (544, 8192, 8192)]:
        assert hip.gemm_sk_plan(M, N, K, whole64=True) == hip.gemm_sk_plan(M, N, K, tuned=False, whole64=True)
    assert hip.gemm_sk_partial_plan(160, 8192, 28672) == (256, 7) and hip.gemm_sk_partial_plan(256, 8192, 28672) is None
    assert hip.gemm_sk_partial_plan(512, 8192, 28672) == (256, 4) and hip.gemm_sk_partial_plan(400, 8192, 28672) is None


def test_counters_lie_as_the_kernel_has_them():
    import os
    import re
    root = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
    with open(os.path.join(root, "csrc", "kernels", "handoff.h")) as fh:
        assert int(re.search(r"constexpr int HO_STRIDE = (\d+);", fh.read()).group(1)) == hip.HANDOFF_STRIDE

"""Times behind three choices that the kernels make from sizes, MI355X, in a graph:

heights  the experts' two bf16 products in tiles of each height and of the one that the sorting kernel picks (ops/moe.py pick), over lists
         of experts' pairs: profiles/cost_moe_bf16.csv
scan     the delta rule's chunks and scan, by the scan's workgroups (csrc/kernels/delta_chunk.hip lsa_delta_chunked): with the library as
         it is, and with builds whose rule is fixed to 32 or 64 value channels a workgroup
order    flash prefill and paged prompt attention of one and of several prompts, by heads and their dimensions (csrc/kernels/common.h
         pair_up): with the library as it is, and with a build whose pair_up returns its argument

usage: [LSA_KERNELS_SO=a build] choices.py heights|scan|order NAME     (a line of csv a case on stdout; NAME: the build's, in it)"""
import os
import random
import sys

import torch

sys.path.insert(0, os.path.dirname(os.path.dirname(os.path.abspath(__file__))))
from llm_sharding_amd.ops import hip  # noqa: E402
from scripts.bench_kernels import timeit  # noqa: E402

DEV = "cuda"


def us(fn, reps):
    return min(timeit(fn, reps, 3) for _ in range(2))


def heights(name):
    from llm_sharding_amd.ops import moe as X
    print("build,experts,width,ff,top,mean,skew,us_128,us_192,us_256,us_320,us_two_heights,us_picked,picked")
    for E, ff, W, top in ((32, 1024, 2048, 8), (16, 1024, 2048, 4), (64, 512, 2048, 8), (8, 4096, 4096, 2)):
        up, down = (torch.randn(E, n, k, device=DEV).mul_(0.02).bfloat16() for n, k in ((2 * ff, W), (W, ff)))
        for mean in (200, 260, 330, 400, 500, 600, 700, 797, 900, 1100, 1500):
            for skew in (0.0, 0.3):
                g = torch.Generator().manual_seed(mean)
                rows = mean * E // top
                pairs = rows * top
                e = (torch.randn(rows, E, generator=g) + skew * torch.randn(E, generator=g)).topk(top, -1).indices
                e = e.to(torch.int32).reshape(-1).to(DEV)
                h = torch.randn(rows, W, device=DEV).bfloat16()
                act, ye = (torch.empty(pairs, n, device=DEV, dtype=torch.bfloat16) for n in (ff, W))
                order, place, spare = (torch.zeros(pairs, dtype=torch.int32, device=DEV) for _ in range(3))
                tiles = torch.empty(4 * X.max_tiles(pairs, E, 128), dtype=torch.int32, device=DEV)
                pick = X.pick((2 * ff, W), (W, ff))

                def both(tr, hs, i=0):
                    n = X.group(e, pairs, E, tr or 128, order, place, tiles, spare, hs)
                    X.gemm(tiles, n, tr, order, top, h, up, 2 * ff, W, act, pairs, X.GLU)
                    X.gemm(tiles, n, tr, order, top, act, down, W, ff, ye, pairs, X.DOWN)
                t = []
                for i in range(4):
                    only = X.Pick(pick.nt)
                    for j in range(4):
                        only.step[j], only.own[j] = ((1.0, 1.0), 1.0) if i == j else ((1e6, 1e6), 1e6)
                    t.append(us(lambda _: both(0, only), 6))
                # the host's choice by the mean, before: 128 rows up to 320 pairs an expert and 256 above
                two = us(lambda _: both(128 if pairs <= 320 * E else 256, None), 6)
                picked = us(lambda _: both(0, pick), 6)
                print(name, E, W, ff, top, mean, skew, *(round(x, 1) for x in (*t, two, picked)),
                      X.HEIGHTS[int(tiles[3]) >> 24], sep=",", flush=True)


def scan(name):
    from llm_sharding_amd.models.stack import DeltaSpec
    from llm_sharding_amd.ops import delta as D
    print("build,heads,dim,vdim,runs,rows,workgroups_of_32,us")
    for heads, dim, vdim in ((16, 128, 128), (32, 128, 128), (16, 64, 128), (64, 128, 64)):
        for runs in (1, 2, 3, 4, 5, 6, 8, 12):
            s = DeltaSpec(heads, heads // 4, dim, vdim, 4, 8, 8, dim ** -0.5, 1e-6)
            n, dk, dv = 1088, *s.state_dims
            rows = runs * n
            w = dict(conv=torch.randn(s.channels, s.taps), decay=torch.rand(heads), dt_bias=torch.randn(heads * dim),
                     norm=torch.ones(vdim))
            w = {k: v.to(DEV) for k, v in w.items()}
            state = tuple(torch.zeros(*x, device=DEV) for x in D.state_shapes(s, runs))
            kc, vc = s.kv_heads * s.dim, heads * vdim
            x = torch.randn(rows, 2 * kc + vc, device=DEV).bfloat16()
            in32, z = torch.randn(rows, heads, device=DEV), torch.randn(rows, heads * dim, device=DEV)
            gate, out = (torch.zeros(rows, vc, device=DEV, dtype=torch.bfloat16) for _ in range(2))
            table = torch.zeros(runs, 64, dtype=torch.int32, device=DEV)
            host = torch.tensor([[i * n, n, i, 0] for i in range(runs)], dtype=torch.int32)
            D.check_runs(host, rows, runs)
            a = D.make_args(s, w, state, x, (0, kc, 2 * kc), in32, 0, z, gate, out, 1e-5, table, 64, runs=host.to(DEV))
            nb = D.chunk_bytes(s)
            (c, p), = D.chunk_groups(host.tolist(), 10 ** 6)
            c, p = c.to(DEV), p.to(DEV)
            ws = torch.empty(c.shape[0] * heads * nb, dtype=torch.uint8, device=DEV)
            o32 = torch.empty(rows, vc, device=DEV)
            print(name, heads, dim, vdim, runs, n, runs * heads * dv // 32,
                  round(us(lambda i: D.chunked(a, c, p, ws, nb, o32), 6), 1), sep=",", flush=True)


def paged(name, rng):
    from llm_sharding_amd.models.stack import AttentionSpec
    from llm_sharding_amd.ops import paged_attn as A
    from llm_sharding_amd.runtime.attn_mixer import Attention
    for nh, nkv, window in ((16, 4, 0), (16, 4, 1024), (32, 8, 0), (64, 8, 0)):
        for S in [[512], [1100], [2048], [1100] * 3, [301] * 5, [rng.randint(100, 600) for _ in range(6)], [2048] * 2]:
            s, rows, pages = AttentionSpec(nh, nkv, 128, 128, 0.09, 20.0, window, 0), sum(S), [-(-n // 64) for n in S]
            table = torch.zeros(len(S), max(pages), dtype=torch.int32)
            for i, n in enumerate(pages):
                table[i, :n] = torch.arange(n) + sum(pages[:i])
            table = table.to(DEV)
            cache = tuple(torch.randn(*x, device=DEV).bfloat16() for x in A.cache_shapes(s, sum(pages)))
            slot = torch.tensor([i for i, n in enumerate(S) for _ in range(n)], dtype=torch.int32, device=DEV)
            pos = torch.tensor([t for n in S for t in range(n)], dtype=torch.int32, device=DEV)
            hscale = torch.full((nh,), s.scale, device=DEV)
            a = A.make_args(s, cache, table, slot, pos, hscale)
            plan = type("Plan", (), {"eng": type("Eng", (), {"device": torch.device(DEV)})})
            td = Attention._tiles(plan, [(sum(S[:i]), n, i, 0) for i, n in enumerate(S)], rows, table)
            q = torch.randn(rows, nh * s.dkp, device=DEV).bfloat16()
            out = torch.zeros(rows, nh * s.dvp, device=DEV, dtype=torch.bfloat16)
            torch.cuda.synchronize()
            print(name, f"paged{window or ''}", nh, nkv, 128, len(S), rows, td.shape[0] * nh // 8,
                  round(us(lambda i: A.tiles(a, td, q, None, out, max(S)), 12), 2), sep=",", flush=True)


def order(name):
    print("build,kernel,heads,kv_heads,dim,prompts,rows,items_an_xcd,us")
    rng = random.Random(0)
    paged(name, rng)
    for nh, nkv, hd in ((32, 32, 128), (16, 16, 64), (32, 8, 64), (64, 8, 128), (24, 8, 128), (32, 32, 64), (40, 40, 128)):
        for S in [[n] for n in (512, 700, 1024, 1300, 1536, 2048, 3000)] + [[301] * 5, [rng.randint(100, 600) for _ in range(6)]]:
            rows, g = sum(S), nh // nkv
            tr = hip.prefill_tile_rows(nh, nkv, rows)
            slot = [i for i, n in enumerate(S) for _ in range(n)]
            pos = [t for n in S for t in range(n)]
            th = hip.build_prefill_tiles(slot, pos, tile_rows=tr)
            groups = nh // (g if 8 % g == 0 else 1)
            items = th.shape[0] * groups // 8 if groups % 8 == 0 else 0
            kc, vc = (torch.randn(len(S), nkv, max(S), hd, device=DEV).bfloat16() for _ in range(2))
            q, td = torch.randn(rows, nh * hd, device=DEV).bfloat16(), th.to(DEV)
            out = torch.zeros(rows, nh * hd, device=DEV, dtype=torch.bfloat16)
            print(name, "flash", nh, nkv, hd, len(S), rows, items,
                  round(us(lambda i: hip.attn_prefill(q, kc, vc, td, nh, nkv, hd, out, tiles_host=th), 12), 2), sep=",", flush=True)


if __name__ == "__main__":
    torch.manual_seed(0)
    {"heights": heights, "scan": scan, "order": order}[sys.argv[1]](sys.argv[2])

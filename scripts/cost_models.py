"""The planners' cost models against the products they were fitted to (profiles/cost_*.csv, MI355X, weights read from memory):
how much slower than the fastest measured configuration the model's choice is, as a geometric mean and at worst, and with
``--fit`` the cooperative GEMV's constants by least squares again. On the CPU.

usage: cost_models.py [--fit]"""
import csv
import math
import os
import sys

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, ROOT)
from llm_sharding_amd.ops import hip, packing  # noqa: E402


def load(name, key):
    """{values of the first ``key`` columns: [(us, the columns between)]}"""
    out = {}
    with open(os.path.join(ROOT, "profiles", name)) as fh:
        rows = csv.reader(fh)
        next(rows)
        for r in rows:
            out.setdefault(tuple(map(int, r[:key])), []).append((float(r[-1]), tuple(map(int, r[key:-1]))))
    return out


def regret(products, choose) -> str:
    off = []
    for k, res in products.items():
        times = {c: us for us, c in res}
        c = choose(k, times)
        if c in times:
            off.append(times[c] / min(times.values()))
    return f"{math.exp(sum(map(math.log, off)) / len(off)):.3f}, worst {max(off):.2f}, {len(off)} products"


def sk(k, times):
    n, kk, m = k
    return min((c for c in times if c[2] == 1), key=lambda c: hip.gemm_sk_cost(m, n, kk, c[0], c[1], c[3]))


def coop(k, times):
    return packing._coop_choice(k[0] // 16, k[1], packing.row_blocks(k[2]), False)


def one_tile(k, times):
    """The model's choice without two tiles per wave and three parts."""
    c = [c for c in times if c[0] == 1 and c[2] == 2 and c[3] in (1, 2, 4, 8) and c[4] <= 2 and c[5] == 3]
    return min(c, key=lambda c: (packing.coop_cost(k[0] // 16, k[1], packing.row_blocks(k[2]), c), c[1] * c[4]), default=None)


def fills(k, times):
    """The smallest split that fills the chip."""
    for kf in (8, 4, 2):
        c = sorted(c for c in times if c[:3] == (1, 8, kf) and c[4:] == (1, 3) and c[3] >= 1)
        if c:
            return next((x for x in c if k[0] // 128 * x[3] >= hip.N_CU), c[-1])


def tiles_us(k, c):
    """csrc/kernels/linear_f32.hip plan"""
    (n, kk, rows), (bm, bn, s) = k, c
    busy, idle = {(128, 256): (2.08, 1.74), (128, 128): (1.14, 0.92), (64, 128): (0.635, 0.525), (64, 64): (0.38, 0.31)}[bm, bn]
    rounds, rem = divmod(-(-rows // bm) * -(-n // bn), 256)
    us, kb, part = rounds * (kk // 32 * busy + 5.2), bm * bn / 256, rem * s
    if rem:
        m = -(-part // 256)
        us += m * (-(-kk // 32 // s) * (busy if rounds or m > 1 else idle + (busy - idle) * part / 256) + 5.2)
        if s > 1:
            us += (0.28 + s * (0.22 + 0.0065 * kb) + 0.00051 * kb * part) * (1.42 if rounds else 1)
    return us


def tiles(k, times):
    return min(times, key=lambda c: tiles_us(k, c))


def fit(products):
    import numpy as np
    from scipy.optimize import least_squares
    data = []
    for k, res in products.items():
        best = min(us for us, _ in res)
        data += [(k, c, us, best) for us, c in res if c[0] == 1 and c[2] == (2 if k[2] > 64 else 4) and 1 <= c[3] <= 8
                 and c[4] <= 2 and c[5] == 3 and us < 2 * best]

    def model(p, k, c):
        fixed, stream, l2, far, meet, merge, fill, waves = p
        n, kk, rows = k
        mr, wg = 16 * packing.row_blocks(rows), n // 16 // c[1] * c[3]
        load = -(-wg // 256) * 256 / wg if wg > 256 else (256 / wg) ** fill
        w, a = n * kk * 2e-6, wg * mr * kk / c[3] * 2e-6
        us = fixed + max(w / 4.9, (w / stream + a / (l2 if w <= 130 else far)) * load * max(1, waves * 256 / (wg * c[1] * c[4])) ** 0.3)
        return us if c[3] == 1 else us + meet + c[3] * mr * n * 8e-6 / merge
    sol = least_squares(lambda p: [math.log(model(p, k, c) / us) * (best / us) ** 2 for k, c, us, best in data],
                        [4, 8, 27, 11, 2.2, 4.7, 0.6, 4], loss="soft_l1", f_scale=0.1)
    print("us fixed, TB/s weights, TB/s activations (L2, beyond it), us and TB/s of a split, power of idle CUs, waves a CU wants:",
          np.round(sol.x, 2), f"{len(data)} points, rms of the logarithm {math.sqrt(2 * sol.cost / len(data)):.3f}")


def main() -> None:
    packing._TUNED = {}
    for what, file in (("", ""), (" (split tiles finished by all their workgroups)", "_shared")):
        print(f"gemm_sk{what}:", regret(load(f"cost_gemm_sk{file}.csv", 3), sk))
        with open(os.path.join(ROOT, "profiles", f"cost_gemm_sk_checks{file}.csv")) as fh:
            rows = list(csv.DictReader(fh))
        for name in ("one_hand_off", "present"):
            off = [float(r[name + "_us"]) / float(r["two_heights_us"]) for r in rows]
            print(f"gemm_sk{what}, products it was not fitted to, {name} / two_heights: {math.exp(sum(map(math.log, off)) / len(off)):.3f}, "
                  f"worst {max(off):.2f}, {sum(x > 1.05 for x in off)} of {len(off)} more than 1.05")

    def against(name, file, now, other):
        with open(os.path.join(ROOT, "profiles", file)) as fh:
            off = [float(now(r)) / float(other(r)) for r in csv.DictReader(fh)]
        print(f"{name}: {math.exp(sum(map(math.log, off)) / len(off)):.3f}, {min(off):.2f} to {max(off):.2f}, {len(off)} cases")
    for what, other in (("two heights by the mean", lambda r: r["us_two_heights"]),
                        ("the fastest of four", lambda r: min(float(r[f"us_{h}"]) for h in (128, 192, 256, 320)))):
        against(f"experts' height picked / {what}", "cost_moe_bf16.csv", lambda r: r["us_picked"], other)
    for w in ("32", "64"):
        against(f"delta rule's scan by its rule / always {w} channels", "delta_scan_width.csv", lambda r: r["us_by_the_rule"],
                lambda r: r[f"us_{w}"])
    against("prompt attention by its rule / plain order", "prompt_order.csv", lambda r: r["us_by_the_rule"], lambda r: r["us_plain_order"])
    products = load("cost_coop.csv", 3)
    for name, pick in (("the model", coop), ("smallest split that fills", fills)):
        for rows in (24, 48, 65, 96, 100, 128):
            print(f"cooperative GEMV, {name}, {rows} rows:", regret({k: r for k, r in products.items() if k[2] == rows}, pick))
        print(f"cooperative GEMV, {name}, larger products at 32 and 64:",
              regret({k: r for k, r in products.items() if k[2] in (32, 64)}, pick))
    for rows in (65, 96, 128):
        print(f"cooperative GEMV, one tile per wave and no three parts, {rows} rows:",
              regret({k: r for k, r in products.items() if k[2] == rows}, one_tile))
    print("fp32 tiles and parts of K:", regret(load("cost_f32_tiles.csv", 3), tiles))
    if "--fit" in sys.argv:
        fit(products)


if __name__ == "__main__":
    main()

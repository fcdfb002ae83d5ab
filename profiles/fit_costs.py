"""Fits the constants of the tiles' cost models to the timings beside this file
and prints them as they stand in the sources: PANEL_COST (panel_plan.hip),
prefill_cost, panel_beats_prefill and panel_beats_verify (gemm.hip), with their errors.

    python profiles/fit_costs.py

panel_times.csv: us of one product on MI355X (f16 activations, three rotating
sets of inputs), for each encoding, matrix and token count on every panel shape
and K split that fits; `splits` 1 is none, n > 1 all tiles n ways, -n only the
tiles of the last partial round. other_tile_us is the tile that served the shape
otherwise (the prefill tile from 49 tokens). Taken with the panel tile's first
decoding; the present one is within 1 % on 25 of its sizes (3 % on 3).

prefill_times.csv: us of Q8_0 with f16 activations on the prefill tile and on the
panel tile by its plan, on matrices of few rows and of short rows.

few_token_times.csv: us through the public entry point on the register verify
tile and on the panel tile by its plan, 4 to 16 tokens, matrices of at least
2^25 weights.
"""
import collections
import csv
import math
import sys
from pathlib import Path

import numpy as np
from scipy.optimize import nnls

HERE = Path(__file__).resolve().parent
sys.path.insert(0, str(HERE.parent))
# TG, RG, WR, WK, DEPTH of the shapes (panel.h), and 16-byte chunks of a raw row unit
SHAPES = [(1, 1, 4, 1, 4), (1, 1, 2, 4, 2), (2, 1, 2, 2, 2), (3, 1, 4, 2, 2), (4, 1, 4, 2, 2),
          (4, 1, 2, 2, 2), (4, 1, 4, 1, 2), (4, 2, 4, 1, 2), (6, 2, 4, 1, 2), (8, 2, 4, 1, 2)]
CHUNKS = {8: 18, 12: 9, 13: 11, 14: 14, 23: 9}
CUS = 256


def cdiv(a, b):
    return -(-a // b)


def occupancy(enc, shape):
    """Workgroups a CU holds, by LDS and registers."""
    t, r, w, k, d = SHAPES[shape]
    lds = max(d * k * 32 * t * 128 + 32 * r * w * k * CHUNKS[enc] * 16, w * k * t * r * 4096 if k > 1 else 0)
    simd = {1: 4, 2: 4, 3: 3, 4: 2}.get(t * r, 2 if t * r <= 8 else 1)
    return max(1, min(160 * 1024 // lds, simd * 4 // (w * k)))


def panel_features(enc, shape, rows, columns, tokens, splits):
    """[rounds, blocks, blocks x further workgroups on the busiest CU, split, MB of partial sums]"""
    t, r, w, k, _ = SHAPES[shape]
    bm, bn, nb, occ = 32 * t, 32 * r * w, columns // 256, occupancy(enc, shape)
    tiles = cdiv(tokens, bm) * cdiv(rows, bn)

    def part(count, blocks):
        v = np.zeros(3)
        whole, rest = divmod(count, CUS * occ)
        n = cdiv(blocks, k)
        v += whole * np.array([1, n, n * (occ - 1)])
        if rest:
            v += np.array([1, n, n * (cdiv(rest, CUS) - 1)])
        return v

    if splits == 1:
        return np.concatenate([part(tiles, nb), [0, 0]])
    if splits > 1:
        sums = min(tiles * bm * bn, tokens * rows) * (splits + 0.5)
        return np.concatenate([part(tiles * splits, cdiv(nb, splits)), [1, sums * 4e-6]])
    tail = tiles % (CUS * (occ if t * r <= 8 else 1))
    v = part(tiles - tail, nb) + part(tail * -splits, cdiv(nb, -splits))
    return np.concatenate([v, [1, tail * bm * bn * (-splits + 0.5) * 4e-6]])


def prefill_split(tiles, nb):
    """prefill_split_plan: whole tiles, split tiles, splits."""
    rem = tiles % CUS
    best, splits = 0.85 * (nb + 1), 1
    for s in range(2, min(nb, 16) + 1):
        if rem == 0 or rem * s > 4 * CUS:
            break
        cost = cdiv(rem * s, CUS) * (cdiv(nb, s) + 1) + rem * s / 100 + 0.3
        if cost < best:
            best, splits = cost, s
    return (tiles - rem, rem, splits) if splits > 1 else (tiles, 0, 1)


def prefill_features(rows, columns, tokens):
    nb = columns // 256
    whole, tail, splits = prefill_split(cdiv(tokens, 256) * cdiv(rows, 256), nb)
    r1, r2 = cdiv(whole, CUS), cdiv(tail * splits, CUS)
    return np.array([r1 + r2, r1 * nb + r2 * cdiv(nb, splits), tail * splits * 65536 * 4e-6])


def fit(features, us):
    a, y = np.array(features), np.array(us)
    x, _ = nnls(a / y[:, None], np.ones(len(y)))
    return x, a @ x / y - 1


def panel():
    times, other = collections.defaultdict(list), {}
    for row in list(csv.reader(open(HERE / "panel_times.csv")))[1:]:
        key = tuple(map(int, row[:4]))
        if row[4]:
            other[key] = float(row[4])
        for item in row[5].split():
            shape, splits, us = item.split(":")
            times[key[0], int(shape)].append((*key[1:], int(splits), float(us)))
    coefficients, rms = {}, []
    for enc in CHUNKS:
        print(f"    {{  // encoding {enc}")
        for shape in range(len(SHAPES)):
            d = times[enc, shape]
            x, err = fit([panel_features(enc, shape, *q[:4]) for q in d], [q[4] for q in d])
            coefficients[enc, shape] = x
            rms.append(float(np.sqrt((err**2).mean())))
            print("        {%d, %.2ff, %.3ff, %.3ff, %.1ff, %.3ff}," % (occupancy(enc, shape), *x))
        print("    },")
    print(f"{sum(map(len, times.values()))} timings, error rms {min(rms):.3f} to {max(rms):.3f}")
    # the model's choice among the measured plans the planner considers
    plans = collections.defaultdict(list)
    for (enc, shape), d in times.items():
        tg, _, _, wk, _ = SHAPES[shape]
        for rows, columns, tokens, splits, us in d:
            groups = cdiv(tokens, 32)
            if (tg > groups and tg > 1) or (tg < 4 and groups > 2 * tg) or abs(splits) * wk > columns // 256:
                continue
            cost = panel_features(enc, shape, rows, columns, tokens, splits) @ coefficients[enc, shape]
            plans[enc, rows, columns, tokens].append((cost, us))
    ratio = [min(v)[1] / min(us for _, us in v) for v in plans.values()]
    print(f"chosen plan over best measured: mean {np.mean(ratio):.3f}, max {max(ratio):.2f} of {len(ratio)} products")
    by_plan = {k: dict() for k in other if k[0] == 8 and k[3] > 48}
    for (enc, shape), d in times.items():
        for rows, columns, tokens, splits, us in d:
            if (enc, rows, columns, tokens) in by_plan:
                by_plan[enc, rows, columns, tokens][shape, splits] = us
    prefill([(*k[1:], other[k], by_plan[k]) for k in by_plan])


def prefill(known):
    """known: rows, columns, tokens, us on the prefill tile, us by panel shape and splits"""
    from tests.test_panel_plan import plan  # the library's own planner

    d = []
    for rows, columns, tokens, us, panels in known:
        p = plan(8, rows, columns, tokens, 1 << 26)
        d.append((rows, columns, tokens, us, panels.get((p[0], p[3] if p[1] == 0 or p[3] == 1 else -p[3]))))
    for r in list(csv.reader(open(HERE / "prefill_times.csv")))[1:]:
        d.append((*map(int, r[:3]), float(r[3]), float(r[4]) if r[4] else None))
    results = np.array([q[0] * q[2] * 4e-6 for q in d])
    x, err = fit(np.column_stack([[prefill_features(*q[:3]) for q in d], results]), [q[3] for q in d])
    print("prefill_cost (Q8_0): %.2f us a round, %.2f a block, %.2f a MB of partial sums, %.2f a MB of results;" % tuple(x),
          "error rms %.3f of %d" % (math.sqrt((err**2).mean()), len(d)))
    both = [(q, mb) for q, mb in zip(d, results) if q[4]]
    tile, panel_us = (np.array([q[i] for q, _ in both]) for i in (3, 4))
    cost = np.array([plan(8, *q[:3], 1 << 26)[8] / 1e3 for q, _ in both])
    model = np.array([prefill_features(*q[:3]) @ x[:3] for q, _ in both])
    for a in np.arange(0, 0.4, 0.1):
        us = np.where(cost + a * np.array([mb for _, mb in both]) < model, panel_us, tile)
        print("panel_beats_prefill with %.1f us a MB of results more: choice over better tile mean %.4f, over prefill at"
              " most %.2f, %d products" % (a, (us / np.minimum(tile, panel_us)).mean(), (us / tile).max(), len(us)))


def few_tokens():
    from tests.test_panel_plan import plan  # the library's own planner

    rows_ = [r for r in list(csv.reader(open(HERE / "few_token_times.csv")))[1:]]
    for enc in (8, 14, 23):
        d = [(*map(int, r[1:4]), float(r[5]), float(r[6])) for r in rows_ if int(r[0]) == enc and r[4] == "f16"]

        def blocks(rows, columns):
            groups = 2 if rows >= 5120 else 1
            return cdiv(cdiv(rows, 16 * groups), CUS) * groups * (columns // 256)

        x, err = fit([[1, blocks(r, c), blocks(r, c) * t] for r, c, t, _, _ in d], [q[3] for q in d])
        verify = np.array([x @ [1, blocks(r, c), blocks(r, c) * t] for r, c, t, _, _ in d])
        plans = [plan(enc, r, c, t, 1 << 26) for r, c, t, _, _ in d]
        cost, split = np.array([p[8] / 1e3 for p in plans]), np.array([p[3] > 1 for p in plans])
        v, p = np.array([q[3] for q in d]), np.array([q[4] for q in d])
        best = None
        for whole in np.arange(0.8, 1.5, 0.05):
            for part in np.arange(0.8, 1.3, 0.05):
                us = np.where(np.where(split, part, whole) * cost < verify, p, v)
                # the mean over the better tile, and a third of what is over the verify tile
                score = (us / np.minimum(v, p)).mean() + 0.3 * (us / v - 1.03).clip(0).mean()
                if best is None or score < best[0]:
                    best = score, whole, part, (us / np.minimum(v, p)).mean(), (us / v).max(), (p / v).max()
        print("panel_beats_verify, encoding %d: a %.1f b %.3f c %.4f (rms %.3f) whole %.2f split %.2f;" %
              (enc, *x, math.sqrt((err**2).mean()), *best[1:3]),
              "choice over better tile mean %.4f, over verify at most %.2f (panel for all %.2f), %d timings" %
              (*best[3:], len(d)))


if __name__ == "__main__":
    panel()
    few_tokens()

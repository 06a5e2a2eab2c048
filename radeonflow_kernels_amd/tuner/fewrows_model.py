"""The time estimate of the few-rows kernels that the automatic plans use (fewrows_plan in csrc/gemm_launcher.hip): the
measurements behind it, its fit, and the shapes where the few-rows and the tiled kernels meet.

  python -m radeonflow_kernels_amd.tuner.fewrows_model --measure FILE    every variant and K split over M = 1 ... 512 and the
                                                                         (N, K) of PAIRS, on operand sets in rotation
  python -m radeonflow_kernels_amd.tuner.fewrows_model --ragged FILE     the same over ragged N: RAGGED_ROWS and RAGGED_PAIRS
  python -m radeonflow_kernels_amd.tuner.fewrows_model --fit FILE        how far the estimate's choice is from the fastest plan
                                                                         measured, and the constants refitted to the file
  python -m radeonflow_kernels_amd.tuner.fewrows_model --meet FILE       ragged shapes: the automatic few-rows plan against
                                                                         tiled plans with their staging copies
FILE has one line per plan: M N K variant split_k us (--meet: for each shape the times of both sides). --measure and --meet
need the GPU, and so does --ragged; the estimate and the fit do not.
"""
import argparse
import os
import tempfile

import numpy as np

from . import long_k_model as long_k

BK = 128
MAX_TILE_COUNTERS = 16384
SPLITS = (1, 2, 3, 4, 5, 6, 8, 12, 14)
# variant: tile rows, columns, waves, workgroups that share a CU, K blocks a wave asks for at a time (ALL: the next one is on its
# way while one is multiplied, so that only the first is waited for); b, c, d (see estimate)
ALL = 1 << 20
VARIANTS = {14: (16, 32, 8, 2, 3), 15: (16, 64, 8, 1, 2), 16: (16, 128, 8, 1, ALL), 17: (32, 32, 8, 2, 2), 18: (32, 64, 8, 1, 2),
            19: (64, 32, 8, 1, 2), 20: (64, 64, 8, 1, ALL), 21: (64, 64, 4, 2, ALL), 22: (16, 32, 8, 2, ALL), 23: (16, 64, 8, 1, ALL),
            24: (32, 32, 8, 2, ALL), 25: (32, 64, 8, 1, ALL), 26: (32, 64, 4, 2, ALL), 27: (32, 128, 4, 1, ALL)}
# (the others are measured, but not chosen from)
FIT = {14: (0.0238, 0.6526, 0.0811), 16: (0.017, 1.6541, 0.0325), 20: (0.2932, 1.9032, 0.0785), 21: (1.3762, 1.0315, 0.0158),
       22: (0.0007, 0.6572, 0.086), 23: (0.0704, 1.4481, 0.0227), 24: (0.0049, 0.9508, 0.0676), 25: (0.0106, 1.7903, 0.0289),
       26: (0.3722, 0.7608, 0.0427), 27: (1.0902, 1.385, 0.0109)}
COMMON = (2.5568, 0.6363, 0.1919, 0.2531, 0.0505)   # launch; handing sums over, and per KiB of them; a batch of a wave's loads; a MB of operands
ANY_BYTES = {16: 1.5, 21: 1.5, 27: 1.5}              # where rows of B start at any byte; the other variants 1.27

ROWS = (1, 7, 16, 24, 32, 48, 64, 100, 128, 200, 256, 333, 512)
PAIRS = ((1536, 7168), (4608, 7168), (7168, 2048), (7168, 256), (576, 7168), (3072, 1536), (7168, 2304), (512, 7168), (4096, 512),
         (4096, 7168), (256, 1024), (1024, 2048), (2048, 4096), (8192, 1024), (8192, 7168), (256, 7168), (200, 2048), (1000, 384),
         (1000, 4096), (2003, 1024), (2003, 7168), (5003, 2048), (5003, 128))
# the ragged N that ANY_BYTES is searched on
RAGGED_ROWS = (1, 7, 16, 24, 40, 48, 64, 100, 150, 200, 333, 500)
RAGGED_PAIRS = ((1000, 2048), (1000, 7168), (1001, 4096), (2003, 2048), (2003, 4096), (2003, 7168), (3001, 3072), (5003, 2048), (5003, 7168),
                (1003, 1024), (2003, 384), (5003, 1024))
# ragged shapes between a few hundred and a few thousand rows: N ragged, M ragged, both
MEET = ((601, 5003, 2048), (700, 5003, 1024), (1000, 1000, 1024), (1000, 1000, 4096), (1000, 2003, 1024), (2000, 2003, 1024),
        (3000, 1000, 384), (700, 1000, 7168), (1008, 5003, 2048), (1500, 1000, 2048), (2000, 5003, 512), (2000, 1000, 7168),
        (4000, 200, 2048), (4096, 1000, 1024), (4001, 2003, 384), (513, 5003, 7168), (800, 200, 7168), (3000, 2003, 2048),
        (300, 5003, 2048), (200, 2003, 7168), (100, 5003, 7168), (500, 200, 7168),
        (601, 1536, 7168), (513, 7168, 256), (1001, 576, 7168), (300, 512, 7168), (250, 1536, 7168), (333, 7168, 2048),
        (130, 4608, 7168), (500, 4096, 512), (200, 3072, 1536))


def _ceil(a, b):
    return -(-a // b)


def _terms(variant, m, n, k, split, num_cu):
    """(parts, KiB of sums, rounds, batches, K blocks of a wave times workgroups sharing a CU, MB fetched), or None if the
    planner does not consider this split."""
    bm, bn, waves, per_cu, depth = VARIANTS[variant]
    qk, items = k // BK, _ceil(m, bm) * _ceil(n, bn)
    if split > qk or (split > 1 and (items * split > 4 * num_cu or items > MAX_TILE_COUNTERS)):
        return None
    kb = _ceil(qk, split)
    parts, own = _ceil(qk, kb), _ceil(kb, waves)
    wgs = items * parts
    return (parts, parts * bm * bn / 1024.0, _ceil(wgs, num_cu * per_cu), _ceil(own, depth), own * (per_cu if wgs > num_cu else 1),
            wgs * kb * (bm + bn) * BK * 1e-6 * 256 / num_cu)


def _features(variant, m, n, k, split, num_cu=256):
    """What the estimate's constants multiply: COMMON's, then b, c and d; or None."""
    t = _terms(variant, m, n, k, split, num_cu)
    if t is None:
        return None
    parts, kib, rounds, batches, blocks, mb = t
    f = rounds * (ANY_BYTES.get(variant, 1.27) if n % 16 else 1.0)
    return (1.0, float(parts > 1), kib if parts > 1 else 0.0, f * batches, k * (m + n) * 1e-6, f, f * blocks, mb)


def estimate(variant, m, n, k, split, num_cu=256, fit=None, common=COMMON):
    """The estimate of fewrows_plan in us, or None."""
    x = _features(variant, m, n, k, split, num_cu)
    return None if x is None else sum(c * y for c, y in zip(tuple(common) + (fit or FIT)[variant], x))


def tile_estimate(m, n, k, split, num_cu=256):
    """The tiled kernels' figure for variant 28 (128 x 128), which is numbered after the few-rows kernels, in the same us."""
    qk, tiles = k // BK, _ceil(m, 128) * _ceil(n, 128)
    kb = _ceil(qk, split)
    parts = _ceil(qk, kb)
    t = _ceil(tiles * parts, num_cu) * (kb * 0.44 + 2.25)
    return 3.1 + 0.67 * (t + (6.03 + 1.27e-6 * parts * m * n if parts > 1 else 0.0))


def long_k_share(n):
    """What part of the long-K estimate of variant 28's plan of one K part the few-rows estimate has to stay below."""
    return 1.0 if n % 1024 == 0 else 0.85


def choice(m, n, k, num_cu=256, fit=None, common=COMMON, tiles=True):
    """The (variant, split_k) the planner picks from variant 14 on. tiles: variant 28 among them (not for ragged operands)."""
    best = None
    for v in fit or FIT:
        for s in SPLITS:
            t = estimate(v, m, n, k, s, num_cu, fit, common)
            if t is None:
                break
            if best is None or t < best[0]:
                best = (t, v, s)
    if tiles:
        few = best
        for s in (1, 2, 3, 4, 6, 8, 12, 16):
            if s <= k // BK and tile_estimate(m, n, k, s, num_cu) < best[0]:
                best = (tile_estimate(m, n, k, s, num_cu), 28, s)
        if best[1:] == (28, 1):
            if m <= 512 and long_k.in_range(m, n, k, num_cu) and few[0] < long_k_share(n) * long_k.estimate(28, m, n, k, 1, long_k.CACHED):
                best = few
    return best[1:]


def refit(rows, rounds=40000, seed=0):
    """Searches the constants from the ones in use: random steps that are kept while the choice's distance from the fastest plan
    of a shape (mean, and a twentieth of the worst), plus 0.15 times the estimate's own error there, does not grow. (FIT, COMMON)."""
    nc, variants = len(COMMON), list(FIT)
    shapes = {}
    for m, n, k, v, s, us in rows:
        shapes.setdefault((m, n, k), {})[v, s] = us
    a, t, seg, best = [], [], [], []
    for shape, times in shapes.items():
        seg.append(len(t))
        best.append(min(times.values()))
        for (v, s), us in times.items():
            if v in FIT:
                x = _features(v, *shape, s)
                row = np.zeros(nc + 3 * len(variants))
                row[:nc] = x[:nc]
                row[nc + 3 * variants.index(v):][:3] = x[nc:]
                a.append(row)
                t.append(us)
    a, t, best, ends = np.array(a), np.array(t), np.array(best), seg[1:] + [len(t)]

    def cost(x):
        est = a @ x
        pick = np.array([b + np.argmin(est[b:e]) for b, e in zip(seg, ends)])
        behind = t[pick] / best
        return behind.mean() - 1 + 0.05 * (behind.max() - 1) + 0.15 * np.sqrt(np.mean(np.log(est[pick] / t[pick]) ** 2))

    x = np.array(tuple(COMMON) + sum((FIT[v] for v in variants), ()))
    rng, now, scale = np.random.default_rng(seed), cost(x), np.maximum(x, 0.02)
    for _ in range(rounds):
        y = x.copy()
        for i in rng.choice(len(x), rng.integers(1, 4), replace=False):
            y[i] = max(0.0, y[i] + scale[i] * rng.normal() * rng.choice([0.03, 0.1, 0.3]))
        c = cost(y)
        if c <= now:
            x, now = y, c
    x = [round(float(v), 4) for v in x]
    return {v: tuple(x[nc + 3 * i:nc + 3 * i + 3]) for i, v in enumerate(variants)}, tuple(x[:nc])


def read(path):
    with open(path) as f:
        rows = [l.split() for l in f if l[:1].isdigit()]
    rows = [tuple(int(x) for x in r[:5]) + (float(r[5]),) for r in rows]
    return [r for r in rows if _terms(r[3], r[0], r[1], r[2], r[4], 256)]


def report(rows, fit, common, what):
    """How far the model is from the measured times, and its choice from the fastest measured plan of each shape."""
    err = [estimate(v, m, n, k, s, fit=fit, common=common) / us for m, n, k, v, s, us in rows if v in FIT]
    shapes = {}
    for m, n, k, v, s, us in rows:
        shapes.setdefault((m, n, k), {})[v, s] = us
    behind = [t[choice(*shape, fit=fit, common=common, tiles=False)] / min(t.values()) for shape, t in shapes.items()]
    print("%s: estimate over measured %.2f ... %.2f, rms of the logarithm %.3f; choice behind the fastest of %d shapes by %.1f %% "
          "on average, %.0f %% at worst" % (what, min(err), max(err), float(np.sqrt(np.mean(np.log(err) ** 2))), len(shapes),
                                             100 * (np.mean(behind) - 1), 100 * (max(behind) - 1)))


def measure(path, pairs=PAIRS, row_counts=ROWS):
    import radeonflow_kernels_amd as rfk
    from . import gemm_tuner as t
    t.settle(rfk)
    with open(path, "w") as f:
        for n, k in pairs:
            for m in row_counts:
                sets = t.operand_sets(m, n, k)
                for v in VARIANTS:
                    for s in SPLITS:
                        if _terms(v, m, n, k, s, 256):
                            f.write("%d %d %d %d %d %.2f\n" % (m, n, k, v, s, t.rotated_us(rfk, sets, rfk.GemmConfig(v, s, 8, 0), 32, 2)))
                f.flush()
            print(n, k, flush=True)


# tiled plans tried on the padded shape (variant, split_k, schedule)
TILED = [(v, s, 0) for v in (7, 9) for s in (1, 2, 3, 4)] + [(v, s, 0) for v in (6, 8, 3, 10) for s in (1, 2, 3)] + \
        [(v, 1, 0) for v in (0, 1, 5, 11, 12, 13)] + [(0, 1, 2), (1, 1, 2), (3, 1, 2), (8, 6, 0)]


def meet(path):
    """Per shape: the automatic plan, the few-rows plan the estimate picks and the fastest tiled plan (named by a plan file for
    the padded shape), all with what they need around them."""
    import radeonflow_kernels_amd as rfk
    from . import gemm_tuner as t
    t.settle(rfk)
    with tempfile.TemporaryDirectory() as d, open(path, "w") as f:
        plans = os.path.join(d, "p.plans")
        for m, n, k in MEET:
            sets = t.operand_sets(m, n, k)
            auto = t.rotated_us(rfk, sets, None, 32)
            few = choice(m, n, k, tiles=False)
            few_us = t.rotated_us(rfk, sets, rfk.GemmConfig(few[0], few[1], 8, 0), 32)
            plan = rfk.select_config(m, n, k)
            best = None
            for v, s, sched in TILED:
                with open(plans, "w") as p:
                    p.write("%d %d %d %d %d 8 %d\n" % (_ceil(m, 16) * 16, _ceil(n, 16) * 16, k, v, s, sched))
                rfk.load_plans(plans)
                got = rfk.select_config(m, n, k)
                if (got.variant, got.split_k, got.stream_k) == (v, s, sched):
                    us = t.rotated_us(rfk, sets, None, 16, 2)
                    best = min(best or (us, v, s, sched), (us, v, s, sched))
                rfk.clear_plans()
            f.write("%d %d %d  auto %d/%d/%d %.2f  few rows %d/%d %.2f (estimate %.2f)  tiled %d/%d/%d %.2f\n" % (
                m, n, k, plan.variant, plan.split_k, plan.stream_k, auto, few[0], few[1], few_us,
                estimate(few[0], m, n, k, few[1]), best[1], best[2], best[3], best[0]))
            f.flush()
            print(m, n, k, flush=True)


def main():
    ap = argparse.ArgumentParser()
    for name in ("measure", "ragged", "fit", "meet"):
        ap.add_argument("--" + name, metavar="FILE")
    a = ap.parse_args()
    if a.measure:
        measure(a.measure)
    if a.ragged:
        measure(a.ragged, RAGGED_PAIRS, RAGGED_ROWS)
    if a.fit:
        rows = read(a.fit)
        report(rows, FIT, COMMON, "%d measurements, constants in use" % len(rows))
        fit, common = refit(rows)
        report(rows, fit, common, "refitted")
        print("COMMON =", common, "\nFIT =", fit)
    if a.meet:
        meet(a.meet)


if __name__ == "__main__":
    main()

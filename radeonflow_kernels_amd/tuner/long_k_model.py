"""The time estimate that weighs tile plans and their K splits against each other where K is long and the chip is not full of the
largest tile (split_tile_us and split_tile_plan in csrc/gemm_launcher.hip): the measurements behind it and its fit.

  python -m radeonflow_kernels_amd.tuner.long_k_model --measure FILE    the tiles of TILES with 1 to 8 K parts over shapes drawn at
                                                                        random, on operand sets in rotation
  python -m radeonflow_kernels_amd.tuner.long_k_model --fit FILE        how far the estimate is from the times, and its constants
                                                                        fitted to the file
FILE has one line per plan: M N K variant split_k us. --measure needs the GPU; the estimate and the fit do not.
"""
import argparse
import math
import random

import numpy as np

BK = 128
# variant: tile rows, columns
TILES = {9: (64, 128), 12: (64, 128), 28: (128, 128), 8: (128, 192), 10: (128, 256), 11: (192, 192), 0: (256, 256)}
# a round of tiles; a K block of it; more of it with the share of the compute units at work
FIT = {9: (0.232, 0.462, 0.027), 12: (0.0, 0.767, 0.401), 28: (0.229, 0.434, 0.246), 8: (0.716, 0.623, 0.255), 10: (1.02, 0.77, 0.097),
       11: (0.981, 0.892, 0.085), 0: (0.885, 1.313, 0.0)}
# launch; per million outputs; per million bytes of A and B; K split, and per million sums
COMMON = (3.281, 0.693, 0.057, 2.471, 1.182)
SPLITS = (1, 2, 3, 4, 5, 6, 8)


def _ceil(a, b):
    return -(-a // b)


def in_range(m, n, k, num_cu=256):
    """Whether the planner weighs this (padded) shape: the sizes measured, less than a round of 256 x 256 tiles, 256 units."""
    return (num_cu == 256 and 48 <= m <= 2608 and 256 <= n <= 8192 and 1024 <= k <= 8192 and n * k <= 6.0e7 and
            _ceil(m, 256) * _ceil(n, 256) <= num_cu)


def _parts(k, split):
    return _ceil(k // BK, _ceil(k // BK, split))


def _terms(variant, m, n, k, split, num_cu=256):
    """What a variant's constants and COMMON multiply."""
    bm, bn = TILES[variant]
    blocks = k // BK // 2 if variant == 12 else _ceil(k // BK, split)      # (12 splits K inside the workgroup)
    workgroups, mn = _ceil(m, bm) * _ceil(n, bn) * split, m * n * 1e-6
    rounds = _ceil(workgroups, num_cu)
    return ((rounds, rounds * blocks, blocks * workgroups / num_cu),
            (1.0, mn, k * (m + n) * 1e-6, float(split > 1), mn * split if split > 1 else 0.0))


def estimate(variant, m, n, k, split, num_cu=256, fit=None, common=COMMON):
    """Microseconds of a plan; split: K parts that there are."""
    own, shared = _terms(variant, m, n, k, split, num_cu)
    return sum(x * c for x, c in zip(own + shared, tuple((fit or FIT)[variant]) + tuple(common)))


def replaced(first, m, n, k, most=float("inf")):
    """(variant, parts) that the planner takes in place of `first`, the plan of its first model, with sums of at most `most` bytes."""
    if first[0] not in FIT or (first[1] > 1 and 128 < m <= 192):
        return first
    many, before = m > 512, estimate(first[0], m, n, k, _parts(k, first[1]))
    best, out = (0.90 if many and first[0] == 12 else 0.94) * before, first
    for v, (bm, bn) in TILES.items():
        if (v == 28 and not many) or (v == 9 and many and first[0] == 12):
            continue
        for s in SPLITS:
            if s > k // BK or _parts(k, s) != s or (v == 12 and (s > 1 or k // BK % 2)) or (v == 9 and s == 1):
                continue
            if s > 1 and (_ceil(m, bm) * _ceil(n, bn) * s > 600 or m * n * s > 45e6 or 4 * m * n * s > most):
                continue
            t = estimate(v, m, n, k, s)
            if t < best and (v != 9 or not many or t < 0.90 * before):
                best, out = t, (v, s)
    return out


def shapes(seed=1, count=330):
    """(M, N, K): 40 % of them the benchmark's pairs of N and K, 30 % powers of two, 30 % any multiples of 16 and 128."""
    r = random.Random(seed)
    pairs = ((1536, 7168), (4608, 7168), (7168, 2048), (576, 7168), (3072, 1536), (7168, 2304), (512, 7168), (4096, 7168))
    out = []
    while len(out) < count:
        x = r.random()
        n, k = (r.choice(pairs) if x < 0.4 else (r.choice((256, 1024, 2048, 8192)), r.choice((1024, 2048, 4096, 7168))) if x < 0.7 else
                (16 * int(round(math.exp(r.uniform(math.log(16), math.log(512))))), 128 * int(round(math.exp(r.uniform(math.log(8), math.log(64)))))))
        m = _ceil(int(round(math.exp(r.uniform(math.log(40), math.log(2600))))), 16) * 16
        if in_range(m, n, k):
            out.append((m, n, k))
    return out


def measure(path):
    import radeonflow_kernels_amd as rfk
    from . import gemm_tuner as t
    t.settle(rfk)
    with open(path, "w") as f:
        for i, (m, n, k) in enumerate(shapes()):
            sets = t.operand_sets(m, n, k)
            for v, (bm, bn) in TILES.items():
                for s in (1,) if v == 12 else SPLITS:
                    workgroups = _ceil(m, bm) * _ceil(n, bn) * s
                    if s > k // BK or _parts(k, s) != s or (v == 12 and k // BK % 2) or workgroups < 48 or workgroups > (600 if s > 1 else 2100):
                        continue
                    if (v == 0 and s == 1 and workgroups > 256) or (s > 1 and m * n * s > 45e6):
                        continue
                    f.write("%d %d %d %d %d %.2f\n" % (m, n, k, v, s, t.rotated_us(rfk, sets, rfk.GemmConfig(v, s, 8, 0), 32, 2)))
            f.flush()
            if i % 10 == 9:
                print(i + 1, flush=True)


def read(path):
    """{shape: {(variant, parts): us}}"""
    out = {}
    with open(path) as f:
        for l in f:
            w = [int(x) for x in l.split()[:5]]
            out.setdefault(tuple(w[:3]), {})[tuple(w[3:])] = float(l.split()[5])
    return out


def refit(data):
    """Constants of least relative error over the plans within 1.5 of their shape's fastest, none negative. (FIT, COMMON)."""
    variants, rows = list(FIT), []
    for shape, times in data.items():
        for (v, s), us in times.items():
            if us < 1.5 * min(times.values()):
                own, shared = _terms(v, *shape, s)
                row = np.zeros(3 * len(variants) + len(COMMON))
                row[3 * variants.index(v):][:3], row[3 * len(variants):] = own, shared
                rows.append(row / us)
    a, use = np.array(rows), np.ones(3 * len(variants) + len(COMMON), bool)
    while True:
        x = np.zeros(len(use))
        x[use] = np.linalg.lstsq(a[:, use], np.ones(len(a)), rcond=None)[0]
        if x.min() >= 0:
            break
        use[np.argmin(x)] = False
    x = [round(float(v), 3) for v in x]
    return {v: tuple(x[3 * i:3 * i + 3]) for i, v in enumerate(variants)}, tuple(x[3 * len(variants):])


def report(data, fit, common, what):
    err, near = [], []
    for shape, times in data.items():
        for (v, s), us in times.items():
            e = estimate(v, *shape, s, fit=fit, common=common) / us - 1
            err.append(e)
            if us < 1.5 * min(times.values()):
                near.append(e)
    rms = lambda x: 100 * float(np.sqrt(np.mean(np.square(x))))
    print("%s: %d plans of %d shapes, %.1f %% off (rms), %.0f %% at worst; the %d within 1.5 of the fastest %.1f %%" % (
        what, len(err), len(data), rms(err), 100 * max(map(abs, err)), len(near), rms(near)))


def main():
    ap = argparse.ArgumentParser()
    for name in ("measure", "fit"):
        ap.add_argument("--" + name, metavar="FILE")
    a = ap.parse_args()
    if a.measure:
        measure(a.measure)
    if a.fit:
        data = read(a.fit)
        report(data, FIT, COMMON, "constants in use")
        fit, common = refit(data)
        report(data, fit, common, "refitted")
        print("COMMON =", common, "\nFIT =", fit)


if __name__ == "__main__":
    main()

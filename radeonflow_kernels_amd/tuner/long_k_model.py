"""The time estimates that weigh tile plans and their K splits against each other where K is long and the chip is not full of the
largest tile (split_tile_us and split_tile_plan in csrc/gemm_launcher.hip): the measurements behind them and their fit.

  python -m radeonflow_kernels_amd.tuner.long_k_model --measure FILE    the tiles of TILES with 1 to 8 K parts over shapes drawn at
                                                                        random, on operand sets in rotation that the Infinity
                                                                        Cache holds and on sets beyond it
  python -m radeonflow_kernels_amd.tuner.long_k_model --fit FILE        how far the estimates are from the times, and their
                                                                        constants fitted to the file
FILE has one line per plan: M N K variant split_k and the us of both rotations. --measure needs the GPU; the estimates and the fit do not.
"""
import argparse
import math
import random

import numpy as np

BK = 128
# variant: tile rows, columns
TILES = {9: (64, 128), 12: (64, 128), 28: (128, 128), 8: (128, 192), 10: (128, 256), 11: (192, 192), 0: (256, 256)}
# operands from the Infinity Cache; from memory:
#   a round of tiles; a K block of it; more of it with the share of the compute units at work, with the share of the rows of B and of A
#   that start inside a cache line
FITS = ({9: (0.0, 0.366, 0.0, 0.07, 0.028), 12: (0.185, 0.592, 0.147, 0.19, 0.059), 28: (0.194, 0.333, 0.132, 0.069, 0.039),
         8: (0.765, 0.496, 0.077, 0.033, 0.039), 10: (0.759, 0.59, 0.077, 0.073, 0.058), 11: (0.875, 0.738, 0.021, 0.036, 0.018),
         0: (1.138, 1.033, 0.023, 0.049, 0.104)},
        {9: (0.169, 0.397, 0.041, 0.047, 0.028), 12: (0.0, 0.63, 0.444, 0.172, 0.066), 28: (0.073, 0.375, 0.23, 0.072, 0.056),
         8: (0.497, 0.574, 0.217, 0.025, 0.072), 10: (0.712, 0.692, 0.076, 0.086, 0.088), 11: (0.76, 0.847, 0.056, 0.038, 0.042),
         0: (1.004, 1.207, 0.0, 0.095, 0.087)})
#   launch; per million outputs; per million bytes of A and B; K split, and per million sums
COMMONS = ((4.531, 0.403, 0.0, 2.274, 1.177), (3.922, 0.531, 0.054, 2.283, 1.173))
CACHED, MEMORY = 0, 1
SPLITS = (1, 2, 3, 4, 5, 6, 8)


def _ceil(a, b):
    return -(-a // b)


def in_range(m, n, k, num_cu=256):
    """Whether the planner weighs this (padded) shape: the sizes measured, less than a round of 256 x 256 tiles, 256 units."""
    return (num_cu == 256 and 48 <= m <= 2608 and 256 <= n <= 8192 and 1024 <= k <= 8192 and n * k <= 6.0e7 and
            _ceil(m, 256) * _ceil(n, 256) <= num_cu)


def _parts(k, split):
    return _ceil(k // BK, _ceil(k // BK, split))


def _cut(length):
    return 1 - min(length & -length, 128) / 128


def _terms(variant, m, n, k, split, num_cu=256):
    """What a variant's constants and COMMON multiply."""
    bm, bn = TILES[variant]
    blocks = k // BK // 2 if variant == 12 else _ceil(k // BK, split)      # (12 splits K inside the workgroup)
    workgroups, mn = _ceil(m, bm) * _ceil(n, bn) * split, m * n * 1e-6
    rounds = _ceil(workgroups, num_cu)
    return ((rounds, rounds * blocks, blocks * workgroups / num_cu, rounds * blocks * _cut(n), rounds * blocks * _cut(m)),
            (1.0, mn, k * (m + n) * 1e-6, float(split > 1), mn * split if split > 1 else 0.0))


def estimate(variant, m, n, k, split, where, num_cu=256):
    """Microseconds of a plan; split: K parts that there are; where: CACHED or MEMORY."""
    own, shared = _terms(variant, m, n, k, split, num_cu)
    return sum(x * c for x, c in zip(own + shared, FITS[where][variant] + COMMONS[where]))


def shares(first, variant, m, n):
    """What part of the estimates of the plan before another's have to stay below."""
    if variant == 9:
        return (0.88 if first == 12 else 0.93), 0.94
    return (0.93 if m <= 512 else 1.0 if first != 12 else 1.06 if n % 1024 == 0 else 0.96), 0.94


def replaced(first, m, n, k, most=float("inf")):
    """(variant, parts) that the planner takes in place of `first`, the plan of its first model, with sums of at most `most` bytes."""
    if first[0] not in TILES:
        return first
    before = [estimate(first[0], m, n, k, _parts(k, first[1]), w) for w in (CACHED, MEMORY)]
    best, out = float("inf"), first
    for v, (bm, bn) in TILES.items():
        if v == 28 and m <= 512:
            continue
        for s in SPLITS:
            if s > k // BK or _parts(k, s) != s or (v == 12 and (s > 1 or k // BK % 2)) or (v == 9 and s == 1):
                continue
            if s > 1 and (_ceil(m, bm) * _ceil(n, bn) * s > 600 or m * n * s > 45e6 or 4 * m * n * s > most):
                continue
            us = [estimate(v, m, n, k, s, w) for w in (CACHED, MEMORY)]
            if us[MEMORY] < best and all(u < share * b for u, share, b in zip(us, shares(first[0], v, m, n), before)):
                best, out = us[MEMORY], (v, s)
    return out


def shapes(seed=1, count=500):
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
            held, beyond = t.operand_sets(m, n, k), t.operand_sets(m, n, k, 600 << 20, 24)
            for v, (bm, bn) in TILES.items():
                for s in (1,) if v == 12 else SPLITS:
                    workgroups = _ceil(m, bm) * _ceil(n, bn) * s
                    if s > k // BK or _parts(k, s) != s or (v == 12 and k // BK % 2) or workgroups < 48 or workgroups > (600 if s > 1 else 2100):
                        continue
                    if (v == 0 and s == 1 and workgroups > 256) or (s > 1 and m * n * s > 45e6):
                        continue
                    us = [min(t.rotated_us(rfk, sets, rfk.GemmConfig(v, s, 8, 0), 32, 2) for _ in range(2)) for sets in (held, beyond)]
                    f.write("%d %d %d %d %d %.2f %.2f\n" % (m, n, k, v, s, *us))
            f.flush()
            if i % 10 == 9:
                print(i + 1, flush=True)


def read(path, where):
    """{shape: {(variant, parts): us}}"""
    out = {}
    with open(path) as f:
        for l in f:
            w = [int(x) for x in l.split()[:5]]
            out.setdefault(tuple(w[:3]), {})[tuple(w[3:])] = float(l.split()[5 + where])
    return out


def refit(data):
    """Constants of least relative error over the plans within 1.5 of their shape's fastest, none negative: one of FITS, one of COMMONS."""
    variants, rows, common = list(TILES), [], len(COMMONS[0])
    for shape, times in data.items():
        for (v, s), us in times.items():
            if us < 1.5 * min(times.values()):
                own, shared = _terms(v, *shape, s)
                row = np.zeros(5 * len(variants) + common)
                row[5 * variants.index(v):][:5], row[5 * len(variants):] = own, shared
                rows.append(row / us)
    a, use = np.array(rows), np.ones(5 * len(variants) + common, bool)
    while True:
        x = np.zeros(len(use))
        x[use] = np.linalg.lstsq(a[:, use], np.ones(len(a)), rcond=None)[0]
        if x.min() >= 0:
            break
        use[np.argmin(x)] = False
    x = [round(float(v), 3) for v in x]
    return {v: tuple(x[5 * i:5 * i + 5]) for i, v in enumerate(variants)}, tuple(x[5 * len(variants):])


def report(data, where, what):
    err, near = [], []
    for shape, times in data.items():
        for (v, s), us in times.items():
            e = estimate(v, *shape, s, where) / us - 1
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
        for where, what in ((CACHED, "operands from the Infinity Cache"), (MEMORY, "operands from memory")):
            data = read(a.fit, where)
            report(data, where, what)
            print("refitted:", *refit(data))


if __name__ == "__main__":
    main()

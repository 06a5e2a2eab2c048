"""The time estimates that decide what a call takes whose operands would have to be staged (any_tile_plan, skinny_staged_us and
one_round_us in csrc/gemm_launcher.hip): the measurements behind them and their fit.

  python -m radeonflow_kernels_amd.tuner.staged_model --measure FILE    the any-alignment tiles with every K split, the skinny-K schedule
                                                                        on staged copies and one round of 128 x 128 tiles over shapes
                                                                        drawn at random, on operand sets in rotation
  python -m radeonflow_kernels_amd.tuner.staged_model --fit FILE        how far the estimates are from the times, and their constants
                                                                        fitted to the file
FILE has one line per plan: M N K off_b off_c variant split_k schedule us, with B off_b bytes and C off_c elements past a cache line.
--measure needs the GPU; the fit does not.
"""
import argparse
import math
import os
import random
import tempfile

import numpy as np

from .fewrows_model import _ceil

ANY_TILES = {29: (128, 128), 30: (128, 256)}
SKINNY, ONE_ROUND = (0, 1, 4), (28, 1, 0)
# launch; per round, per K block, more of it where rows of A and of B start at any byte (variants 29 and 30); K split, and per million
# sums; per million outputs, and more where rows of C are not whole cache lines, and where those of B (and so mostly of C) start at any byte
ANY = (1.837, 2.54, 0.58, 0.093, 0.105, 3.835, 0.792, 0.093, 0.285, 3.021, 1.029, 0.21, 0.562, 0.168)
# launch and K blocks; per million outputs, and K blocks; copy of A; copy of B; C's way back, per million outputs up to 15 and beyond
SKINNY_STAGED = (2.137, 1.033, 0.265, 0.098, 2.591, 2.948, 1.522, 0.921, 0.369)
ONE_ROUND_US = (3.458, 0.526, 0.434)


def shapes(seed=5):
    """(M, N, K, off_b, off_c): M or N or both ragged; short K with a large C, where A, B or C is staged; and one round of 128 x 128
    tiles, which needs no staging."""
    r = random.Random(seed)

    def log_int(lo, hi):
        return int(round(math.exp(r.uniform(math.log(lo), math.log(hi)))))

    out = []
    while len(out) < 260:
        if r.random() < 0.45:
            n, k = r.choice(((1536, 7168), (4608, 7168), (7168, 2048), (7168, 256), (576, 7168), (3072, 1536), (7168, 2304), (512, 7168),
                             (4096, 512), (4096, 7168)))
            m = log_int(64, 8192)
            m += m % 16 == 0
        else:
            n, k = r.choice((1000, 2003, 5003, log_int(200, 8192), log_int(200, 8192))), 128 * r.choice((1, 2, 3, 4, 8, 12, 16, 32, 56))
            m = log_int(64, 8192)
            if r.random() < 0.5:
                m = _ceil(m, 16) * 16
        if 2097152 <= m * n * k < 3e11 and (m % 16 or n % 16):
            out.append((m, n, k, 0, 0))
    while len(out) < 400:
        n, k, m, kind = 64 * r.randint(16, 128), 128 * r.randint(1, 4), log_int(300, 8192), r.choice("nnacb")
        n -= r.choice((1, 2, 4, 8, 8, 12, 15)) if kind == "n" else 0
        if kind == "a":
            m += m % 16 == 0
        elif r.random() < 0.6:
            m = _ceil(m, 16) * 16
        mn, qk = _ceil(m, 16) * 16 * _ceil(n, 16) * 16, k // 128
        if _ceil(n, 16) % 4 == 0 and (mn >= 4.1e6 if qk == 1 else mn >= 6e6 if qk == 2 else mn >= 2e6 and (qk == 3 or _ceil(n, 256) <= 16)):
            out.append((m, n, k, 5 if kind == "b" else 0, 4 if kind == "c" else 0))
    while len(out) < 430:
        m, n, k = 16 * r.randint(8, 400), 64 * r.randint(4, 128), 128 * r.choice((3, 4))
        if 96 <= _ceil(m, 128) * _ceil(n, 128) <= 256 and (k == 512 or m * n >= 2e6):
            out.append((m, n, k, 0, 0))
    return out


def _flags(m, n, off_b, off_c):
    """Whether A, B (or C) need staging, rows of A and of B start at any byte, rows of C are not whole cache lines."""
    return m % 16 != 0, n % 16 != 0 or off_b % 16 or off_c % 8, m % 4 != 0, n % 4 != 0 or off_b % 4, n % 64 != 0 or off_c % 64


def any_terms(m, n, k, off_b, off_c, variant, split):
    """What ANY's constants multiply."""
    bm, bn = ANY_TILES[variant]
    _, _, bytes_a, bytes_b, cut_c = _flags(m, n, off_b, off_c)
    mp, np_, qk = _ceil(m, 16) * 16, _ceil(n, 16) * 16, k // 128
    kb, mn = _ceil(qk, split), mp * np_ * 1e-6
    parts = _ceil(qk, kb)
    rounds = _ceil(_ceil(mp, bm) * _ceil(np_, bn) * parts, 256)
    x = [1.0] + [0.0] * 8 + [float(parts > 1), mn * parts if parts > 1 else 0.0, mn, mn * bool(cut_c), mn * bool(bytes_b)]
    at = 1 if variant == 29 else 5
    x[at:at + 4] = [rounds, rounds * kb, rounds * kb * bool(bytes_a), rounds * kb * bool(bytes_b)]
    return x


def skinny_terms(m, n, k, off_b, off_c):
    """What SKINNY_STAGED's constants multiply."""
    copy_a, staged_b, _, _, cut_c = _flags(m, n, off_b, off_c)
    mn, qk = _ceil(m, 16) * 16 * _ceil(n, 16) * 16 * 1e-6, k // 128
    back, copy_b = float(bool(staged_b and cut_c)), float(n % 16 != 0 or off_b % 16 != 0)
    return [1.0, qk, mn, qk * mn, float(copy_a), copy_b, back, back * min(mn, 15.0), back * max(mn - 15.0, 0.0)]


def measure(path):
    import radeonflow_kernels_amd as rfk
    import torch
    from . import gemm_tuner as t

    def moved(x, off, dtype):
        flat = torch.empty(x.numel() + off, dtype=dtype, device="cuda")[off:].view(x.shape)
        return flat.copy_(x)

    t.settle(rfk)
    with tempfile.TemporaryDirectory() as d, open(path, "w") as f:
        plans = os.path.join(d, "p.plans")
        for i, (m, n, k, off_b, off_c) in enumerate(shapes()):
            sets = [(a, moved(b.T.view(torch.uint8), off_b, torch.uint8).view(b.dtype).T, sa, sb, moved(c, off_c, c.dtype))
                    for a, b, sa, sb, c in t.operand_sets(m, n, k)]
            copy_a, copy_b = _flags(m, n, off_b, off_c)[:2]
            todo = [(v, s, 0) for v in ANY_TILES for s in (1, 2, 3, 4, 6, 8) if s <= k // 128 and (s == 1 or m * n * s <= 4e7)]
            if not (copy_a or copy_b):
                todo = [ONE_ROUND]
            elif k <= 512 and _ceil(n, 16) % 4 == 0:
                todo.append(SKINNY)
            for plan in todo:
                cfg = rfk.GemmConfig(plan[0], plan[1], 8, 0)
                if plan == SKINNY:                       # on staged copies: named by a plan file for the padded shape
                    with open(plans, "w") as p:
                        p.write("%d %d %d 0 1 8 4\n" % (_ceil(m, 16) * 16, _ceil(n, 16) * 16, k))
                    rfk.load_plans(plans)
                    cfg = None
                f.write("%d %d %d %d %d %d %d %d %.2f\n" % ((m, n, k, off_b, off_c) + plan + (t.rotated_us(rfk, sets, cfg, 32),)))
                rfk.clear_plans()
            f.flush()
            if i % 10 == 9:
                print(i + 1, flush=True)


def read(path):
    """{shape with offsets: {plan: us}}"""
    out = {}
    with open(path) as f:
        for l in f:
            w = [int(x) for x in l.split()[:8]]
            out.setdefault(tuple(w[:5]), {})[tuple(w[5:])] = float(l.split()[8])
    return out


def fit(path):
    data = read(path)
    # plans within 1.6 of the shape's fastest: the others are never taken
    rows = {"ANY": [(any_terms(*s, *p[:2]), us) for s, t in data.items() for p, us in t.items() if p[0] in ANY_TILES and us < 1.6 * min(t.values())],
            "SKINNY_STAGED": [(skinny_terms(*s), t[SKINNY]) for s, t in data.items() if t.get(SKINNY, 1e9) < 1.6 * min(t.values())],
            "ONE_ROUND_US": [((1.0, s[2] // 128, s[0] * s[1] * 1e-6), t[ONE_ROUND]) for s, t in data.items() if ONE_ROUND in t]}
    fitted = {}
    for name, r in rows.items():
        x, us = np.array([a for a, _ in r]), np.array([b for _, b in r])
        fitted[name] = np.linalg.lstsq(x / us[:, None], np.ones(len(us)), rcond=None)[0]
        for what, c in (("in use", globals()[name]), ("fitted", fitted[name])):
            e = x @ np.array(c) / us
            print("%s %s: %d times, estimate over measured %.2f ... %.2f, rms of the logarithm %.3f" % (
                name, what, len(us), e.min(), e.max(), np.sqrt(np.mean(np.log(e) ** 2))))
        print(name, "=", tuple(round(float(v), 3) for v in fitted[name]))
    behind = []
    for s, t in data.items():                            # the choice between the two on shapes that have both
        if SKINNY in t:
            best_any = min((float(np.dot(any_terms(*s, *p[:2]), ANY)), us) for p, us in t.items() if p[0] in ANY_TILES)
            took = best_any[1] if best_any[0] < np.dot(skinny_terms(*s), SKINNY_STAGED) else t[SKINNY]
            behind.append(took / min(t.values()))
    print("choice between them, constants in use: behind the faster by %.1f %% on average of %d shapes, %.0f %% at worst" % (
        100 * (np.mean(behind) - 1), len(behind), 100 * (max(behind) - 1)))


def main():
    ap = argparse.ArgumentParser()
    for name in ("measure", "fit"):
        ap.add_argument("--" + name, metavar="FILE")
    a = ap.parse_args()
    if a.measure:
        measure(a.measure)
    if a.fit:
        fit(a.fit)


if __name__ == "__main__":
    main()

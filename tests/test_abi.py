"""CPU-only checks of the C ABI: libgemm.so loads, exports what include/rf_gemm.h declares, and rejects bad
arguments before touching a device."""
import ctypes
import os
import re
import subprocess
import sys

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def _declared_functions():
    text = open(os.path.join(ROOT, "include", "rf_gemm.h")).read()
    text = re.sub(r"/\*.*?\*/", "", text, flags=re.S)
    return sorted(set(re.findall(r"\b(run|rf_[a-z0-9_]+)\s*\(", text)))


def test_library_exports_every_declared_symbol():
    from radeonflow_kernels_amd import gemm
    lib = ctypes.CDLL(gemm.LIB_PATH)
    names = _declared_functions()
    assert "run" in names and "rf_fp8_gemm" in names and len(names) >= 10
    for n in names:
        assert hasattr(lib, n), "libgemm.so does not export %s" % n
    assert sorted(gemm.EXPORTS) == names


def _declared_parameter_counts():
    text = open(os.path.join(ROOT, "include", "rf_gemm.h")).read()
    text = re.sub(r"/\*.*?\*/", "", text, flags=re.S)
    out = {}
    for name, params in re.findall(r"\b(run|rf_[a-z0-9_]+)\s*\(([^)]*)\)\s*;", text):
        params = params.strip()
        out[name] = 0 if params in ("", "void") else params.count(",") + 1
    return out


def test_python_binding_declares_as_many_arguments_as_the_header():
    """A ctypes prototype with the wrong number or kind of arguments silently truncates 64-bit device pointers to
    32 bits: every entry point the mirror calls with pointers must carry argtypes of the header's length, and
    every pointer parameter must be a pointer type."""
    from radeonflow_kernels_amd import gemm
    L = gemm.lib()
    counts = _declared_parameter_counts()
    with_pointers = [n for n in counts if n not in ("rf_gemm_num_variants", "rf_gemm_destroy", "rf_gemm_last_error",
                                                    "rf_gemm_clear_plans")]
    for name in with_pointers:
        at = getattr(L, name).argtypes
        assert at is not None, "%s has no ctypes prototype" % name
        assert len(at) == counts[name], "%s: %d argtypes, header declares %d" % (name, len(at), counts[name])
    text = re.sub(r"/\*.*?\*/", "", open(os.path.join(ROOT, "include", "rf_gemm.h")).read(), flags=re.S)
    for name, params in re.findall(r"\b(run|rf_[a-z0-9_]+)\s*\(([^)]*)\)\s*;", text):
        if name not in with_pointers:
            continue
        for decl, ct in zip(params.split(","), getattr(L, name).argtypes):
            is_ptr = "*" in decl or "hipStream_t" in decl
            ct_ptr = ct is ctypes.c_void_p or ct is ctypes.c_char_p or hasattr(ct, "contents")
            assert is_ptr == ct_ptr, "%s: parameter '%s' bound as %r" % (name, decl.strip(), ct)


def test_perf_metrics_layout_matches_the_reference_struct():
    from radeonflow_kernels_amd.gemm import PerfMetrics, PerfMetricEntry, GemmConfig
    assert ctypes.sizeof(PerfMetricEntry) == 28
    assert ctypes.sizeof(PerfMetrics) == 4 + 20 * 28 == 564
    assert PerfMetrics.entries.offset == 4
    assert PerfMetricEntry.time.offset == 20 and PerfMetricEntry.gflops.offset == 24
    assert ctypes.sizeof(GemmConfig) == 16


def test_status_codes_without_a_device():
    from radeonflow_kernels_amd import gemm
    L = gemm.lib()
    buf = ctypes.create_string_buffer(64)
    p = ctypes.addressof(buf)
    assert L.rf_fp8_gemm(p, p, p, p, p, 16, 16, 100, None) == 1          # K not a multiple of 128
    assert b"K=100" in L.rf_gemm_last_error()
    assert L.rf_fp8_gemm(p, p, p, p, p, 16, 16, 0, None) == 1
    assert L.rf_fp8_gemm(p, p, p, p, p, -1, 16, 128, None) == 1
    assert L.rf_fp8_gemm(None, p, p, p, p, 16, 16, 128, None) == 2        # null pointer
    assert L.rf_gemm_num_variants() >= 1
    info = [ctypes.c_int() for _ in range(5)]
    assert L.rf_gemm_variant_info(0, *[ctypes.byref(x) for x in info]) == 0
    assert info[0].value % 16 == 0 and info[4].value <= 160 * 1024        # fits the 160 KiB LDS of a gfx950 CU
    assert L.rf_gemm_variant_info(999, *[ctypes.byref(x) for x in info]) == 4


def test_run_aborts_on_an_unsupported_shape_like_the_reference_launcher():
    code = ("import ctypes,sys; sys.path.insert(0,%r); from radeonflow_kernels_amd import gemm; L=gemm.lib(); "
            "b=ctypes.create_string_buffer(64); p=ctypes.addressof(b); L.run(p,p,p,p,p,64,64,100,None,None)" % ROOT)
    r = subprocess.run([sys.executable, "-c", code], stdout=subprocess.PIPE, stderr=subprocess.PIPE, text=True, timeout=120)
    assert r.returncode == -6                                              # SIGABRT
    assert "Unsupported shape M=64, K=100, N=64" in r.stdout


def test_python_mirror_rejects_cpu_tensors_and_wrong_layouts():
    import pytest
    import torch
    import radeonflow_kernels_amd as rfk
    a = torch.zeros((16, 128), dtype=torch.uint8).view(torch.float8_e4m3fn)
    with pytest.raises(ValueError):
        rfk.fp8_mm(a, a, torch.zeros(16, 1), torch.zeros(1, 1), torch.zeros((16, 16), dtype=torch.bfloat16))


def test_plan_files_parse_without_a_device(tmp_path):
    """rf_gemm_load_plans only reads and validates the file (plans are matched against shapes at launch): the tuner's
    line format, the brace format of csrc/tuned_plans.inc, comments; a bad line fails the whole file and names it."""
    from radeonflow_kernels_amd import gemm
    L = gemm.lib()
    good = tmp_path / "plans.txt"
    good.write_text("# shape            variant split group schedule\n"
                    "6144 4608 7168 0 1 16 2\n"
                    "{1024, 1536, 7168, 3, 4, 8, 0},   // 24.2 us\n"
                    "\n"
                    "  512 512 256 1 2 4 0   # trailing comment\n")
    try:
        assert gemm.load_plans(str(good)) == 3
        inc = os.path.join(ROOT, "radeonflow_kernels_amd", "csrc", "tuned_plans.inc")
        assert gemm.load_plans(inc) == sum(1 for l in open(inc) if l.startswith("{"))
        n = ctypes.c_int(-1)
        for text, line in (("512 512 256 1 2 4\n", 1),                       # six fields
                           ("512 512 256 1 2 4 0\n512 512 200 1 1 4 0\n", 2),   # K not a multiple of 128
                           ("512 512 256 99 1 4 0\n", 1),                    # no such variant
                           ("512 512 256 0 2 4 2\n", 1),                     # persistent schedule with a K split
                           ("512 512 256 0 1 4 0 7\n", 1)):                  # eight fields
            bad = tmp_path / "bad.txt"
            bad.write_text(text)
            assert L.rf_gemm_load_plans(str(bad).encode(), ctypes.byref(n)) == 4
            assert ("bad.txt:%d" % line).encode() in L.rf_gemm_last_error()
            assert n.value == -1
        assert L.rf_gemm_load_plans(str(tmp_path / "missing.txt").encode(), None) == 4
        assert L.rf_gemm_load_plans(None, None) == 2
    finally:
        gemm.clear_plans()


def test_compiled_in_plan_table_only_holds_plans_its_shapes_can_run():
    """Every line of csrc/tuned_plans.inc names an existing variant, a split that leaves every part at least one K
    block, and the persistent schedules only where the shape allows them (a plan that cannot run is skipped at lookup,
    so a bad line would silently fall back to the cost model)."""
    from radeonflow_kernels_amd import gemm
    L = gemm.lib()
    inc = os.path.join(ROOT, "radeonflow_kernels_amd", "csrc", "tuned_plans.inc")
    plans = [tuple(int(x) for x in re.findall(r"-?\d+", l.split("}")[0])) for l in open(inc) if l.startswith("{")]
    assert len(plans) >= 29 and len(set(p[:3] for p in plans)) == len(plans)        # one plan per shape
    for m, n, k, variant, split, group, schedule in plans:
        bm, bn = ctypes.c_int(), ctypes.c_int()
        assert L.rf_gemm_variant_info(variant, ctypes.byref(bm), ctypes.byref(bn), None, None, None) == 0
        assert m % 16 == 0 and n % 16 == 0 and k % 128 == 0 and 1 <= split <= k // 128 and group >= 1
        assert schedule in (0, 2, 3, 4), "the stream-K schedule is never tabled"
        if schedule == 4:
            assert variant == 0 and split == 1 and k in (128, 256, 384, 512) and n % 64 == 0
        if schedule in (2, 3):
            assert L.rf_gemm_variant_has_persistent(variant) == 1 and split == 1
            assert m >= bm.value and n % bn.value == 0 and (k // 128) % 2 == 0
        if schedule == 3:
            # measured on 256 compute units: whole rounds first, then a last round that is at most half full (on a
            # device with another count the plan is checked again at lookup and skipped if it does not fit)
            tiles = -(-m // 256) * (n // 256)
            left = tiles % 256
            assert variant == 0 and tiles >= 256 and 0 < left and (left + 7) // 8 * 8 + left <= 256


def test_tuner_never_writes_a_stream_k_winner_into_a_table_or_plan_file(tmp_path):
    """Stream-K needs one tile per compute unit of the device it runs on, so tables and plan files carry the fastest
    plan of another schedule instead."""
    from radeonflow_kernels_amd.tuner import gemm_tuner as t
    cand = lambda sk, us: dict(variant=0, split_k=1, group_m=4, stream_k=sk, us=us, tflops=1.0)
    assert t.best_for_table([cand(1, 10.0), cand(2, 11.0), cand(0, 12.0)])["stream_k"] == 2
    assert t.best_for_table([cand(1, 10.0)]) is None and t.best_for_table([]) is None
    out = tmp_path / "plans.inc"
    t.emit_plans({(512, 512, 256): [cand(1, 10.0), cand(0, 12.0)], (256, 256, 256): [cand(1, 9.0)]}, str(out))
    lines = [l for l in out.read_text().splitlines() if l.startswith("{")]
    assert len(lines) == 1 and lines[0].startswith("{512, 512, 256, 0, 1, 4, 0}")


def test_tuner_replaces_a_tabled_plan_only_when_a_sweep_finds_one_two_percent_faster(tmp_path):
    """Both times come from the same sweep; shapes that were not swept keep their lines, a plan that can no longer run is
    replaced. An emit of nothing over a copy of the compiled-in table writes the same bytes."""
    from radeonflow_kernels_amd.tuner import gemm_tuner as t
    cand = lambda variant, us: dict(variant=variant, split_k=1, group_m=8, stream_k=0, us=us, tflops=1.0)
    inc = tmp_path / "plans.inc"
    inc.write_text("{16, 16, 128, 3, 1, 8, 0},   // 5.00 us\n{32, 16, 128, 3, 1, 8, 0},   // 5.00 us\n"
                   "{48, 16, 128, 3, 1, 8, 0},   // 5.00 us\n{64, 16, 128, 3, 1, 8, 0},   // 5.00 us\n")
    t.emit_plans({(16, 16, 128): [cand(7, 9.85), cand(3, 10.0)], (32, 16, 128): [cand(7, 9.8), cand(3, 10.0)],
                  (48, 16, 128): [cand(7, 11.0)], (80, 16, 128): [cand(7, 1.0)]}, str(inc))
    assert {s: int(l.split(",")[3]) for s, l in t.read_plans(str(inc)).items()} == {
        (16, 16, 128): 3, (32, 16, 128): 7, (48, 16, 128): 7, (64, 16, 128): 3, (80, 16, 128): 7}
    before = open(t.PLANS_INC).read()
    inc.write_text(before)
    t.emit_plans({}, str(inc))
    assert inc.read_text() == before


def test_tuner_times_every_plan_of_the_compiled_in_table():
    """A sweep that leaves a tabled plan out would replace it unseen: the table's lines, 128 x 128 tiles of variant 28 beyond 512
    rows and with every tile order among them, are all timed (they were skipped when kernels for few rows were told by their
    number); the any-alignment tiles are not."""
    import radeonflow_kernels_amd as rfk
    from radeonflow_kernels_amd.tuner import gemm_tuner as t
    inc = os.path.join(ROOT, "radeonflow_kernels_amd", "csrc", "tuned_plans.inc")
    plans = [tuple(int(x) for x in re.findall(r"-?\d+", l.split("}")[0])) for l in open(inc) if l.startswith("{")]
    for p in plans:
        assert p[3:] in set(t.plans_to_time(rfk, *p[:3], 256)), p
    timed = set(t.plans_to_time(rfk, 1024, 3072, 1536, 256))
    assert {(28, s, g, 0) for s in (1, 2, 4, 12) for g in t.GROUPS} <= timed
    kinds = {v["variant"]: v["kind"] for v in rfk.variants()}
    assert "any alignment" in kinds.values() and {kinds[p[0]] for p in timed} == {"tile"}
    for shape in ((64, 3072, 1536), (848, 576, 1024)):
        assert {kinds[p[0]] for p in t.plans_to_time(rfk, *shape, 256)} == {"tile", "few rows"}
    assert rfk.lib().rf_gemm_variant_kind(-1) == -1 == rfk.lib().rf_gemm_variant_kind(len(kinds))


@pytest.mark.parametrize("m,n,k,schedule", [(8192, 7160, 256, 4), (6000, 4090, 128, 4), (5727, 7676, 256, 4), (7137, 4404, 384, 4), (1504, 3889, 384, 0),
                                            (700, 3001, 512, 0), (570, 4096, 384, 0), (1318, 8192, 384, 4)])
def test_short_k_on_staged_copies_is_weighed_against_the_any_alignment_tiles(m, n, k, schedule):
    """Short K, a large C and a ragged N: the skinny-K schedule on staged copies had no estimate and so was never taken (the first four
    shapes: 98, 47, 76 and 61 us on the tiles, 66, 33, 54 and 48 on the schedule); a smaller C stays on the tiles, and with only M ragged
    both sides keep what they had."""
    import radeonflow_kernels_amd as rfk
    plan = rfk.plan_for(m, n, k, 256)
    assert plan.stream_k == schedule and (schedule == 4 or plan.variant in (29, 30))


@pytest.mark.parametrize("m,n,k", [(40, 2003, 7168), (48, 2003, 7168), (1, 5003, 7168), (16, 5003, 7168), (40, 2007, 7168)])
def test_few_rows_on_a_wide_ragged_b_leave_the_tiles_whose_lines_are_cut(m, n, k):
    """Rows of 128 columns that start at any byte are two cache lines each: variant 16 took these shapes at 12.1 to 12.6 us where variants
    23 and 25 take 10.6 to 11.2; with aligned rows it keeps them."""
    import radeonflow_kernels_amd as rfk
    assert rfk.plan_for(m, n, k, 256).variant in (23, 25)
    assert rfk.plan_for(40, 2064, 7168, 256).variant == 16


def test_planner_arithmetic_on_the_host_for_any_compute_unit_count(tmp_path):
    """rf_gemm_plan_for needs no device. With 256 compute units a tabled shape gets its tabled plan; with any other count
    the table (measured on 256) is left aside and the cost model counts rounds for the count given: every plan names an
    existing variant and a split that leaves each part a K block, the persistent schedules only where the shape allows
    them, the half-tile schedule only when the last round of 256 x 256 tiles on that many units is at most half full,
    never stream-K, and the skinny-K schedule for up to four K blocks with a large C whatever the count. A loaded plan
    file still wins on every count."""
    import radeonflow_kernels_amd as rfk
    inc = os.path.join(ROOT, "radeonflow_kernels_amd", "csrc", "tuned_plans.inc")
    table = {p[:3]: p[3:] for p in (tuple(int(x) for x in re.findall(r"-?\d+", l.split("}")[0])) for l in open(inc)
                                     if l.startswith("{"))}
    for shape in ((6144, 4608, 7168), (1024, 1536, 7168), (1024, 576, 7168), (6144, 7168, 256)):
        c = rfk.plan_for(*shape, 256)
        assert (c.variant, c.split_k, c.group_m, c.stream_k) == table[shape]
    nv = rfk.lib().rf_gemm_num_variants()
    for ncu in (8, 64, 104, 128, 228, 304):
        for (m, n, k) in list(table)[::7] + [(8192, 4608, 7168), (4096, 4096, 4096), (640, 640, 640), (48, 48, 128)]:
            c = rfk.plan_for(m, n, k, ncu)
            assert 0 <= c.variant < nv and 1 <= c.split_k <= k // 128 and c.stream_k in (0, 2, 3, 4), (ncu, m, n, k, c)
            bm, bn = ctypes.c_int(), ctypes.c_int()
            assert rfk.lib().rf_gemm_variant_info(c.variant, ctypes.byref(bm), ctypes.byref(bn), None, None, None) == 0
            if c.stream_k in (2, 3):
                assert c.split_k == 1 and m >= bm.value and n % bn.value == 0 and (k // 128) % 2 == 0
            if c.stream_k == 3:
                tiles = -(-m // 256) * (n // 256)
                left = tiles % ncu
                assert c.variant == 0 and tiles >= ncu and 0 < left and (left + 7) // 8 * 8 + left <= ncu
            if c.stream_k == 4:
                assert k in (128, 256, 384, 512) and m % 16 == 0 and n % 64 == 0
        assert rfk.plan_for(6144, 7168, 256, ncu).stream_k == 4
        assert rfk.plan_for(2048, 2048, 256, ncu).stream_k != 4            # below six million outputs
        assert rfk.plan_for(4096, 4096, 512, ncu).stream_k == 4            # three or four K blocks: from two million on
        assert rfk.plan_for(6144, 7168, 384, ncu).stream_k == 4
        assert rfk.plan_for(6144, 7168, 512, ncu).stream_k != 4            # K = 512: up to sixteen strips only
        assert rfk.plan_for(512, 2048, 512, ncu).stream_k != 4
        assert rfk.plan_for(4096, 4096, 640, ncu).stream_k != 4
    # fewer units, more rounds: 2048 x 2048 x 7168 is 64 tiles of 256 x 256: no K split is worth it on 8 units
    assert rfk.plan_for(2048, 2048, 7168, 8).split_k == 1
    # ragged shapes are planned at their padded size
    c, d = rfk.plan_for(1000, 1530, 1024, 128), rfk.plan_for(1008, 1536, 1024, 128)
    assert (c.variant, c.split_k, c.stream_k) == (d.variant, d.split_k, d.stream_k)
    plans = tmp_path / "p.plans"
    plans.write_text("4096 4096 4096 1 2 4 0\n")
    try:
        assert rfk.load_plans(str(plans)) == 1
        for ncu in (64, 256):
            c = rfk.plan_for(4096, 4096, 4096, ncu)
            assert (c.variant, c.split_k, c.group_m, c.stream_k) == (1, 2, 4, 0)
    finally:
        rfk.clear_plans()
    cfg = rfk.GemmConfig()
    assert rfk.lib().rf_gemm_plan_for(16, 16, 100, 256, ctypes.byref(cfg)) == 1
    assert rfk.lib().rf_gemm_plan_for(16, 16, 128, 0, ctypes.byref(cfg)) == 1
    assert rfk.lib().rf_gemm_plan_for(16, 16, 128, 256, None) == 2


def test_few_rows_plans_that_cannot_run_are_skipped_at_lookup(tmp_path):
    """Plan files may name a few-rows variant for a shape it does not take: 2^25 rows, more tiles than arrival counters with a
    K split, another schedule than one workgroup per tile. Such a plan is skipped (it failed the call); one that fits is used."""
    import radeonflow_kernels_amd as rfk
    plans = tmp_path / "few.plans"
    big = 16385 * 32
    plans.write_text("33554432 16 128 14 1 8 0\n16 33554432 128 14 1 8 0\n16 %d 256 14 2 8 0\n16 %d 384 14 1 8 0\n"
                     "16 256 256 14 1 8 4\n16 %d 256 14 2 8 0\n" % (big, big, big - 32))
    try:
        assert rfk.load_plans(str(plans)) == 6
        assert rfk.plan_for(33554432, 16, 128, 256).variant < 14
        assert rfk.plan_for(16, 33554432, 128, 256).variant < 14
        assert rfk.plan_for(16, big, 256, 256).split_k == 1
        assert rfk.plan_for(16, 256, 256, 256).stream_k != 4
        for shape, split in (((16, big, 384), 1), ((16, big - 32, 256), 2)):
            got = rfk.plan_for(*shape, 256)
            assert (got.variant, got.split_k) == (14, split)
    finally:
        rfk.clear_plans()


def test_grouped_variant_choice_on_the_host():
    """rf_grouped_variant_for needs no device. The queue form (5) is taken where its last tiles of 64..256 rows save at
    least 7 % of the rows the other 256-wide forms compute and it has 17/16 items per compute unit (2.5 below K = 4096);
    groups the other forms fit as well, or too few items, keep those forms; tiny problems take the form with the most
    workgroups; bad arguments are refused."""
    import numpy as np
    import radeonflow_kernels_amd as rfk

    def offs(sizes):
        return [0] + [int(x) for x in np.cumsum(sizes)]

    rng = np.random.default_rng(1)
    cuts = np.sort(rng.choice(np.arange(1, 8192 // 16), 31, replace=False)) * 16
    uneven = [0] + [int(x) for x in cuts] + [8192]                       # 32 groups of 16..816 rows
    assert rfk.grouped_variant_for(uneven, 4096, 7168) == 5
    assert rfk.grouped_variant_for(uneven, 4096, 7168, num_cu=304) == 5
    assert rfk.grouped_variant_for(offs([256] * 32), 4096, 7168) in (0, 4)      # nothing to save
    assert rfk.grouped_variant_for(offs([128] * 64), 4096, 7168) == 1
    assert rfk.grouped_variant_for(offs([384] * 20), 4096, 7168) in (1, 4)
    small = offs([int(x) * 16 for x in np.random.default_rng(5).integers(1, 25, 16)])    # 16 groups of 16..384 rows
    assert rfk.grouped_variant_for(small, 2048, 7168) != 5              # 170 items for 256 units
    assert rfk.grouped_variant_for(small, 7168, 7168) == 5              # the same groups, 3.5 times the column tiles
    assert rfk.grouped_variant_for(uneven, 4096, 2048) == 5             # 816 items: 3.2 per unit
    assert rfk.grouped_variant_for(uneven, 2048, 2048) != 5             # 408 items: 1.6 per unit, short items
    assert rfk.grouped_variant_for(offs([64] * 8), 1024, 512) == 3      # no form fills the units: the most workgroups
    for bad in (([0, 16, 8], 256, 256), ([1, 16], 256, 256), ([0, 16], 256, 100), ([0, 16], 0, 256)):
        with pytest.raises(RuntimeError):
            rfk.grouped_variant_for(*bad)


def test_grouped_few_rows_choice_on_the_host():
    """Groups of up to 16 rows take a few-rows form (6, 7 or 9), up to 32 rows the 32-row one (8); longer groups, ragged widths
    and more than 1 GB of weights keep the tiled forms."""
    import radeonflow_kernels_amd as rfk

    def choice(rows, groups, n, k):
        return rfk.grouped_variant_for([rows * g for g in range(groups + 1)], n, k)

    assert choice(2, 8, 2048, 7168) == 9 and choice(2, 16, 2048, 7168) == 7 and choice(16, 32, 2048, 7168) == 6
    assert choice(17, 32, 2048, 7168) == 8 and choice(32, 32, 2048, 7168) == 8
    assert choice(33, 32, 2048, 7168) < 6 and choice(16, 32, 2056, 7168) < 6 and choice(16, 64, 4096, 7168) < 6
    # few tiles: 128 x 128 while they are alone on their compute unit, then 128 x 256; short K keeps the most workgroups
    assert choice(100, 8, 2048, 7168) == 2 and choice(300, 8, 2048, 7168) == 1 and choice(100, 8, 2048, 1024) == 3


def test_few_rows_estimate_of_the_tuner_is_the_planners():
    """The Python statement of the few-rows kernels' time estimate (tuner/fewrows_model.py, where it is measured and fitted) picks
    the planner's variant and K split wherever the planner takes a few-rows plan by estimate: shapes outside the table, other
    compute unit counts, ragged ones planned at their padded size."""
    import random
    import radeonflow_kernels_amd as rfk
    from radeonflow_kernels_amd.tuner import fewrows_model as fm
    rng, seen = random.Random(3), set()
    for i in range(400):
        m, n = rng.choice((16, 32, 48, 80, 144, 272, 400)), 16 * rng.randint(2, 500)
        k, num_cu = 128 * rng.randint(1, 64), rng.choice((64, 255, 256, 304))
        got = rfk.plan_for(m, n, k, num_cu)
        if got.variant >= 14:
            assert (got.variant, got.split_k) == fm.choice(m, n, k, num_cu), (m, n, k, num_cu)
            seen.add(got.variant)
    assert len(seen) >= 5, seen


def test_benchmark_hashes_every_gemm_source():
    """The traffic figures under profiles/ belong to a hash of the GEMM's sources: the launcher and every header it reaches,
    but for the quantisers' and the C ABI."""
    import bench
    csrc = os.path.join(ROOT, "radeonflow_kernels_amd", "csrc")
    reached, todo = set(), ["gemm_launcher.hip"]
    while todo:
        name = todo.pop()
        if name not in reached:
            reached.add(name)
            todo += [os.path.basename(x) for x in re.findall(r'#include "([^"]+\.h)"', open(os.path.join(csrc, name)).read())
                     if os.path.dirname(x) == ""]
    assert sorted(bench.KERNEL_SOURCES) == sorted(reached - {"quantize_kernels.h"})


def test_few_rows_plans_for_a_small_n_and_any_tiles_instead_of_a_staged_skinny_k():
    """Up to 4096 rows the few-rows kernels (variants 14 to 27) are in the choice while N is small; the skinny-K schedule behind a
    staging copy gives way to the tiles that take ragged operands (29, 30) where those fill about one round. Both on 256 units."""
    import radeonflow_kernels_amd as rfk
    few = lambda *a: 14 <= rfk.plan_for(*a).variant <= 27
    assert few(528, 256, 2048, 256) and few(1833, 256, 2048, 256) and few(848, 576, 1024, 256) and few(665, 1536, 384, 256)
    assert not few(1833, 256, 2048, 304) and not few(4112, 256, 2048, 256) and not few(1040, 2048, 2048, 256)
    skinny = lambda *a: rfk.plan_for(*a).stream_k == 4
    for m, n, k in ((570, 4096, 384), (3003, 1024, 512), (8005, 1024, 128), (843, 7168, 256)):
        assert rfk.plan_for(m, n, k, 256).variant in (29, 30) and skinny(m, n, k, 304)
        assert not rfk.plan_for((m + 15) // 16 * 16, n, k, 256).variant in (29, 30)
    assert skinny(1318, 8192, 384, 256) and skinny(5005, 7168, 256, 256)


def test_short_k_plans_by_the_shape_of_the_output():
    """K of three and four blocks: 128 x 128 tiles with eight waves where they are one round of 256 units, the skinny-K schedule
    beyond; one K block: the skinny-K schedule from 4.1 million outputs on."""
    import radeonflow_kernels_amd as rfk
    plan = lambda m, n, k, cu=256: (lambda c: "skinny" if c.stream_k == 4 else c.variant)(rfk.plan_for(m, n, k, cu))
    assert plan(592, 4096, 512) == plan(848, 4096, 384) == plan(592, 3072, 512) == 28
    assert plan(1168, 4096, 512) == "skinny" and plan(592, 4096, 512, 304) == "skinny"      # 320 tiles; another device
    assert plan(592, 7168, 128) == "skinny" and plan(560, 7168, 128) != "skinny" and plan(592, 7168, 256) != "skinny"


def test_staged_model_states_the_estimates_of_the_launcher():
    """tuner/staged_model.py, where they are measured and fitted, picks what the launcher picks between the skinny-K schedule on staged
    copies and the any-alignment tiles (beyond 4096 rows, where no few-rows kernel is considered), K split included."""
    import numpy as np
    import radeonflow_kernels_amd as rfk
    from radeonflow_kernels_amd.tuner import staged_model as sm
    seen = []
    for i, (m, n, k, _, _) in enumerate(sm.shapes(11)):
        m, n, k = m + 4097, -(-n // 64) * 64 - i % 16, min(k, 256)          # N padded to 16 is a multiple of 64: the schedule can run
        if n % 16 == 0 or m * n < 6e6:
            continue
        tiles = min((float(np.dot(sm.any_terms(m, n, k, 0, 0, v, s), sm.ANY)), (v, s, 0)) for v in sm.ANY_TILES for s in (1, 2)
                    if s <= k // 128 and (s == 1 or m * n * s < 3.9e7))
        skinny = float(np.dot(sm.skinny_terms(m, n, k, 0, 0), sm.SKINNY_STAGED))
        if abs(tiles[0] / skinny - 1) > 0.01:
            got = rfk.plan_for(m, n, k, 256)
            assert (got.variant, got.split_k, got.stream_k) == (tiles[1] if tiles[0] < skinny else sm.SKINNY), (m, n, k)
            seen.append(got.stream_k)
    assert min(seen.count(0), seen.count(4)) > 20


def test_long_k_on_a_part_of_the_chip_is_split():
    """split_tile_plan: wide tiles in K parts where the model that ranks whole tiles kept one part; not for tabled shapes, staged B or C,
    other compute unit counts, short K, or a chip full of the largest tile. Odd rows take the plan of the padded shape."""
    import radeonflow_kernels_amd as rfk
    plan = lambda *a: (lambda c: (c.variant, c.split_k, c.stream_k))(rfk.plan_for(*a))
    assert plan(1232, 1616, 7552, 256) == plan(1228, 1616, 7552, 256) == (11, 4, 0)
    assert plan(544, 4096, 7168, 256) == plan(543, 4096, 7168, 256) == (10, 3, 0) and plan(304, 1632, 2176, 256) == (9, 3, 0)
    assert plan(1024, 1536, 7168, 256) == (28, 2, 0) and plan(1232, 1616, 7552, 304) == (28, 2, 0)
    assert plan(1232, 1608, 7552, 256) != (11, 4, 0) and plan(1232, 1616, 896, 256)[1] == 1 and plan(8192, 8192, 7168, 256)[1] == 1
    # the few-rows kernels where they are well below the tiled plan of one part, not against a K split
    assert plan(256, 3824, 2560, 256) == plan(384, 2048, 2048, 256) == (21, 1, 0) and plan(128, 7344, 4608, 256) == (28, 4, 0)


@pytest.mark.parametrize("shape,plan", [
    ((272, 8192, 7168), (28, 1)), ((256, 8176, 6016), (28, 1)), ((480, 4608, 7168), (28, 1)), ((448, 4608, 7168), (28, 1)),
    ((1616, 1664, 7296), (28, 1)), ((1936, 2272, 7552), (8, 1)), ((960, 4608, 7168), (8, 1)), ((608, 2944, 8064), (28, 2)),
    ((112, 7040, 2304), (12, 1)), ((128, 6912, 2816), (12, 1)), ((224, 4368, 3840), (12, 1))])
def test_long_k_keeps_plans_that_are_faster_where_the_infinity_cache_holds_the_operands(shape, plan):
    """Shapes that an estimate of operands from memory alone moved to plans 6 to 45 % slower (the last three: to few-rows kernels) where
    the operands come from the Infinity Cache."""
    import radeonflow_kernels_amd as rfk
    got = rfk.plan_for(*shape, 256)
    assert (got.variant, got.split_k, got.stream_k) == (*plan, 0)


@pytest.mark.parametrize("shape,plan", [
    ((160, 7968, 6656), (28, 2)), ((176, 7808, 7296), (28, 2)), ((144, 8000, 6784), (28, 2)), ((176, 6016, 6912), (28, 2)),
    ((144, 8192, 7168), (28, 2)), ((176, 7424, 8064), (28, 2)), ((144, 5808, 8192), (8, 4)), ((144, 3584, 3840), (28, 4)),
    ((640, 1536, 3584), (12, 1)), ((592, 1536, 3328), (12, 1)), ((1024, 704, 3072), (12, 1)),
    ((560, 1792, 3200), (28, 1))])
def test_long_k_keeps_plans_that_a_k_split_made_slower(shape, plan):
    """Shapes that split_tile_plan moved to a K split 3 to 25 % slower than the plan that they have without it."""
    import radeonflow_kernels_amd as rfk
    got = rfk.plan_for(*shape, 256)
    assert (got.variant, got.split_k, got.stream_k) == (*plan, 0)


@pytest.mark.parametrize("shape,plan", [
    ((256, 4064, 1664), (28, 1)), ((144, 6208, 1408), (28, 1)), ((208, 4064, 1152), (28, 1)), ((160, 5440, 1152), (28, 1)),
    ((192, 5376, 1280), (12, 1)), ((160, 5824, 1024), (12, 1)), ((240, 2944, 2048), (12, 1)), ((208, 3456, 2304), (12, 1)),
    ((128, 7296, 1152), (28, 1))])
def test_long_k_keeps_tiled_plans_that_few_rows_kernels_made_slower(shape, plan):
    """Shapes that the second comparison moved to few-rows kernels 3 to 13 % slower than the tiles they have without it."""
    import radeonflow_kernels_amd as rfk
    got = rfk.plan_for(*shape, 256)
    assert (got.variant, got.split_k, got.stream_k) == (*plan, 0)


@pytest.mark.parametrize("shape,plan", [((2349, 2064, 26496), (8, 1)), ((1796, 1264, 34304), (10, 3)), ((1904, 512, 24576), (28, 4)),
                                        ((336, 4096, 8320), (28, 2)), ((1360, 1536, 8320), (28, 1)), ((2240, 224, 3328), (12, 1))])
def test_long_k_estimate_is_not_used_beyond_the_sizes_it_was_measured_on(shape, plan):
    """K above 8192 and N below 256: the plans of the model that ranks whole tiles."""
    import radeonflow_kernels_amd as rfk
    got = rfk.plan_for(*shape, 256)
    assert (got.variant, got.split_k, got.stream_k) == (*plan, 0)


def test_long_k_model_states_the_choice_of_the_launcher():
    """tuner/long_k_model.py, where the estimates are measured and fitted: the plans that it puts in place of those of the first model, and
    every plan of its range that is not tabled is one that it would not replace."""
    import radeonflow_kernels_amd as rfk
    from radeonflow_kernels_amd.tuner import long_k_model as lk
    for first, shape in (((28, 1), (1360, 1536, 7168)), ((28, 1), (544, 4096, 7168)), ((28, 1), (304, 1632, 2176)), ((12, 1), (848, 512, 3328)),
                         ((28, 1), (176, 7872, 5376)), ((28, 2), (160, 7968, 6656)), ((12, 1), (640, 1536, 3584)), ((12, 1), (1024, 1024, 4096)),
                         ((28, 8), (48, 4064, 7168))):
        got = rfk.plan_for(*shape, 256)
        assert (got.variant, got.split_k) == lk.replaced(first, *shape), shape
    assert lk.replaced((28, 1), 1328, 1648, 7424) == (11, 4) and lk.replaced((28, 1), 1328, 1648, 7424, 32 << 20) == (10, 3)
    with open(os.path.join(ROOT, "radeonflow_kernels_amd", "csrc", "tuned_plans.inc")) as f:
        tabled = {tuple(int(x) for x in re.findall(r"\d+", l)[:3]) for l in f if l.lstrip().startswith("{")}
    seen = 0
    for shape in lk.shapes(7, 1500):
        plan = rfk.plan_for(*shape, 256)
        if shape not in tabled and plan.variant in lk.TILES and plan.stream_k == 0:
            parts = -(-(shape[2] // 128) // -(-(shape[2] // 128) // plan.split_k))
            to = lk.replaced((plan.variant, parts), *shape)
            # (a plan that took the place of variant 12 may itself give way to variant 9, which 12 does not)
            assert to == (plan.variant, parts) or (to[0] == 9 and shape[0] > 512), (shape, plan, to)
            seen += 1
    assert seen > 400

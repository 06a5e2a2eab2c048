"""CPU tests of the launcher's rules on sizes (csrc/plan_limits.h)."""
import ctypes
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.fixture(scope="module")
def limits(tmp_path_factory):
    """The rules, compiled for the host."""
    d = tmp_path_factory.mktemp("limits")
    src = d / "limits.cpp"
    src.write_text('#include "%s"\nextern "C" int staged(int x, int tile, int other, int k, int p) '
                   '{ return rf::staged_length(x, tile, other, k, p != 0); }\n'
                   'extern "C" int fits(int m, int n, int k) { return rf::persistent_offsets_fit(m, n, k); }\n'
                   'extern "C" int streamed(double bytes, int queue, int columns) { return rf::grouped_weights_streamed(bytes, queue != 0, columns); }\n'
                   % os.path.join(ROOT, "radeonflow_kernels_amd", "csrc", "plan_limits.h"))
    so = str(d / "limits.so")
    subprocess.run(["g++", "-O1", "-shared", "-fPIC", "-o", so, str(src)], check=True)
    lib = ctypes.CDLL(so)
    lib.streamed.argtypes = [ctypes.c_double, ctypes.c_int, ctypes.c_int]
    return lib


@pytest.mark.parametrize("m,n,k", [(2097100, 7168, 2048), (599183, 4608, 7168), (2097030, 7168, 2048), (599160, 4608, 7168)])
def test_staged_rows_stay_within_the_persistent_schedule(limits, m, n, k):
    """K * M just below 2^32 at the planned size: the plan is a persistent one, and the staged rows still allow it (the first two
    went up to the next whole line, whose K * M is 2^32 or more, and the launch was refused; the others have room for it)."""
    import radeonflow_kernels_amd as rfk
    planned, lines = -(-m // 16) * 16, -(-m // 128) * 128
    plan = rfk.plan_for(m, n, k, 256)
    assert plan.stream_k in (2, 3) and limits.fits(planned, n, k)
    tile = {v["variant"]: v["block_m"] for v in rfk.variants()}[plan.variant]
    got = limits.staged(planned, tile, n, k, 1)
    assert planned <= got <= lines and limits.fits(got, n, k)
    assert got == (lines if limits.fits(lines, n, k) else planned)


def test_staged_rows_are_whole_lines_where_that_adds_no_tile(limits):
    for tile in (64, 128, 192, 256):
        for x in list(range(16, 1200, 16)) + [2097104, 33554400, 2147483632]:
            lines = -(-x // 128) * 128
            want = lines if -(-lines // tile) == -(-x // tile) and lines < 2 ** 31 else x
            assert limits.staged(x, tile, 4608, 7168, 0) == want, (x, tile)
            assert limits.staged(x, tile, 4608, 7168, 1) == (want if 7168 * want < 2 ** 32 else x), (x, tile)


def test_weights_the_infinity_cache_can_hold_are_read_without_the_hint(limits):
    """Strips: 13 to 18 groups of 2048 x 7168 (191 to 264 MB) and 23 to 32 of 4096 x 2048 (193 to 268 MB) were up to 36 % slower with
    the non-temporal hint on weights that were in the cache; 294 MB and more are as fast or faster with it everywhere, in strips of
    512 columns whatever the cache cannot hold. The queue form gains from it from 200 MB on."""
    for groups, n, k, want in ((13, 2048, 7168, 0), (18, 2048, 7168, 0), (19, 7168, 2048, 0), (9, 4096, 7168, 0), (23, 4096, 2048, 0),
                               (34, 4096, 2048, 0), (20, 2048, 7168, 1), (10, 4096, 7168, 1), (25, 2048, 7168, 1), (36, 4096, 2048, 1)):
        for columns in (128, 256):
            assert limits.streamed(groups * n * k, 0, columns) == want, (groups, n, k)
    assert limits.streamed(33 * 4096 * 2048, 0, 512) == 1 and limits.streamed(32 * 4096 * 2048, 0, 512) == 0
    assert limits.streamed(26 * 4096 * 2048, 1, 256) == 1 and limits.streamed(23 * 4096 * 2048, 1, 256) == 0


def test_plan_table_slot_is_defined_for_every_set_of_staging_flags(tmp_path):
    """Evaluated by the compiler, which refuses a constant expression that overflows a signed product (flags of 4 and more did):
    every set of flags there is, the largest sizes."""
    src = tmp_path / "slot.cpp"
    src.write_text('#include "%s"\ntemplate <int S> constexpr bool below() {\n    constexpr unsigned a = rf::plan_slot(2147483647, 2147483647, 2147483520, S, 1024), '
                   'b = rf::plan_slot(1, 1, 128, S, 1024);\n    static_assert(a < 1024 && b < 1024, "");\n    if constexpr (S > 0) return below<S - 1>();\n'
                   '    return true;\n}\nstatic_assert(below<(1 << rf::kStageBits) - 1>(), "");\n' % os.path.join(ROOT, "radeonflow_kernels_amd", "csrc", "plan_limits.h"))
    subprocess.run(["g++", "-std=c++17", "-fsyntax-only", str(src)], check=True)

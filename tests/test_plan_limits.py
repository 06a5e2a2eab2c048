"""CPU test of how long the rows of a staged operand become (csrc/plan_limits.h) under the plan that was chosen for them."""
import ctypes
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.fixture(scope="module")
def limits(tmp_path_factory):
    """rf::staged_length and rf::persistent_offsets_fit, compiled for the host."""
    d = tmp_path_factory.mktemp("limits")
    src = d / "limits.cpp"
    src.write_text('#include "%s"\nextern "C" int staged(int x, int tile, int other, int k, int p) '
                   '{ return rf::staged_length(x, tile, other, k, p != 0); }\n'
                   'extern "C" int fits(int m, int n, int k) { return rf::persistent_offsets_fit(m, n, k); }\n'
                   % os.path.join(ROOT, "radeonflow_kernels_amd", "csrc", "plan_limits.h"))
    so = str(d / "limits.so")
    subprocess.run(["g++", "-O1", "-shared", "-fPIC", "-o", so, str(src)], check=True)
    return ctypes.CDLL(so)


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

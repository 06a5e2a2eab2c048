"""The staging copy of ragged operands: rows shorter than a workgroup, odd widths, the last bytes of the matrix."""
import numpy as np
import pytest
import torch

from helpers import bf16_bits, exact_problem, oracle_bf16, to_gpu

pytestmark = pytest.mark.gpu


# widths of one piece, of pieces that do not divide a workgroup's 256 threads, of exactly 256 pieces and of one piece more; an
# explicit tiled plan refuses ragged shapes, so the grouped entry point with one group and a tiled form makes the copy run
@pytest.mark.parametrize("m", [1, 15, 17, 81, 1001, 4095, 4097])
def test_staged_rows_bit_exact(m):
    import radeonflow_kernels_amd as rfk
    n, k = 256, 256 if m > 64 else 32768
    data = exact_problem(m, n, k, seed=m)
    exp = oracle_bf16(data)
    g, buf = to_gpu(data, 300)
    a, b, sa, sb, c = g
    c.fill_(-1.0)
    rfk.fp8_mm_grouped(a, b.T.contiguous().T.unsqueeze(0), sa, sb.T.contiguous().T.unsqueeze(0), c, [0, m], variant=1)
    torch.cuda.synchronize()
    assert np.array_equal(bf16_bits(c), exp)
    assert float(buf[m * n:].float().min()) == -7.0 == float(buf[m * n:].float().max())


# more rows than the few-rows kernels take with a ragged width, so the plan is a tiled one: tiles that store into the ragged C
# and, where K is split (17 columns of it long), a padded C written back; widths below a piece of eight, rows of a
# workgroup's 256 pieces and a few more; c at an odd element, also with a width that needs nothing else
@pytest.mark.parametrize("m,n,k,off_c", [(4112, 5, 512, 0), (4100, 130, 256, 0), (4128, 2045, 128, 1), (4099, 2057, 128, 0),
                                         (4112, 17, 7168, 0), (4112, 17, 7168, 3), (4112, 1008, 256, 5)])
def test_staged_output_bit_exact(m, n, k, off_c):
    import radeonflow_kernels_amd as rfk
    data = exact_problem(m, n, k, seed=n)
    exp = oracle_bf16(data)
    g, _ = to_gpu(data, 300)
    buf = torch.full((m * n + 300,), -7.0, dtype=torch.bfloat16, device="cuda")
    c = buf[off_c:off_c + m * n].view(m, n)
    rfk.fp8_mm(*g[:4], c)
    torch.cuda.synchronize()
    assert np.array_equal(bf16_bits(c), exp)
    rest = torch.cat([buf[:off_c], buf[off_c + m * n:]]).float()
    assert float(rest.min()) == -7.0 == float(rest.max())


def test_every_tile_kernel_stores_into_any_c(tmp_path):
    """Plan files name each tile variant for the padded shape: its form for a ragged C gives the oracle's bits and leaves what
    lies around C alone."""
    import radeonflow_kernels_amd as rfk
    m, n, k = 4101, 205, 256
    data = exact_problem(m, n, k, seed=7)
    exp = oracle_bf16(data)
    g, _ = to_gpu(data, 300)
    plan = tmp_path / "p.plans"
    for variant in range(12):
        plan.write_text("4112 208 256 %d 1 8 0\n" % variant)
        buf = torch.full((m * n + 301,), -7.0, dtype=torch.bfloat16, device="cuda")
        try:
            assert rfk.load_plans(str(plan)) == 1 and rfk.plan_for(m, n, k, 256).variant == variant
            rfk.fp8_mm(*g[:4], buf[1:1 + m * n].view(m, n))
            torch.cuda.synchronize()
        finally:
            rfk.clear_plans()
        assert np.array_equal(bf16_bits(buf[1:1 + m * n].view(m, n)), exp), variant
        assert float(buf[0]) == -7.0 and float(buf[1 + m * n:].float().min()) == -7.0 == float(buf[1 + m * n:].float().max())


# 530 rows are planned as 544 and staged as 640 (whole lines) where that adds no tile: every schedule, K in one and in several
# parts (whose sums are of the true rows only), tiles of 192 rows that 640 would need one more of; 520 rows need no more lines
# with 64-row units than with 16; N = 500 (B staged, planned as 512 or 496)
@pytest.mark.parametrize("m,n,k,plan", [(530, 512, 512, "3 1 8 0"), (530, 512, 512, "8 3 8 0"), (530, 512, 512, "5 1 8 0"),
                                        (530, 512, 512, "28 4 8 0"), (530, 512, 512, "0 1 8 2"), (530, 512, 512, "0 1 8 4"),
                                        (520, 512, 256, "0 1 8 4"), (530, 512, 512, "0 1 8 1"), (577, 500, 384, "10 1 8 0"),
                                        (577, 490, 384, "8 1 8 0"), (577, 490, 384, "3 3 8 0"), (641, 130, 256, "28 1 8 0")])
def test_staged_rows_of_whole_lines(tmp_path, m, n, k, plan):
    import radeonflow_kernels_amd as rfk
    data = exact_problem(m, n, k, seed=m + n)
    exp = oracle_bf16(data)
    g, buf = to_gpu(data, 300)
    path = tmp_path / "p.plans"
    path.write_text("%d %d %d %s\n" % ((m + 15) // 16 * 16, (n + 15) // 16 * 16, k, plan))
    try:
        assert rfk.load_plans(str(path)) == 1
        for fill in (-1.0, 3.0):
            g[4].fill_(fill)
            rfk.fp8_mm(*g)
            torch.cuda.synchronize()
            assert np.array_equal(bf16_bits(g[4]), exp)
    finally:
        rfk.clear_plans()
    assert float(buf[m * n:].float().min()) == -7.0 == float(buf[m * n:].float().max())

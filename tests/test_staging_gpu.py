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

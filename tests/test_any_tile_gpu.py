"""The any-alignment tile kernels (variants 29 and 30): operands of any width at any byte through registers, K split into parts that
reduce_splitk_any_c adds."""
import numpy as np
import pytest
import torch

from helpers import bf16_bits, exact_problem, oracle_bf16, to_gpu

pytestmark = pytest.mark.gpu
ANY_TILES = (29, 30)


@pytest.fixture(scope="module")
def rfk():
    import radeonflow_kernels_amd as r
    assert torch.cuda.is_available(), "these tests need the GPU"
    r.lib()
    return r


# one element, one short of and one past the tiles' 128 rows and 128 and 256 columns, whole tiles, one K block (the matrix's cut
# last one comes first), even and odd numbers of them, K parts of unequal length
@pytest.mark.parametrize("m,n,k", [(1, 1, 128), (3, 5, 256), (127, 255, 384), (128, 256, 128), (129, 257, 640), (200, 130, 896),
                                   (16, 1000, 1280), (300, 515, 2176)])
def test_any_tile_bit_exact(rfk, m, n, k):
    """Exact data: the oracle's bits for every plan, nothing stored past the end of C."""
    data = exact_problem(m, n, k, seed=3 * m + n + k)
    exp = oracle_bf16(data)
    g, buf = to_gpu(data, 300)
    for v in ANY_TILES:
        for split in (1, 2, 3, 5, 9):
            if split > k // 128:
                continue
            g[4].fill_(-1.0)
            rfk.fp8_mm(*g, config=rfk.GemmConfig(v, split, 4, 0))
            torch.cuda.synchronize()
            assert np.array_equal(bf16_bits(g[4]), exp), "variant %d split %d" % (v, split)
    assert float(buf[m * n:].float().min()) == -7.0 == float(buf[m * n:].float().max())


@pytest.mark.parametrize("off_a,off_b,off_c", [(1, 0, 0), (0, 3, 0), (6, 2, 1), (15, 13, 3)])
@pytest.mark.parametrize("m,n", [(144, 272), (131, 259)])
def test_any_tile_takes_operands_at_any_byte(rfk, m, n, off_a, off_b, off_c):
    """Operands that start off_a, off_b bytes (C: off_c elements) into aligned buffers that end with them."""
    k = 640
    data = exact_problem(m, n, k, seed=m + off_a)
    exp = oracle_bf16(data)
    a, b, sa, sb = to_gpu(data)[:4]

    def shifted(t, off):
        rows, cols = t.shape
        flat = torch.empty(rows * cols + off, dtype=torch.uint8, device="cuda")
        flat[off:].copy_(t.T.contiguous().view(torch.uint8).reshape(-1))
        return flat[off:].view(torch.float8_e4m3fn).view(cols, rows).T

    for cfg in (rfk.GemmConfig(29, 1, 8, 0), rfk.GemmConfig(30, 2, 8, 0), None):
        c = torch.zeros(m * n + off_c, dtype=torch.bfloat16, device="cuda")[off_c:].view(m, n)
        rfk.fp8_mm(shifted(a, off_a), shifted(b, off_b), sa, sb, c, config=cfg)
        torch.cuda.synchronize()
        assert np.array_equal(bf16_bits(c), exp), "plan %r" % (cfg,)


@pytest.mark.parametrize("m,n,k", [(513, 2003, 256), (700, 203, 7168), (3001, 1531, 256)])
def test_any_tile_automatic_static_and_captured(rfk, m, n, k):
    """Shapes whose automatic plan is such a tile, with and without a K split: the same bits from the automatic plan, the entry that
    allocates nothing, and replays of a captured launch with other work in between; and the bits of the same K parts on the tiled
    kernels, with rounding in every product."""
    plan = rfk.select_config(m, n, k)
    assert plan.variant in ANY_TILES
    data = exact_problem(m, n, k, seed=m)
    exp = oracle_bf16(data)
    g = to_gpu(data)
    for call in (rfk.fp8_mm, rfk.fp8_mm_static):
        g[4].zero_()
        call(*g)
        torch.cuda.synchronize()
        assert np.array_equal(bf16_bits(g[4]), exp)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        rfk.fp8_mm(*g)
    for rep in range(3):
        g[4].fill_(-1.0)
        rfk.fp8_mm(g[0], g[1], g[2], g[3], torch.empty_like(g[4]))
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        assert np.array_equal(bf16_bits(g[4]), exp), "replay %d" % rep


@pytest.mark.parametrize("split", [1, 3])
def test_any_tile_bits_of_the_tiled_kernel(rfk, split):
    """Rounding in every product: the sums of the 128 x 128 tile kernel with the same K parts, to the bit."""
    m, n, k, fp8 = 208, 336, 2304, torch.float8_e4m3fn
    gen = torch.Generator(device="cuda").manual_seed(split)
    a = torch.randint(0, 120, (k, m), dtype=torch.uint8, device="cuda", generator=gen).view(fp8).T
    b = torch.randint(0, 120, (k, n), dtype=torch.uint8, device="cuda", generator=gen).view(fp8).T
    sa = (torch.rand((k // 128, m), device="cuda", generator=gen) * 1e-2).T
    sb = (torch.rand((k // 128, (n + 127) // 128), device="cuda", generator=gen) * 1e-2).T
    outs = []
    for v in (1, 28) + ANY_TILES:
        c = torch.zeros((m, n), dtype=torch.bfloat16, device="cuda")
        rfk.fp8_mm(a, b, sa, sb, c, config=rfk.GemmConfig(v, split, 8, 0))
        torch.cuda.synchronize()
        outs.append(bf16_bits(c))
    for o in outs[1:]:
        assert np.array_equal(o, outs[0])


def test_any_tile_nan_and_infinity(rfk):
    """A NaN code and an infinite scale reach their row and column of C and no other element."""
    m, n, k = 130, 259, 512
    a, b, sa, sb, c = exact_problem(m, n, k, 7)
    a8, b8, sa = a.view(torch.uint8).clone(), b.view(torch.uint8).clone(), sa.clone()
    a8[m // 2, 17] = 0x7F
    b8[n - 1, k - 1] = 0xFF
    sa[m - 1, 0] = float("inf")
    data = (a8.view(a.dtype), b8.view(b.dtype), sa, sb, c)
    clean = oracle_bf16((a, b, torch.where(torch.isinf(sa), torch.zeros_like(sa), sa), sb, c)).reshape(m, n)
    g = to_gpu(data)
    for v, split in ((29, 1), (30, 1), (29, 2)):
        rfk.fp8_mm(*g, config=rfk.GemmConfig(v, split, 8, 0))
        torch.cuda.synchronize()
        got = g[4].float().cpu()
        assert torch.isnan(got[m // 2]).all() and torch.isnan(got[:, n - 1]).all()
        keep = np.ones((m, n), bool)
        keep[[m // 2, m - 1]] = False
        keep[:, n - 1] = False
        assert np.array_equal(bf16_bits(g[4]).reshape(m, n)[keep], clean[keep])
        assert not torch.isfinite(got[m - 1]).any()


# rows of A or B of 17 million bytes: 127 of them, and C and the K parts' sums, are beyond 2^31
@pytest.mark.parametrize("m,n,plans", [(130, 17000003, ((29, 1), (30, 1))), (17000003, 16, ((29, 1), (30, 1), (29, 2)))])
def test_any_tile_offsets_beyond_31_bits(rfk, m, n, plans):
    k, fp8 = 256, torch.float8_e4m3fn
    gen = torch.Generator(device="cuda").manual_seed(n)

    def signed_ones_and_twos(shape):                           # codes of 1, 2, -1 and -2
        x = torch.randint(0, 4, shape, dtype=torch.uint8, device="cuda", generator=gen)
        return 0x38 + ((x & 1) << 3) + ((x & 2) << 6)

    a, b = (signed_ones_and_twos((k, x)).view(fp8) for x in (m, n))
    sa = torch.randint(1, 3, (2, m), device="cuda", generator=gen).float()
    sb = torch.randint(1, 3, (2, (n + 127) // 128), device="cuda", generator=gen).float()
    buf = torch.full((m * n + 300,), -7.0, dtype=torch.bfloat16, device="cuda")
    c = buf[:m * n].view(m, n)
    step = 1 << 20
    for v, split in plans:
        c.fill_(-7.0)
        rfk.fp8_mm(a.T, b.T, sa.T, sb.T, c, config=rfk.GemmConfig(v, split, 8, 0))
        for x0 in range(0, max(m, n), step):                   # sums of integers below 2^12: exact in any order
            rows, cols = (slice(None), slice(x0, x0 + step)) if n > m else (slice(x0, x0 + step), slice(None))
            exp = 0
            for kb in range(2):
                part = a[kb * 128:kb * 128 + 128, rows].float().T @ b[kb * 128:kb * 128 + 128, cols].float()
                exp = exp + part * sa[kb, rows][:, None] * sb[kb].repeat_interleave(128)[:n][cols][None, :]
            assert torch.equal(c[rows, cols], exp.bfloat16()), (v, split, x0)
        assert float(buf[m * n:].float().min()) == -7.0 == float(buf[m * n:].float().max()), (v, split)

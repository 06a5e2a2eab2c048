"""The few-rows kernels (variants 14 to 21): any shape and alignment, K split between waves and between workgroups."""
import numpy as np
import pytest
import torch

from helpers import bf16_bits, exact_problem, oracle_bf16, to_gpu

pytestmark = pytest.mark.gpu
FEW_ROWS = range(14, 22)


@pytest.fixture(scope="module")
def rfk():
    import radeonflow_kernels_amd as r
    assert torch.cuda.is_available(), "these tests need the GPU"
    r.lib()
    return r


# edges of the 16-row tiles and of the 32 to 128 column strips, one K block (seven idle waves), K blocks that do and do not
# divide among eight waves and splits; M = 1 and N = 1: loads of the last rows are cut at the matrix's end
@pytest.mark.parametrize("m,n,k", [(1, 1, 128), (1, 7168, 256), (2, 130, 1152), (15, 33, 2432), (16, 144, 1024), (17, 127, 3200),
                                   (31, 257, 640), (33, 500, 2048), (64, 96, 7168), (65, 129, 896), (130, 47, 384)])
def test_fewrows_bit_exact_on_any_shape(rfk, m, n, k):
    """Exact data: every plan gives the oracle's bits whatever its summation order, nothing is stored past the end of C; two
    launches in a row (the arrival counters of a K split are back at zero)."""
    data = exact_problem(m, n, k, seed=5 * m + n + k)
    exp = oracle_bf16(data)
    g, buf = to_gpu(data, 300)
    for v in FEW_ROWS:
        for split in (1, 2, 5):
            if split > k // 128:
                continue
            for rep in range(2):
                g[4].fill_(-1.0)
                rfk.fp8_mm(*g, config=rfk.GemmConfig(v, split, 1, 0))
                torch.cuda.synchronize()
                assert np.array_equal(bf16_bits(g[4]), exp), "variant %d split %d launch %d" % (v, split, rep)
    assert float(buf[m * n:].float().min()) == -7.0 == float(buf[m * n:].float().max())


# tiles whose waves have their next K block on its way (16, 20, 21 and 22 to 27): waves with none, one, two and several K blocks,
# counts that differ between the waves, the matrix's cut last K block as a wave's first, second and later one
@pytest.mark.parametrize("m,n,k", [(1, 33, 128), (17, 100, 896), (33, 300, 1024), (31, 257, 1152), (100, 130, 2176), (64, 1000, 4096)])
def test_fewrows_pipelined_tiles_bit_exact(rfk, m, n, k):
    data = exact_problem(m, n, k, seed=m + n + k)
    exp = oracle_bf16(data)
    g, buf = to_gpu(data, 300)
    for v in (16, 20, 21) + tuple(range(22, 28)):
        for split in (1, 2, 5):
            if split > k // 128:
                continue
            g[4].fill_(-1.0)
            rfk.fp8_mm(*g, config=rfk.GemmConfig(v, split, 1, 0))
            torch.cuda.synchronize()
            assert np.array_equal(bf16_bits(g[4]), exp), "variant %d split %d" % (v, split)
    assert float(buf[m * n:].float().min()) == -7.0 == float(buf[m * n:].float().max())


@pytest.mark.parametrize("off_a,off_b,off_c", [(1, 0, 0), (0, 3, 0), (7, 15, 1), (16, 16, 2)])
def test_fewrows_takes_operands_at_any_byte(rfk, off_a, off_b, off_c):
    """Operands that start off_a, off_b bytes (C: off_c elements) into 16-byte aligned buffers, under the automatic plan and an
    explicit one; the buffers end with the operands, so a load past the end would leave the allocation's data."""
    m, n, k = 24, 176, 1280
    data = exact_problem(m, n, k, seed=11)
    exp = oracle_bf16(data)
    a, b, sa, sb = to_gpu(data)[:4]

    def shifted(t, off):
        rows, cols = t.shape
        flat = torch.empty(rows * cols + off, dtype=torch.uint8, device="cuda")
        flat[off:].copy_(t.T.contiguous().view(torch.uint8).reshape(-1))
        return flat[off:].view(torch.float8_e4m3fn).view(cols, rows).T

    for cfg in (None, rfk.GemmConfig(18, 3, 1, 0)):
        c = torch.zeros(m * n + off_c, dtype=torch.bfloat16, device="cuda")[off_c:].view(m, n)
        rfk.fp8_mm(shifted(a, off_a), shifted(b, off_b), sa, sb, c, config=cfg)
        torch.cuda.synchronize()
        assert np.array_equal(bf16_bits(c), exp), "plan %r" % (cfg,)


def test_fewrows_static_entry_and_graph_replay(rfk):
    """The allocation-free entry (its own counters and slots) and replays of a captured launch give the same bits."""
    m, n, k = 7, 1536, 7168
    plan = rfk.select_config(m, n, k)
    assert plan.variant in FEW_ROWS and plan.split_k > 1
    data = exact_problem(m, n, k, seed=3)
    exp = oracle_bf16(data)
    g = to_gpu(data)
    rfk.fp8_mm(*g)
    torch.cuda.synchronize()
    assert np.array_equal(bf16_bits(g[4]), exp)
    for rep in range(2):
        g[4].zero_()
        rfk.fp8_mm_static(*g)
        torch.cuda.synchronize()
        assert np.array_equal(bf16_bits(g[4]), exp)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        rfk.fp8_mm_static(*g)
    for rep in range(3):
        g[4].fill_(-1.0)
        rfk.fp8_mm(g[0], g[1], g[2], g[3], torch.empty_like(g[4]))
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        assert np.array_equal(bf16_bits(g[4]), exp), "replay %d" % rep


# groups at the edges of the 16 and 32 row blocks and over them, idle ones, starting at any byte; K blocks fewer than, as many as
# and no multiple of a workgroup's waves; widths that end inside a 256, 128 and 64 column strip
@pytest.mark.parametrize("rows,n,k", [([1], 16, 2048), ([3, 0, 16, 17, 1, 32, 33], 144, 1152), ([15, 16, 48], 272, 128),
                                      ([0, 2, 70, 5] * 3, 320, 3328), ([int(x) for x in np.arange(64) % 5], 256, 1024)])
@pytest.mark.parametrize("shift", [0, 5])
def test_grouped_fewrows_bits_of_the_tiled_form(rfk, rows, n, k, shift):
    """Rounding in every product: the few-rows forms sum K blocks in order and so give the bits of the 128 x 256 tiles, on
    operands back to back (a at any byte, its buffer ending with it) and in the padded layout; rows of C past the groups keep
    their fill."""
    fp8, groups = torch.float8_e4m3fn, len(rows)
    offs = [0] + [int(x) for x in np.cumsum(rows)]
    m = offs[-1]
    gen = torch.Generator(device="cuda").manual_seed(m + n + k)
    raw = torch.randint(0, 120, (k * m + shift,), dtype=torch.uint8, device="cuda", generator=gen)
    a = raw[shift:].view(k, m).view(fp8).T
    b = torch.randint(0, 120, (groups, k, n), dtype=torch.uint8, device="cuda", generator=gen).view(fp8).permute(0, 2, 1)
    sa = (torch.rand((k // 128, m), device="cuda", generator=gen) * 1e-2).T
    sb = (torch.rand((groups, k // 128, (n + 127) // 128), device="cuda", generator=gen) * 1e-2).permute(0, 2, 1)
    pad = rfk.grouped_padded_offsets(offs)
    a_pad, sa_pad = torch.zeros((k, pad[-1]), dtype=torch.uint8, device="cuda"), torch.ones((k // 128, pad[-1]), device="cuda")
    for g in range(groups):
        a_pad[:, pad[g]:pad[g] + rows[g]] = a.T.view(torch.uint8)[:, offs[g]:offs[g + 1]]
        sa_pad[:, pad[g]:pad[g] + rows[g]] = sa.T[:, offs[g]:offs[g + 1]]

    def launch(call, x, sx, variant):
        buf = torch.full((m * n + 300,), -7.0, dtype=torch.bfloat16, device="cuda")
        call(x, b, sx, sb, buf[:m * n].view(m, n), offs, variant=variant)
        torch.cuda.synchronize()
        return bf16_bits(buf)

    expect = launch(rfk.fp8_mm_grouped, a, sa, 1)
    for variant in (6, 7, 8, 9, -1):
        assert np.array_equal(launch(rfk.fp8_mm_grouped, a, sa, variant), expect), variant
        assert np.array_equal(launch(rfk.fp8_mm_grouped_padded, a_pad.view(fp8).T, sa_pad.T, variant), expect), variant


# groups of at most 16 rows for the strips, of up to 300 for the queue's tiles of four heights and of one and two row tiles; a
# partial last strip of any width, an odd number of K blocks. Weights of the groups that have rows: 328 MB for the strips and 369
# for the queue (both read with the non-temporal hint), 197 (without) and 221 (with it), 82 and 90 (both without)
@pytest.mark.parametrize("variants,rows", [((6, 7, 8, 10, -1), [1, 0, 16, 7, 3]), ((5,), [64, 0, 300, 65, 130, 200, 256, 1, 257, 20])])
@pytest.mark.parametrize("groups", [50, 30, 12])
def test_grouped_streamed_weights_bits_of_the_tiled_form(rfk, variants, rows, groups):
    n, k, fp8 = 2064, 3968, torch.float8_e4m3fn
    rows = (rows * groups)[:groups]
    offs = [0] + [int(x) for x in np.cumsum(rows)]
    m = offs[-1]
    gen = torch.Generator(device="cuda").manual_seed(groups + m)
    a = torch.randint(0, 120, (k, m), dtype=torch.uint8, device="cuda", generator=gen).view(fp8).T
    b = torch.randint(0, 120, (groups, k, n), dtype=torch.uint8, device="cuda", generator=gen).view(fp8).permute(0, 2, 1)
    sa = (torch.rand((k // 128, m), device="cuda", generator=gen) * 1e-2).T
    sb = (torch.rand((groups, k // 128, (n + 127) // 128), device="cuda", generator=gen) * 1e-2).permute(0, 2, 1)

    def launch(variant):
        buf = torch.full((m * n + 300,), -7.0, dtype=torch.bfloat16, device="cuda")
        rfk.fp8_mm_grouped(a, b, sa, sb, buf[:m * n].view(m, n), offs, variant=variant)
        torch.cuda.synchronize()
        return bf16_bits(buf)

    expect = launch(1)
    for variant in variants:
        assert np.array_equal(launch(variant), expect), variant


def test_fewrows_k_splits_on_two_streams_at_once(rfk):
    """Different numbers of K parts on two streams, launches queued deep: every stream has counters and slots of its own, so each
    result is the one the same plan gives alone."""
    problems = [(to_gpu(exact_problem(m, n, k, m + k)), oracle_bf16(exact_problem(m, n, k, m + k)), cfg)
                for m, n, k, cfg in ((7, 1536, 7168, rfk.GemmConfig(14, 4, 8, 0)), (40, 1000, 4096, rfk.GemmConfig(17, 7, 8, 0)))]
    streams = [torch.cuda.Stream() for _ in problems]
    outs = [[torch.full_like(g[4], -1.0) for _ in range(40)] for g, _, _ in problems]
    torch.cuda.synchronize()
    for i in range(40):
        for (g, _, cfg), s, out in zip(problems, streams, outs):
            with torch.cuda.stream(s):
                rfk.fp8_mm(*g[:4], out[i], config=cfg)
    torch.cuda.synchronize()
    for (_, exp, _), out in zip(problems, outs):
        for i, c in enumerate(out):
            assert np.array_equal(bf16_bits(c), exp), i


def _signed_ones_and_twos(shape, gen):
    """e4m3fn codes of +-1 and +-2."""
    r = torch.randint(0, 4, shape, dtype=torch.uint8, device="cuda", generator=gen)
    return 0x38 + ((r & 1) << 3) + ((r & 2) << 6)


# 127 rows of a K block from 16,909,320 columns on are more than 2^31 bytes: a width that starts at any byte and one of aligned
# rows, and the same many rows of A
@pytest.mark.parametrize("m,n", [(3, 17000003), (3, 17000016), (17000003, 16)])
def test_fewrows_offsets_beyond_31_bits(rfk, m, n):
    k, fp8 = 256, torch.float8_e4m3fn
    gen = torch.Generator(device="cuda").manual_seed(n)
    a, b = (_signed_ones_and_twos((k, x), gen).view(fp8) for x in (m, n))
    sa = torch.randint(1, 3, (2, m), device="cuda", generator=gen).float()
    sb = torch.randint(1, 3, (2, (n + 127) // 128), device="cuda", generator=gen).float()
    buf = torch.full((m * n + 300,), -7.0, dtype=torch.bfloat16, device="cuda")
    c = buf[:m * n].view(m, n)
    plans = FEW_ROWS if m == 3 else (14, 18, 21)
    for v in plans:
        c.fill_(-7.0)
        rfk.fp8_mm(a.T, b.T, sa.T, sb.T, c, config=rfk.GemmConfig(v, 1, 8, 0))
        step = 1 << 20
        for x0 in range(0, max(m, n), step):                   # sums of integers below 2^12: exact in any order
            rows, cols = (slice(None), slice(x0, x0 + step)) if n > m else (slice(x0, x0 + step), slice(None))
            exp = 0
            for kb in range(2):
                part = a[kb * 128:kb * 128 + 128, rows].float().T @ b[kb * 128:kb * 128 + 128, cols].float()
                scale_n = sb[kb].repeat_interleave(128)[:n][cols]
                exp = exp + part * sa[kb, rows][:, None] * scale_n[None, :]
            assert torch.equal(c[rows, cols], exp.bfloat16()), (v, x0)
        assert float(buf[m * n:].float().min()) == -7.0 == float(buf[m * n:].float().max()), v


def _with_nans_and_infinities(m, n, k, seed):
    """Exact data with NaN codes in one row of A and one column of B and infinite scales; the expected bits, K blocks folded one
    after the other, and where they are NaN."""
    from oracle import cref
    a, b, sa, sb, c = exact_problem(m, n, k, seed)
    fp8 = torch.float8_e4m3fn
    a8, b8, sa, sb = a.view(torch.uint8).clone(), b.view(torch.uint8).clone(), sa.clone(), sb.clone()
    a8[m // 2, 17] = 0x7F
    b8[n - 1, k - 1] = 0xFF
    sa[m - 1, 0] = float("inf")
    sb[0, k // 128 - 1] = float("-inf")
    sa[0, k // 128 - 1] = 0.0                                  # 0 * -inf
    exp = cref.ref_gemm_blockfold(*(x.T.contiguous().view(torch.uint8).numpy() for x in (a8, b8)),
                                  *(x.T.contiguous().numpy() for x in (sa, sb)), rows=np.arange(m))[1]
    nan = (exp & 0x7FFF) > 0x7F80
    assert nan[m // 2].all() and nan[:, n - 1].all() and nan[0, :min(n, 128)].all() and not nan.all()
    assert ((exp[m - 1] & 0x7FFF) == 0x7F80).any()
    return (a8.view(fp8), b8.view(fp8), sa, sb, c), exp, nan


def _assert_same_values_and_nans(c, exp, nan, what):
    got = bf16_bits(c)
    assert np.array_equal((got & 0x7FFF) > 0x7F80, nan), what
    assert np.array_equal(got[~nan], exp[~nan]), what


@pytest.mark.parametrize("m,n,k", [(7, 300, 1280), (40, 160, 1024)])
def test_fewrows_nan_codes_and_infinite_scales(rfk, m, n, k):
    """NaN and infinity come out where the oracle has them, under every variant with and without a K split (a sum of splits
    meets infinities of one sign only: one K block per row and column has them)."""
    data, exp, nan = _with_nans_and_infinities(m, n, k, 4)
    g = to_gpu(data)
    for cfg in [None] + [rfk.GemmConfig(v, s, 8, 0) for v in FEW_ROWS for s in (1, 3)]:
        g[4].fill_(-1.0)
        rfk.fp8_mm(*g, config=cfg)
        torch.cuda.synchronize()
        _assert_same_values_and_nans(g[4], exp, nan, "plan %r" % (cfg,))


def test_stores_into_any_c_keep_nans_and_infinities(rfk, tmp_path):
    """The tile kernels' stores into a ragged C (plan files name the tile for the padded shape)."""
    m, n, k = 4101, 205, 256
    data, exp, nan = _with_nans_and_infinities(m, n, k, 9)
    g = to_gpu(data)
    plan = tmp_path / "p.plans"
    for variant in range(12):
        plan.write_text("4112 208 256 %d 1 8 0\n" % variant)
        buf = torch.full((m * n + 1,), -7.0, dtype=torch.bfloat16, device="cuda")
        c = buf[1:].view(m, n)
        try:
            assert rfk.load_plans(str(plan)) == 1 and rfk.plan_for(m, n, k, 256).variant == variant
            rfk.fp8_mm(*g[:4], c)
            torch.cuda.synchronize()
        finally:
            rfk.clear_plans()
        _assert_same_values_and_nans(c, exp, nan, variant)


@pytest.mark.parametrize("m,n,k", [(513, 256, 2048), (1833, 256, 2048), (848, 576, 1024), (665, 1536, 384), (2500, 256, 2048)])
def test_fewrows_as_the_plan_of_many_rows(rfk, m, n, k):
    """More than 512 rows and a small N: the automatic plan is a few-rows kernel, with the oracle's bits from both entries."""
    assert 14 <= rfk.select_config(m, n, k).variant <= 27
    data = exact_problem(m, n, k, seed=m)
    exp = oracle_bf16(data)
    g, buf = to_gpu(data, 300)
    for call in (rfk.fp8_mm, rfk.fp8_mm_static):
        g[4].fill_(-1.0)
        call(*g)
        torch.cuda.synchronize()
        assert np.array_equal(bf16_bits(g[4]), exp)
    assert float(buf[m * n:].float().min()) == -7.0 == float(buf[m * n:].float().max())

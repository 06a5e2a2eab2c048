"""GPU test of rf_fp8_gemm_static, the entry point that allocates nothing: its output equals rf_fp8_gemm's bit for bit
on calls that use the static scratch array in different ways, one after the other."""
import ctypes

import numpy as np
import pytest
import torch

from oracle import ref_kernel as rk
from helpers import RTOL, ATOL, assert_close_to_oracle, bf16_bits, oracle_bf16, to_gpu

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def rfk():
    import radeonflow_kernels_amd as r
    assert torch.cuda.is_available(), "these tests need the GPU"
    r.lib()
    return r


def _both(rfk, data):
    g = to_gpu(data)
    rfk.fp8_mm(*g)
    torch.cuda.synchronize()
    want = bf16_bits(g[4]).copy()
    g[4].fill_(-3.0)
    free_before = torch.cuda.mem_get_info()[0]
    rfk.fp8_mm_static(*g)
    torch.cuda.synchronize()
    assert torch.cuda.mem_get_info()[0] == free_before, "the call changed the amount of free device memory"
    return bf16_bits(g[4]), want


def test_static_entry_matches_the_allocating_entry_on_two_calls_in_a_row(rfk):
    """First the C1 shape (split-K: 25 MB of partial sums in the scratch array), then a smaller ragged shape (staging
    copies and split-K partials at other offsets of the same array, which still holds the first call's data), then a
    shape that needs no scratch memory at all. Every result equals rf_fp8_gemm's bits and the oracle within tolerance."""
    assert rfk.lib().rf_gemm_static_scratch_bytes() == 32 << 20
    m, n, k = 1024, 1536, 7168
    assert rfk.select_config(m, n, k).split_k > 1
    for shape, seed in (((m, n, k), 21), ((250, 576, 2048), 22), ((512, 512, 1024), 23), ((1000, 1536, 7168), 24)):
        data = rk.generate_input_blockquant(*shape, seed)
        got, want = _both(rfk, data)
        assert np.array_equal(got, want), "shape %r differs from rf_fp8_gemm" % (shape,)
        assert_close_to_oracle(torch.from_numpy(got.view(np.int16)).view(torch.bfloat16), oracle_bf16(data), RTOL, ATOL,
                               "static %r" % (shape,))


def test_static_entry_fits_the_plan_to_its_scratch_array(rfk, tmp_path):
    """Shapes whose plan under rf_fp8_gemm needs more than the 32 MiB array still run, and allocate nothing:
    * M = 5001 with K = 7168 (36 MB of A): not staged, on tiles that take it as it is, with the K parts that fit;
    * the same with a ragged N as well;
    * a plan file that asks for four K parts of 16.8 MB each: cut down to one part;
    * a stream-K plan from a plan file: replaced by the automatic plan.
    Exact data, so every fitted plan must give the oracle's bits (and rf_fp8_gemm's); then data with rounding in it
    against the oracle within tolerance; the canary behind C stays intact; a small split-K shape afterwards still matches
    rf_fp8_gemm bit for bit (the array holds the earlier calls' data)."""
    from helpers import exact_problem
    L = rfk.lib()

    def static_run(data, canary=4096):
        g, buf = to_gpu(data, canary_elems=canary)
        g[4].fill_(-3.0)
        free_before = torch.cuda.mem_get_info()[0]
        rfk.fp8_mm_static(*g)
        torch.cuda.synchronize()
        assert torch.cuda.mem_get_info()[0] == free_before, "the call changed the amount of free device memory"
        assert bool((buf[g[4].numel():].float() == -7.0).all()), "store past the end of C"
        return g[4]

    for (m, n, k) in ((5001, 512, 7168), (5001, 500, 7168)):
        assert k * ((m + 15) // 16 * 16) > (32 << 20)
        data = exact_problem(m, n, k, seed=m + n)
        assert np.array_equal(bf16_bits(static_run(data)), oracle_bf16(data)), (m, n, k)
        noisy = rk.generate_input_blockquant(m, n, k, seed=m)
        assert_close_to_oracle(static_run(noisy), oracle_bf16(noisy), RTOL, ATOL, "static, row ranges %r" % ((m, n, k),))
    plans = tmp_path / "big.plans"
    plans.write_text("2048 2048 1024 1 4 8 0\n4096 4096 512 0 1 8 1\n")
    try:
        assert rfk.load_plans(str(plans)) == 2
        for (m, n, k) in ((2048, 2048, 1024), (4096, 4096, 512)):
            got = rfk.select_config(m, n, k)
            assert (got.split_k, got.stream_k) == ((4, 0) if k == 1024 else (1, 1))
            data = exact_problem(m, n, k, seed=k)
            assert np.array_equal(bf16_bits(static_run(data)), oracle_bf16(data)), (m, n, k)
            noisy = rk.generate_input_blockquant(m, n, k, seed=k + 1)
            assert_close_to_oracle(static_run(noisy), oracle_bf16(noisy), RTOL, ATOL, "static, fitted plan %r" % ((m, n, k),))
    finally:
        rfk.clear_plans()
    data = rk.generate_input_blockquant(256, 1536, 7168, 25)
    got, want = _both(rfk, data)
    assert np.array_equal(got, want)


def test_static_entry_writes_a_large_ragged_c_in_place(rfk):
    """Short K, a ragged N and 33.6 MB of C: the plan stages B and C, which do not fit the array; one launch, and not one per range of
    rows with its copies."""
    from helpers import exact_problem
    m, n, k = 4112, 4090, 256
    assert rfk.select_config(m, n, k).stream_k == 4
    data = exact_problem(m, n, k, seed=1)
    g, buf = to_gpu(data, canary_elems=4096)
    hip, graph, count = ctypes.CDLL("libamdhip64.so"), ctypes.c_void_p(), ctypes.c_size_t()
    stream = torch.cuda.Stream()
    with torch.cuda.stream(stream):
        handle = ctypes.c_void_p(stream.cuda_stream)
        assert hip.hipStreamBeginCapture(handle, 2) == 0                 # hipStreamCaptureModeRelaxed
        try:
            rfk.fp8_mm_static(*g)
        finally:
            assert hip.hipStreamEndCapture(handle, ctypes.byref(graph)) == 0
        assert hip.hipGraphGetNodes(graph, None, ctypes.byref(count)) == 0 and count.value == 1
        hip.hipGraphDestroy(graph)
    g[4].fill_(-3.0)
    rfk.fp8_mm_static(*g)
    torch.cuda.synchronize()
    assert np.array_equal(bf16_bits(g[4]), oracle_bf16(data))
    assert bool((buf[g[4].numel():].float() == -7.0).all()), "store past the end of C"


@pytest.mark.parametrize("n", [512, 500])
@pytest.mark.parametrize("piece", ["0 1 8 0", "28 2 8 0", "21 1 8 0", "29 1 8 0", "30 2 8 0"])
def test_static_entry_in_row_ranges_takes_every_kind_of_plan(rfk, tmp_path, n, piece):
    """A 36 MB staging copy of A, which a plan file's tile for the whole shape asks for: row ranges of 2512 and 2489 (padded to 2496)
    rows, each with the plan that the file has for it: tiles with and without K parts, few-rows kernels, any-alignment tiles (these
    were refused for a range with padded rows)."""
    from helpers import exact_problem
    m, k = 5001, 7168
    plans = tmp_path / "ranges.plans"
    plans.write_text("5008 512 7168 0 1 8 0\n2512 512 7168 %s\n2496 512 7168 %s\n" % (piece, piece))
    data = exact_problem(m, n, k, seed=n)
    g, buf = to_gpu(data, canary_elems=4096)
    g[4].fill_(-3.0)
    try:
        assert rfk.load_plans(str(plans)) == 3
        rfk.fp8_mm_static(*g)
        torch.cuda.synchronize()
    finally:
        rfk.clear_plans()
    assert np.array_equal(bf16_bits(g[4]), oracle_bf16(data))
    assert bool((buf[g[4].numel():].float() == -7.0).all()), "store past the end of C"


def _plan_bits(rfk, ops, m, n, cfg):
    """Bits of the first m rows of an aligned problem under an explicit plan."""
    a, b, sa, sb = ops
    c = torch.zeros((a.shape[0], n), dtype=torch.bfloat16, device="cuda")
    rfk.fp8_mm(a, b, sa, sb, c, config=rfk.GemmConfig(*cfg, 8, 0))
    torch.cuda.synchronize()
    return bf16_bits(c[:m])


def _static_bits_and_plans(rfk, m, n, k, plans):
    """rf_fp8_gemm_static on data whose sums round, so that the bits tell the number of K parts, and each plan's bits on the same
    problem with its rows padded to a multiple of 16."""
    gen = torch.Generator(device="cuda").manual_seed(m + n + k)
    mp, qk, fp8 = -(-m // 16) * 16, k // 128, torch.float8_e4m3fn
    a, sa = torch.randint(0, 120, (k, mp), dtype=torch.uint8, device="cuda", generator=gen), torch.rand((qk, mp), device="cuda", generator=gen)
    a ^= torch.randint(0, 2, (k, mp), dtype=torch.uint8, device="cuda", generator=gen) << 7
    b, sb = torch.randint(0, 120, (k, n), dtype=torch.uint8, device="cuda", generator=gen).view(fp8).T, torch.rand((qk, -(-n // 128)), device="cuda", generator=gen).T
    c = torch.full((m, n), -3.0, dtype=torch.bfloat16, device="cuda")
    rfk.fp8_mm_static(a[:, :m].contiguous().view(fp8).T, b, sa[:, :m].contiguous().T, sb, c)
    torch.cuda.synchronize()
    ops = (a.view(fp8).T, b, sa.T, sb)
    return bf16_bits(c), [_plan_bits(rfk, ops, m, n, p) for p in plans]


def test_static_entry_counts_the_rows_of_c_for_a_staged_k_split(rfk):
    """Sums that fit beside the staged A as the 659 rows that are written, but not as the 672 that are computed: the plan's four
    parts, which were cut to three."""
    m, n, k = 659, 2720, 6400
    cfg = rfk.select_config(m, n, k)
    assert cfg.split_k == 4 and cfg.stream_k == 0
    staged = k * 672 + k // 128 * 672 * 4
    assert staged + 4 * 4 * m * n <= rfk.lib().rf_gemm_static_scratch_bytes() < staged + 4 * 4 * 672 * n
    got, (four, three) = _static_bits_and_plans(rfk, m, n, k, [(cfg.variant, 4), (cfg.variant, 3)])
    assert not np.array_equal(four, three)
    assert np.array_equal(got, four)


# aligned and beyond the array by itself, A staged beside the sums; the plan before the rule for long K in one part and in two
@pytest.mark.parametrize("m,n,k,runs", [(1328, 1648, 7424, (10, 3)), (560, 3216, 7040, (11, 4)), (2092, 1104, 7168, (28, 1)),
                                        (2005, 816, 5888, (28, 2)), (1125, 1952, 7936, (8, 2)), (942, 1904, 6016, (8, 3))])
def test_static_entry_fits_a_long_k_plan_to_its_scratch_array(rfk, m, n, k, runs):
    """Plans of split_tile_plan whose sums do not fit: the one that runs is neither theirs nor theirs with fewer parts unless that
    is estimated fastest among those that fit. Data that round tell the K parts by their bits."""
    cfg, qk = rfk.select_config(m, n, k), k // 128
    staged = (k + 4 * qk) * -(-m // 16) * 16 if m % 16 else 0
    fit = (rfk.lib().rf_gemm_static_scratch_bytes() - staged) // (4 * m * n)
    assert cfg.split_k > fit and cfg.stream_k == 0 and runs[1] <= fit
    others = [(cfg.variant, p) for p in range(1, cfg.split_k + 1) if p != runs[1] and -(-qk // -(-qk // p)) == p]
    got, bits = _static_bits_and_plans(rfk, m, n, k, [runs] + others)
    assert np.array_equal(got, bits[0])
    assert not any(np.array_equal(got, x) for x in bits[1:])

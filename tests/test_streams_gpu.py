"""GPU tests of the launch path's temporary memory: launches on different streams of one device do not share buffers,
buffer growth never waits for the device, and plans that cannot run are skipped at lookup."""
import ctypes

import numpy as np
import pytest
import torch

from oracle import ref_kernel as rk
from helpers import bf16_bits, exact_problem, oracle_bf16, to_gpu

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def rfk():
    import radeonflow_kernels_amd as r
    assert torch.cuda.is_available(), "these tests need the GPU"
    r.lib()
    return r


def _alone(rfk, g):
    g[4].zero_()
    rfk.fp8_mm(*g)
    torch.cuda.synchronize()
    return bf16_bits(g[4]).copy()


def test_split_k_and_ragged_launches_on_three_streams_match_their_single_stream_results(rfk):
    """Two split-K GEMMs of the C1 shape and one ragged-M GEMM (staged through the pad buffer, split along K as well)
    run concurrently on three streams with different data, several launches deep. Each result equals, bit for bit,
    what the same call gives when it has the device to itself."""
    m, n, k = 1024, 1536, 7168
    assert rfk.select_config(m, n, k).split_k > 1, "this test wants a split-K plan for the C1 shape"
    problems = [to_gpu(rk.generate_input_blockquant(m, n, k, seed)) for seed in (101, 202)]
    problems.append(to_gpu(rk.generate_input_blockquant(1000, 1536, 7168, 303)))        # ragged M: staged copy
    alone = [_alone(rfk, g) for g in problems]
    assert not np.array_equal(alone[0], alone[1])
    streams = [torch.cuda.Stream() for _ in problems]
    for g in problems:
        g[4].zero_()
    torch.cuda.synchronize()
    for _ in range(6):                                   # deep queues, so the launches really overlap
        for g, s in zip(problems, streams):
            with torch.cuda.stream(s):
                rfk.fp8_mm(*g)
    torch.cuda.synchronize()
    for i, g in enumerate(problems):
        assert np.array_equal(bf16_bits(g[4]), alone[i]), "problem %d differs when run beside the others" % i


@pytest.mark.timeout(120)
def test_run_with_metrics_then_a_call_that_grows_the_buffers_does_not_wait_for_the_device(rfk):
    """run(metrics) leaves a timing callback pending on the stream; the next call needs a larger split-K workspace and
    a larger staging buffer. Neither may wait for the device while holding a lock the callback needs (the host would
    wait for the device, the device for the callback, the callback for the lock)."""
    from radeonflow_kernels_amd import gemm
    L = rfk.lib()
    L.rf_gemm_destroy()                                  # start from empty buffers
    s = torch.cuda.Stream()
    small = to_gpu(exact_problem(250, 256, 2048, 5))     # ragged, small buffers
    big = to_gpu(exact_problem(1000, 1536, 7168, 6))     # ragged, larger staging copy and split-K workspace
    exp_small, exp_big = oracle_bf16(exact_problem(250, 256, 2048, 5)), oracle_bf16(exact_problem(1000, 1536, 7168, 6))
    pms = [gemm.PerfMetrics() for _ in range(4)]
    ptr = ctypes.c_void_p(s.cuda_stream)
    with torch.cuda.stream(s):
        for i, g in enumerate((small, big, small, big)):
            a, b, sa, sb, c = g
            L.run(a.data_ptr(), b.data_ptr(), sa.data_ptr(), sb.data_ptr(), c.data_ptr(), a.shape[0], b.shape[0],
                  a.shape[1], ctypes.byref(pms[i]), ptr)     # no synchronisation between the calls
    s.synchronize()
    torch.cuda.synchronize()
    assert all(pm.entries[0].time > 0 for pm in pms)
    assert np.array_equal(bf16_bits(small[4]), exp_small)
    assert np.array_equal(bf16_bits(big[4]), exp_big)


def test_more_streams_than_buffer_sets(rfk):
    """Only launches that need temporary memory take a buffer set, and there are 32 sets per device. 40 streams (made
    with hipStreamCreate: torch hands out 32 distinct ones) run a one-kernel plan each (no set is used, nothing changes
    hands), then 32 of them run a split-K plan (all sets taken), then a 33rd does: the least recently used set changes
    hands without a host wait, and the results stay bit-exact. The same on a stream that is being captured into a graph
    is refused with RF_ERR_BAD_CONFIG, the capture stays valid, and rf_fp8_gemm_static records the same GEMM into it
    instead; the replayed graph gives the same bits."""
    hip = ctypes.CDLL("libamdhip64.so")
    L = rfk.lib()
    L.rf_gemm_destroy()
    direct = exact_problem(256, 256, 256, 31)
    exp_direct = oracle_bf16(direct)
    assert rfk.select_config(256, 256, 256).split_k == 1
    split = exact_problem(128, 512, 7168, 32)
    exp_split = oracle_bf16(split)
    assert rfk.select_config(128, 512, 7168).split_k > 1
    handles = []
    for _ in range(40):
        h = ctypes.c_void_p()
        assert hip.hipStreamCreate(ctypes.byref(h)) == 0
        handles.append(h)
    assert len({h.value for h in handles}) == 40

    def launch(fn, g, h):
        a, b, sa, sb, c = g
        return fn(a.data_ptr(), b.data_ptr(), sa.data_ptr(), sb.data_ptr(), c.data_ptr(), a.shape[0], b.shape[0],
                  a.shape[1], h)

    try:
        gd = [to_gpu(direct) for _ in handles]
        gs = [to_gpu(split) for _ in range(34)]
        torch.cuda.synchronize()
        for g, h in zip(gd, handles):
            assert launch(L.rf_fp8_gemm, g, h) == 0
        torch.cuda.synchronize()
        assert all(np.array_equal(bf16_bits(g[4]), exp_direct) for g in gd)
        for g, h in zip(gs[:33], handles[:33]):          # the 33rd takes over the first stream's set
            assert launch(L.rf_fp8_gemm, g, h) == 0
        gs[0][4].zero_()
        torch.cuda.synchronize()
        assert launch(L.rf_fp8_gemm, gs[0], handles[0]) == 0     # and the first stream takes over the second's
        torch.cuda.synchronize()
        assert all(np.array_equal(bf16_bits(g[4]), exp_split) for g in gs[:33])
        # a 34th stream that needs temporary memory, under capture: refused, and the capture goes on
        cap, g = handles[35], gs[33]
        graph, graph_exec = ctypes.c_void_p(), ctypes.c_void_p()
        assert hip.hipStreamBeginCapture(cap, 2) == 0            # hipStreamCaptureModeRelaxed
        rc = launch(L.rf_fp8_gemm, g, cap)
        msg = L.rf_gemm_last_error().decode()
        rc_static = launch(L.rf_fp8_gemm_static, g, cap)
        assert hip.hipStreamEndCapture(cap, ctypes.byref(graph)) == 0
        assert rc == 4 and "captured" in msg, (rc, msg)
        assert rc_static == 0
        assert hip.hipGraphInstantiate(ctypes.byref(graph_exec), graph, None, None, 0) == 0
        g[4].zero_()
        torch.cuda.synchronize()
        for _ in range(2):
            assert hip.hipGraphLaunch(graph_exec, cap) == 0
            assert hip.hipStreamSynchronize(cap) == 0
            assert np.array_equal(bf16_bits(g[4]), exp_split)
            g[4].zero_()
            torch.cuda.synchronize()
        hip.hipGraphExecDestroy(graph_exec)
        hip.hipGraphDestroy(graph)
    finally:
        torch.cuda.synchronize()
        L.rf_gemm_destroy()
        for h in handles:
            hip.hipStreamDestroy(h)


def test_stream_k_plan_for_a_shape_with_fewer_tiles_than_compute_units_is_skipped(rfk, tmp_path):
    """A stream-K plan splits each tile between at most two workgroups, which needs at least one tile per compute unit.
    A plan file that asks for it on a smaller shape is ignored for that shape; the result stays bit-exact."""
    sk = [v["variant"] for v in rfk.variants() if v["stream_k"]]
    assert sk, "no variant with a stream-K form"
    m, n, k = 512, 512, 1024                             # 4 tiles of 256 x 256
    before = rfk.select_config(m, n, k)
    path = tmp_path / "sk.plans"
    path.write_text("%d %d %d %d 1 1 1\n" % (m, n, k, sk[0]))
    try:
        assert rfk.load_plans(str(path)) == 1
        got = rfk.select_config(m, n, k)
        assert got.stream_k != 1
        assert (got.variant, got.split_k, got.stream_k) == (before.variant, before.split_k, before.stream_k)
        data = exact_problem(m, n, k, seed=9)
        g = to_gpu(data)
        rfk.fp8_mm(*g)
        rfk.fp8_mm(*g)                                   # a stale arrival counter would show on the second launch
        torch.cuda.synchronize()
        assert np.array_equal(bf16_bits(g[4]), oracle_bf16(data))
        ragged = exact_problem(m - 8, n, k, seed=10)     # the staged path picks its plan by the same rule
        g = to_gpu(ragged)
        rfk.fp8_mm(*g)
        torch.cuda.synchronize()
        assert np.array_equal(bf16_bits(g[4]), oracle_bf16(ragged))
    finally:
        rfk.clear_plans()


def test_small_grouped_problem_takes_the_variant_with_the_most_workgroups(rfk):
    """8 groups of 64 rows, N = 1024: no tile shape gives every compute unit a workgroup, so the automatic choice is
    the one with the most workgroups; its result equals the explicit 128 x 64 variant's bit for bit."""
    from oracle import cref
    rng = np.random.default_rng(4)
    groups, rows, n, k = 8, 64, 1024, 512
    m_total = groups * rows
    fp8 = torch.float8_e4m3fn
    vals = np.array([0, 1, 2, 3, -1, -2, -3], np.float32)
    a = torch.from_numpy(cref.f32_to_e4m3fn(rng.choice(vals, (k, m_total)))).view(fp8).cuda().T
    b = torch.from_numpy(cref.f32_to_e4m3fn(rng.choice(vals, (groups, k, n)))).view(fp8).cuda().transpose(1, 2)
    sa = torch.from_numpy(rng.choice(np.array([0.5, 1, 2], np.float32), (k // 128, m_total))).cuda().T
    sb = torch.from_numpy(rng.choice(np.array([0.5, 1, 2], np.float32), (groups, k // 128, n // 128))).cuda().transpose(1, 2)
    offs = [g * rows for g in range(groups + 1)]
    out = {}
    for variant in (-1, 3):
        c = torch.zeros((m_total, n), dtype=torch.bfloat16, device="cuda")
        rfk.fp8_mm_grouped(a, b, sa, sb, c, offs, variant=variant)
        torch.cuda.synchronize()
        out[variant] = bf16_bits(c)
    assert np.any(out[3] != 0) and np.array_equal(out[-1], out[3])


@pytest.mark.parametrize("rows,n,k", [((32,), 1536, 7168), ((1,), 200, 7168), ((40, 700, 300, 500), 4096, 4096)])
def test_a_captured_launch_is_one_kernel_and_replays_right(rfk, rows, n, k):
    """fp8_mm with a K split summed inside the launch (plans of an aligned and of a small ragged shape) and the grouped queue
    form use counters: captured on a stream that has never run anything, each is one graph node, and three replays with eager
    calls of the same stream between them give the eager result."""
    hip = ctypes.CDLL("libamdhip64.so")
    grouped = len(rows) > 1
    offs = [0] + [int(x) for x in np.cumsum(rows)]
    m = offs[-1]
    data = exact_problem(m, n, k, seed=m + n)
    g = to_gpu(data)
    exp = oracle_bf16(data)

    def launch():
        if grouped:                                      # every group with the same weights
            rfk.fp8_mm_grouped_padded(a_pad, b3, sa_pad, sb3, g[4], offs, variant=5)
        else:
            rfk.fp8_mm(*g)

    if grouped:
        pad = rfk.grouped_padded_offsets(offs)
        a_pad = torch.zeros((k, pad[-1]), dtype=torch.uint8, device="cuda")
        sa_pad = torch.ones((k // 128, pad[-1]), device="cuda")
        for i, r in enumerate(rows):
            a_pad[:, pad[i]:pad[i] + r] = g[0].T.view(torch.uint8)[:, offs[i]:offs[i + 1]]
            sa_pad[:, pad[i]:pad[i] + r] = g[2].T[:, offs[i]:offs[i + 1]]
        a_pad, sa_pad = a_pad.view(torch.float8_e4m3fn).T, sa_pad.T
        b3 = g[1].T.view(torch.uint8).repeat(len(rows), 1, 1).view(torch.float8_e4m3fn).transpose(1, 2)
        sb3 = g[3].T.repeat(len(rows), 1, 1).transpose(1, 2)
    elif n % 16 == 0:
        assert rfk.select_config(m, n, k).split_k > 1
    rfk.lib().rf_gemm_destroy()                          # the capture's stream is the first to use counters
    handle, graph, graph_exec = ctypes.c_void_p(), ctypes.c_void_p(), ctypes.c_void_p()
    assert hip.hipStreamCreate(ctypes.byref(handle)) == 0
    stream = torch.cuda.ExternalStream(handle.value)
    try:
        with torch.cuda.stream(stream):
            assert hip.hipStreamBeginCapture(handle, 2) == 0     # hipStreamCaptureModeRelaxed
            try:
                launch()
            finally:
                assert hip.hipStreamEndCapture(handle, ctypes.byref(graph)) == 0
            count = ctypes.c_size_t()
            assert hip.hipGraphGetNodes(graph, None, ctypes.byref(count)) == 0 and count.value == 1
            assert hip.hipGraphInstantiate(ctypes.byref(graph_exec), graph, None, None, 0) == 0
            for replay in range(3):
                g[4].fill_(-1.0)
                torch.cuda.synchronize()
                assert hip.hipGraphLaunch(graph_exec, handle) == 0
                torch.cuda.synchronize()
                assert np.array_equal(bf16_bits(g[4]), exp), "replay %d" % replay
                g[4].fill_(-1.0)
                launch()
                torch.cuda.synchronize()
                assert np.array_equal(bf16_bits(g[4]), exp), "eager call after replay %d" % replay
            hip.hipGraphExecDestroy(graph_exec)
            hip.hipGraphDestroy(graph)
    finally:
        torch.cuda.synchronize()
        rfk.lib().rf_gemm_destroy()
        hip.hipStreamDestroy(handle)


def test_small_few_rows_calls_under_capture_need_no_buffer_set(rfk):
    """All 32 buffer sets belong to other streams, and a stream under capture cannot take one over. Automatic few-rows plans
    with a K split give way to K in one part (small ragged shapes) or to the tiled plan (an aligned shape whose tiled plan
    needs no memory) and are recorded all the same; an explicit plan with a K split is refused."""
    hip = ctypes.CDLL("libamdhip64.so")
    L = rfk.lib()
    L.rf_gemm_destroy()
    handles = []
    for _ in range(33):
        h = ctypes.c_void_p()
        assert hip.hipStreamCreate(ctypes.byref(h)) == 0
        handles.append(h)

    def launch(g, h, cfg=None):
        a, b, sa, sb, c = g
        return L.rf_fp8_gemm_ex(a.data_ptr(), b.data_ptr(), sa.data_ptr(), sb.data_ptr(), c.data_ptr(), a.shape[0], b.shape[0],
                                a.shape[1], cfg, h)

    try:
        split = to_gpu(exact_problem(16, 1536, 7168, 1))
        assert rfk.select_config(16, 1536, 7168).split_k > 1
        for h in handles[:32]:
            assert launch(split, h) == 0
            torch.cuda.synchronize()
        for (m, n, k) in ((1, 200, 7168), (3, 130, 5120), (256, 1024, 2304)):
            assert L.rf_gemm_workspace_bytes(m, n, k) > 0
            data = exact_problem(m, n, k, m + n)
            g, exp = to_gpu(data), oracle_bf16(data)
            torch.cuda.synchronize()
            cap, graph, graph_exec = handles[32], ctypes.c_void_p(), ctypes.c_void_p()
            assert hip.hipStreamBeginCapture(cap, 2) == 0            # hipStreamCaptureModeRelaxed
            rc = launch(g, cap)
            rc_explicit = launch(g, cap, ctypes.byref(rfk.GemmConfig(14, 2, 8, 0)))
            assert hip.hipStreamEndCapture(cap, ctypes.byref(graph)) == 0
            assert rc == 0 and rc_explicit == 4, (m, n, k)
            assert hip.hipGraphInstantiate(ctypes.byref(graph_exec), graph, None, None, 0) == 0
            for _ in range(3):
                g[4].fill_(-1.0)
                torch.cuda.synchronize()
                assert hip.hipGraphLaunch(graph_exec, cap) == 0
                torch.cuda.synchronize()
                assert np.array_equal(bf16_bits(g[4]), exp), (m, n, k)
                assert launch(split, handles[0]) == 0                # eager work between the replays
                torch.cuda.synchronize()
            hip.hipGraphExecDestroy(graph_exec)
            hip.hipGraphDestroy(graph)
    finally:
        torch.cuda.synchronize()
        L.rf_gemm_destroy()
        for h in handles:
            hip.hipStreamDestroy(h)


def test_staged_calls_under_capture_without_a_buffer_set_take_tiles_that_need_none(rfk):
    """All 32 buffer sets belong to other streams, and a stream under capture cannot take one over. Ragged shapes whose plan runs on
    staged copies (the skinny-K schedule, 256 x 256 tiles) are recorded all the same, on tiles that take operands as they are."""
    hip = ctypes.CDLL("libamdhip64.so")
    L = rfk.lib()
    L.rf_gemm_destroy()
    handles = []
    for _ in range(33):
        h = ctypes.c_void_p()
        assert hip.hipStreamCreate(ctypes.byref(h)) == 0
        handles.append(h)

    def launch(g, h):
        a, b, sa, sb, c = g
        return L.rf_fp8_gemm(a.data_ptr(), b.data_ptr(), sa.data_ptr(), sb.data_ptr(), c.data_ptr(), a.shape[0], b.shape[0], a.shape[1], h)

    try:
        split = to_gpu(exact_problem(16, 1536, 7168, 1))
        for h in handles[:32]:
            assert launch(split, h) == 0
            torch.cuda.synchronize()
        for (m, n, k), schedule in (((2608, 4090, 128), 4), ((3056, 5003, 256), 0)):
            plan = rfk.select_config(m, n, k)
            assert (plan.variant, plan.stream_k) == (0, schedule)
            data = exact_problem(m, n, k, m + n)
            g, exp = to_gpu(data), oracle_bf16(data)
            torch.cuda.synchronize()
            cap, graph, graph_exec = handles[32], ctypes.c_void_p(), ctypes.c_void_p()
            assert hip.hipStreamBeginCapture(cap, 2) == 0            # hipStreamCaptureModeRelaxed
            rc = launch(g, cap)
            assert hip.hipStreamEndCapture(cap, ctypes.byref(graph)) == 0
            assert rc == 0, (m, n, k, L.rf_gemm_last_error())
            assert hip.hipGraphInstantiate(ctypes.byref(graph_exec), graph, None, None, 0) == 0
            for _ in range(3):
                g[4].fill_(-1.0)
                torch.cuda.synchronize()
                assert hip.hipGraphLaunch(graph_exec, cap) == 0
                torch.cuda.synchronize()
                assert np.array_equal(bf16_bits(g[4]), exp), (m, n, k)
                assert launch(split, handles[0]) == 0                # eager work between the replays
                torch.cuda.synchronize()
            hip.hipGraphExecDestroy(graph_exec)
            hip.hipGraphDestroy(graph)
    finally:
        torch.cuda.synchronize()
        L.rf_gemm_destroy()
        for h in handles:
            hip.hipStreamDestroy(h)


@pytest.mark.parametrize("m,n,k", [(1, 200, 7168), (7, 1536, 7168), (100, 72, 256), (1024, 1536, 7168), (1000, 1536, 7168)])
def test_workspace_bytes_covers_the_plan_that_runs(rfk, m, n, k):
    """rf_gemm_init with rf_gemm_workspace_bytes: for a tabled, a padded and a small ragged shape the figure is that of a K
    split's partial sums under the plan the call takes (reported as variant -1 for the small ones: few-rows kernels)."""
    got = rfk.lib().rf_gemm_workspace_bytes(m, n, k)
    plan = rfk.select_config(m, n, k)
    qk = k // 128

    def bytes_of(v, split):
        parts = -(-qk // -(-qk // split))
        if parts == 1:
            return 0
        if v["variant"] >= 14:
            return -(-m // v["block_m"]) * v["block_m"] * -(-n // v["block_n"]) * v["block_n"] * 4 * parts
        return -(-m // 16) * 16 * -(-n // 16) * 16 * 4 * parts

    if plan.variant >= 0:
        assert got == bytes_of(rfk.variants()[plan.variant], plan.split_k)
    else:
        assert got in {bytes_of(v, split) for v in rfk.variants() if v["variant"] >= 14 for split in range(1, qk + 1)}
        assert (got > 0) == (k > 1024)                     # 56 K blocks in few tiles are split, two are not


def test_automatic_grouped_calls_under_capture_without_a_buffer_set_take_a_form_without_queues(rfk):
    """All 32 buffer sets belong to other streams: a grouped call whose automatic choice is the queue form is recorded on a 33rd
    stream all the same (in the padded layout, which needs no staging), with the queue form's bits; the explicit queue form is
    refused."""
    hip = ctypes.CDLL("libamdhip64.so")
    L = rfk.lib()
    L.rf_gemm_destroy()
    rows = [16 * int(x) for x in np.random.default_rng(5).integers(1, 25, 16)]
    offs = [0] + [int(x) for x in np.cumsum(rows)]
    m, n, k = offs[-1], 4096, 4096
    num_cu = torch.cuda.get_device_properties(0).multi_processor_count
    assert rfk.grouped_variant_for(offs, n, k, num_cu) == 5
    gen = torch.Generator(device="cuda").manual_seed(1)
    fp8 = torch.float8_e4m3fn
    a = torch.randint(0, 120, (k, m), dtype=torch.uint8, device="cuda", generator=gen).view(fp8).T
    b = torch.randint(0, 120, (len(rows), k, n), dtype=torch.uint8, device="cuda", generator=gen).view(fp8).transpose(1, 2)
    sa = (torch.rand((k // 128, m), device="cuda", generator=gen) * 1e-2).T
    sb = (torch.rand((len(rows), k // 128, n // 128), device="cuda", generator=gen) * 1e-2).transpose(1, 2)
    c = torch.zeros((m, n), dtype=torch.bfloat16, device="cuda")
    rfk.fp8_mm_grouped_padded(a, b, sa, sb, c, offs, variant=5)
    torch.cuda.synchronize()
    exp = bf16_bits(c).copy()
    L.rf_gemm_destroy()
    split = to_gpu(exact_problem(16, 1536, 7168, 1))
    handles = []
    for _ in range(33):
        h = ctypes.c_void_p()
        assert hip.hipStreamCreate(ctypes.byref(h)) == 0
        handles.append(h)
    graph, graph_exec, cap = ctypes.c_void_p(), ctypes.c_void_p(), handles[32]
    try:
        for h in handles[:32]:
            with torch.cuda.stream(torch.cuda.ExternalStream(h.value)):
                rfk.fp8_mm(*split)
            torch.cuda.synchronize()
        c.fill_(-1.0)
        torch.cuda.synchronize()
        with torch.cuda.stream(torch.cuda.ExternalStream(cap.value)):
            assert hip.hipStreamBeginCapture(cap, 2) == 0                # hipStreamCaptureModeRelaxed
            try:
                rfk.fp8_mm_grouped_padded(a, b, sa, sb, c, offs)
                with pytest.raises(RuntimeError, match="captured"):
                    rfk.fp8_mm_grouped_padded(a, b, sa, sb, c, offs, variant=5)
            finally:
                assert hip.hipStreamEndCapture(cap, ctypes.byref(graph)) == 0
        assert hip.hipGraphInstantiate(ctypes.byref(graph_exec), graph, None, None, 0) == 0
        for replay in range(3):
            c.fill_(-1.0)
            torch.cuda.synchronize()
            assert hip.hipGraphLaunch(graph_exec, cap) == 0
            torch.cuda.synchronize()
            assert np.array_equal(bf16_bits(c), exp), replay
            rfk.fp8_mm(*split)
            torch.cuda.synchronize()
        hip.hipGraphExecDestroy(graph_exec)
        hip.hipGraphDestroy(graph)
    finally:
        torch.cuda.synchronize()
        L.rf_gemm_destroy()
        for h in handles:
            hip.hipStreamDestroy(h)


@pytest.mark.parametrize("m,runs", [(1232, (28, 1)), (1228, (29, 1))])
def test_long_k_plans_under_capture_without_a_buffer_set_take_one_k_part(rfk, m, runs):
    """All 32 buffer sets belong to other streams, and a stream under capture cannot take one over: a shape that split_tile_plan moves
    to four K parts is recorded as one kernel of one K part, on the plan without that rule or, with A to be staged, on the tiles that
    take operands as they are. Data that round tell which plan ran."""
    hip = ctypes.CDLL("libamdhip64.so")
    L = rfk.lib()
    L.rf_gemm_destroy()
    n, k = 1616, 7552
    assert rfk.select_config(m, n, k).split_k == 4
    gen, fp8 = torch.Generator(device="cuda").manual_seed(m), torch.float8_e4m3fn
    a, b = (torch.randint(0, 120, (k, x), dtype=torch.uint8, device="cuda", generator=gen).view(fp8).T for x in (m, n))
    sa, sb = (torch.rand((k // 128, x), device="cuda", generator=gen).T for x in (m, -(-n // 128)))
    c = torch.zeros((m, n), dtype=torch.bfloat16, device="cuda")

    def bits(config=None):
        c.fill_(-1.0)
        rfk.fp8_mm(a, b, sa, sb, c, config=config)
        torch.cuda.synchronize()
        return bf16_bits(c).copy()

    exp = bits(rfk.GemmConfig(*runs, 8, 0))
    split = to_gpu(exact_problem(16, 1536, 7168, 1))
    handles = []
    for _ in range(33):
        h = ctypes.c_void_p()
        assert hip.hipStreamCreate(ctypes.byref(h)) == 0
        handles.append(h)
    graph, graph_exec, count, cap = ctypes.c_void_p(), ctypes.c_void_p(), ctypes.c_size_t(), handles[32]
    try:
        L.rf_gemm_destroy()
        for h in handles[:32]:
            with torch.cuda.stream(torch.cuda.ExternalStream(h.value)):
                rfk.fp8_mm(*split)
            torch.cuda.synchronize()
        with torch.cuda.stream(torch.cuda.ExternalStream(cap.value)):
            assert hip.hipStreamBeginCapture(cap, 2) == 0                # hipStreamCaptureModeRelaxed
            try:
                rfk.fp8_mm(a, b, sa, sb, c)
            finally:
                assert hip.hipStreamEndCapture(cap, ctypes.byref(graph)) == 0
        assert hip.hipGraphGetNodes(graph, None, ctypes.byref(count)) == 0 and count.value == 1
        assert hip.hipGraphInstantiate(ctypes.byref(graph_exec), graph, None, None, 0) == 0
        for replay in range(3):
            c.fill_(-1.0)
            torch.cuda.synchronize()
            assert hip.hipGraphLaunch(graph_exec, cap) == 0
            torch.cuda.synchronize()
            assert np.array_equal(bf16_bits(c), exp), replay
            with torch.cuda.stream(torch.cuda.ExternalStream(handles[0].value)):
                rfk.fp8_mm(*split)                                       # eager work between the replays
            torch.cuda.synchronize()
        hip.hipGraphExecDestroy(graph_exec)
        hip.hipGraphDestroy(graph)
        assert not np.array_equal(bits(), exp), "with a buffer set the plan has four K parts"
    finally:
        torch.cuda.synchronize()
        L.rf_gemm_destroy()
        for h in handles:
            hip.hipStreamDestroy(h)

// Tile kernels for operands at any alignment: rows of A of M bytes and rows of B of N bytes, whatever M and N are.
#pragma once
#include "fp8_gemm_fewrows.h"

namespace rf {

template <int BM_, int BN_, int WAVES_M_, int WAVES_N_>
struct AnyGeom {
    static constexpr int BM = BM_, BN = BN_, NW = WAVES_M_ * WAVES_N_, NT = NW * 64;
    static constexpr int CPR_A = BM / 16, CPR_B = BN / 16;
    static constexpr int IA = BK * CPR_A / NT, IB = BK * CPR_B / NT;      // 16-byte loads per thread and K block
    static constexpr int LDS_BYTES = TileGeom<BM_, BN_, WAVES_M_, WAVES_N_, 2>::LDS_BYTES;
    static_assert(BK * CPR_A % NT == 0 && BK * CPR_B % NT == 0, "whole loads per thread");
};

// tile_mainloop with the operands through registers: 16-byte loads at any byte into one of two register sets, from there into the stage
// that the next K block reads. Bound by the latency of the loads and by LDS, which every byte is written to and read from by all waves:
// a K block of a 128 x 128 tile takes 0.58 us, of a 128 x 256 tile 0.79, rows that start at any byte up to 0.4 us more. No copy of A or B
// and none of C: 200 x 5003 x 2048 19.5 -> 14.3 us (few-rows kernels), 4096 x 1000 x 1024 19.8 -> 11.1 (128 x 128 tiles on a copy of B).
template <int BM, int BN, int WAVES_M, int WAVES_N>
__device__ __forceinline__ void tile_mainloop_any(
    const uint8_t *__restrict__ A, const uint8_t *__restrict__ B, const float *__restrict__ SA,
    const float *__restrict__ SB, int M, int ldm, int N, int QK, int m0, int n0, int kb_begin, int kb_end, uint8_t *lds,
    f32x4 (&acc)[BM / WAVES_M / 16][BN / WAVES_N / 16]) {
    using G = TileGeom<BM, BN, WAVES_M, WAVES_N, 2>;
    using Y = AnyGeom<BM, BN, WAVES_M, WAVES_N>;
    constexpr int WM = G::WM, WN = G::WN, TM = G::TM, TN = G::TN, NT = G::NT, IA = Y::IA, IB = Y::IB;
    constexpr int STAGE_A = G::STAGE_A, STAGE_B = G::STAGE_B, STAGE_S = G::STAGE_S;
    constexpr int OFF_B = 2 * STAGE_A, OFF_S = 2 * (STAGE_A + STAGE_B), OFF_SB = BM * 4;
    static_assert(WN <= 128 && 128 % WN == 0, "a wave's columns have one b_scale");
    static_assert((TM & (TM - 1)) == 0 && (TN & (TN - 1)) == 0, "a fragment's address is the wave's first one with the tile's index XORed in");
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int L = lane & 15, g = lane >> 4, wm = wave % WAVES_M, wn = wave / WAVES_M;
    const int QN = (N + 127) / 128;

    // ---- loads: load i of a thread is the 16-byte chunk tid % CPR of K row i * NT / CPR + tid / CPR, at any byte ----
    static_assert(NT % Y::CPR_A == 0 && NT % Y::CPR_B == 0, "a thread keeps its chunk");
    const int chunk_a = tid % Y::CPR_A, row_a = tid / Y::CPR_A, chunk_b = tid % Y::CPR_B, row_b = tid / Y::CPR_B;
    constexpr int STEP_A = NT / Y::CPR_A, STEP_B = NT / Y::CPR_B;         // K rows between two loads
    // (a chunk past M or N: the row's first, any bytes will do)
    const uint32_t off_a0 = (uint32_t)row_a * (uint32_t)ldm + (uint32_t)(m0 + 16 * chunk_a < M ? m0 + 16 * chunk_a : m0),
                   off_b0 = (uint32_t)row_b * (uint32_t)N + (uint32_t)(n0 + 16 * chunk_b < N ? n0 + 16 * chunk_b : n0);
    auto off_a = [&](int i) { return off_a0 + (uint32_t)(i * STEP_A) * (uint32_t)ldm; };
    auto off_b = [&](int i) { return off_b0 + (uint32_t)(i * STEP_B) * (uint32_t)N; };
    auto dst_a = [&](int i) {
        const int row = row_a + i * STEP_A;
        return (uint32_t)(row * BM + ((chunk_a ^ swizzle_of_row<BM>(row)) << 4));
    };
    auto dst_b = [&](int i) {
        const int row = row_b + i * STEP_B;
        return (uint32_t)(OFF_B + row * BN + ((chunk_b ^ swizzle_of_row<BN>(row)) << 4));
    };
    // scales: threads 0 .. BM - 1 the rows of the tile, the next four its column blocks, the others repeat the last one
    static_assert(NT >= BM + 4, "a thread per scale");
    const float *src_s;
    uint32_t dst_s, step_s;
    if (tid < BM) {
        const int r = tid % WM;
        int m = m0 + (tid / WM) * WM + 16 * (r % TM) + r / TM;
        if (m > M - 1) m = M - 1;
        src_s = SA + m;
        step_s = (uint32_t)ldm;
        dst_s = OFF_S + tid * 4;
    } else {
        const int l = tid - BM < 3 ? tid - BM : 3;
        int nbq = (n0 >> 7) + l;
        if (nbq > QN - 1) nbq = QN - 1;
        src_s = SB + nbq;
        step_s = (uint32_t)QN;
        dst_s = OFF_S + OFF_SB + l * 4;
    }
    // bytes from a K block's first row to the end of the matrix (below 2^32 always suffices)
    auto rest = [&](int kb, int ld) {
        const unsigned long long r = (unsigned long long)(QK - kb) * BK * (unsigned)ld;
        return r < 0xffffffffull ? (uint32_t)r : 0xffffffffu;
    };
    u32x4_lds raw[2][IA + IB];                                           // two K blocks on their way
    float rs[2];
    const int kb_last = kb_end - 1;
    auto clamp_kb = [&](int kb) { return kb < kb_last ? kb : kb_last; };
    auto load_item = [&](auto set_c, int d, int kb) {
        constexpr int set = decltype(set_c)::value;
        kb = clamp_kb(kb);
        if (d < IA) raw[set][d] = load16<true>(A + (size_t)kb * BK * ldm, off_a(d), rest(kb, ldm));
        else if (d < IA + IB) raw[set][d] = load16<true>(B + (size_t)kb * BK * N, off_b(d - IA), rest(kb, N));
        else rs[set] = src_s[(size_t)kb * step_s];
    };
    auto write_item = [&](auto set_c, int d, int stage) {
        constexpr int set = decltype(set_c)::value;
        if (d < IA) *(u32x4_lds *)(lds + stage * STAGE_A + dst_a(d)) = raw[set][d];
        else if (d < IA + IB) *(u32x4_lds *)(lds + stage * STAGE_B + dst_b(d - IA)) = raw[set][d];
        else *(float *)(lds + stage * STAGE_S + dst_s) = rs[set];
    };
    // the matrix's last K block: bytes of cut loads back to their places
    auto uncut = [&](auto set_c, int kb) {
        constexpr int set = decltype(set_c)::value;
        if (kb != QK - 1) return;
#pragma unroll
        for (int d = 0; d < IA; d++) raw[set][d] = shift_back(raw[set][d], off_a(d), rest(kb, ldm));
#pragma unroll
        for (int d = 0; d < IB; d++) raw[set][IA + d] = shift_back(raw[set][IA + d], off_b(d), rest(kb, N));
    };
    constexpr int NL = IA + IB + 1;

    // ---- LDS -> MFMA operands (see tile_mainloop) ----
    const int krow = 32 * g + (L >> 1);
    const uint32_t aoff_base = krow * BM + (((wm * TM) ^ swizzle_of_row<BM>(krow)) << 4) + 8 * (L & 1);
    const uint32_t boff_base = OFF_B + krow * BN + (((wn * TN) ^ swizzle_of_row<BN>(krow)) << 4) + 8 * (L & 1);
    const uint32_t soff = OFF_S + (wm * WM + L * TM) * 4;
    const int ncol0 = n0 + wn * WN;
    const uint32_t sboff = OFF_S + OFF_SB + (((ncol0 >> 7) - (n0 >> 7)) << 2);
    constexpr int NMFMA = TM * TN, PR = (NMFMA % 4 == 0 && TN > 3) ? 4 : 3, LAG = PR - 1, BAR_SLOT = (TM - 1) * TN;
    static_assert(NMFMA % PR == 0 && LAG < TN && LAG < PR && TM % 2 == 0, "same schedule as tile_mainloop");
    constexpr int PER_SLOT = (NL + BAR_SLOT - 2) / (BAR_SLOT - 1);       // writes (and loads) per slot, done a slot before the barrier
#pragma unroll
    for (int j = 0; j < TM; j++)
#pragma unroll
        for (int i = 0; i < TN; i++) acc[j][i] = (f32x4){0.f, 0.f, 0.f, 0.f};
    i32x8 bfrag[TN], afrag[2];
    f32x4 pring[PR];
    float s[TM], sraw[TM], sb_raw = 0.f;
#pragma unroll
    for (int r = 0; r < PR; r++) pring[r] = (f32x4){0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int j = 0; j < TM; j++) s[j] = 0.f;
    auto rd = [&](uint32_t stage_base, uint32_t off) {
        return __builtin_amdgcn_ds_read_tr8_b64_v2i32((RF_LDS i32x2 *)(lds + stage_base + off));
    };
    auto read_bfrag = [&](int i, int stage) {
#pragma unroll
        for (int t = 0; t < 4; t++) {
            i32x2 v = rd(stage * STAGE_B, (boff_base ^ (i << 4)) + t * 8 * BN);
            bfrag[i][2 * t] = v[0];
            bfrag[i][2 * t + 1] = v[1];
        }
    };
    auto read_afrag = [&](int buf, int j, int stage) {
#pragma unroll
        for (int t = 0; t < 4; t++) {
            i32x2 v = rd(stage * STAGE_A, (aoff_base ^ (j << 4)) + t * 8 * BM);
            afrag[buf][2 * t] = v[0];
            afrag[buf][2 * t + 1] = v[1];
        }
    };
    auto read_scales = [&](int stage) {
#pragma unroll
        for (int q = 0; q < TM / 2; q++) {
            f32x2 v = *(RF_LDS f32x2 *)(lds + stage * STAGE_S + soff + q * 8);
            sraw[2 * q] = v[0];
            sraw[2 * q + 1] = v[1];
        }
        sb_raw = *(RF_LDS float *)(lds + stage * STAGE_S + sboff);
    };
    // prologue
#pragma unroll
    for (int d = 0; d < NL; d++) load_item(IntTag<0>{}, d, kb_begin);
#pragma unroll
    for (int d = 0; d < NL; d++) load_item(IntTag<1>{}, d, kb_begin + 1);
    __builtin_amdgcn_sched_barrier(0);
    uncut(IntTag<0>{}, kb_begin);
#pragma unroll
    for (int d = 0; d < NL; d++) write_item(IntTag<0>{}, d, 0);
#pragma unroll
    for (int d = 0; d < NL; d++) load_item(IntTag<0>{}, d, kb_begin + 2);
    __builtin_amdgcn_sched_barrier(0);
    __syncthreads();
    read_bfrag(0, 0);
    read_afrag(0, 0, 0);
    read_scales(0);
#pragma unroll
    for (int i = 1; i < TN; i++) read_bfrag(i, 0);
    // One K block: the stage it reads (cur), the register set of the next one (set). In its first slots block kb + 1 goes from
    // its registers into the other stage, and block kb + 3 is asked for in its place.
    auto k_block = [&](auto cur_c, auto set_c, int kb) {
        constexpr int cur = decltype(cur_c)::value, nxt = 1 - cur;
        const float s_last = s[TM - 1];
        uncut(set_c, clamp_kb(kb + 1));
#pragma unroll
        for (int j = 0; j < TM; j++) s[j] = sraw[j] * sb_raw;
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int t = 0; t < NMFMA; t++) {
            const int j = t / TN, i = t % TN;
            if (t == BAR_SLOT) {
                __syncthreads();
                __builtin_amdgcn_sched_barrier(0);
            }
            pring[t % PR] = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(
                bfrag[i], afrag[j & 1], (f32x4){0.f, 0.f, 0.f, 0.f}, 0, 0, 0, 0, 0, 0);
            asm volatile("" : "+v"(pring[t % PR]));
            __builtin_amdgcn_sched_barrier(0);
            if (j + 1 < TM) {
                if (i == 0) read_afrag((j + 1) & 1, j + 1, cur);
            } else {
                read_bfrag(i, nxt);
                if (i == 0) {
                    read_afrag(0, 0, nxt);
                    read_scales(nxt);
                }
            }
#pragma unroll
            for (int d = t * PER_SLOT; d < (t + 1) * PER_SLOT && d < NL; d++) write_item(set_c, d, nxt);
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int d = t * PER_SLOT; d < (t + 1) * PER_SLOT && d < NL; d++) load_item(set_c, d, kb + 3);
            if (t >= LAG) {
                const int u = t - LAG, ju = u / TN, iu = u % TN;
#pragma unroll
                for (int e = 0; e < 4; e++)
                    acc[ju][iu][e] = __builtin_fmaf(s[ju], pring[u % PR][e], acc[ju][iu][e]);
                asm volatile("" : "+v"(acc[ju][iu]));
            } else {
                const int u = NMFMA + t - LAG, ju = u / TN, iu = u % TN;
#pragma unroll
                for (int e = 0; e < 4; e++)
                    acc[ju][iu][e] = __builtin_fmaf(s_last, pring[u % PR][e], acc[ju][iu][e]);
                asm volatile("" : "+v"(acc[ju][iu]));
            }
            __builtin_amdgcn_sched_barrier(0);
        }
    };
    int kb = kb_begin;
    for (; kb + 1 < kb_end; kb += 2) {
        k_block(IntTag<0>{}, IntTag<1>{}, kb);
        k_block(IntTag<1>{}, IntTag<0>{}, kb + 1);
    }
    if (kb < kb_end) k_block(IntTag<0>{}, IntTag<1>{}, kb);
#pragma unroll
    for (int t = 0; t < LAG; t++) {
        const int u = NMFMA + t - LAG, ju = u / TN, iu = u % TN;
#pragma unroll
        for (int e = 0; e < 4; e++) acc[ju][iu][e] = __builtin_fmaf(s[TM - 1], pring[u % PR][e], acc[ju][iu][e]);
    }
}

// PARTIAL: the fp32 sums of K part blockIdx.y to ws[part][M rounded up to 16][ld_ws] (see reduce_splitk_any_c).
template <int BM, int BN, int WAVES_M, int WAVES_N, bool PARTIAL>
__global__ __launch_bounds__(WAVES_M *WAVES_N * 64) void gemm_fp8_blockscale_tile_any(
    const uint8_t *__restrict__ A, const uint8_t *__restrict__ B, const float *__restrict__ SA,
    const float *__restrict__ SB, void *__restrict__ out, int M, int ldm, int N, int K, int kb_per_split, int tiles_m, int tiles_n,
    int group_m) {
    using G = TileGeom<BM, BN, WAVES_M, WAVES_N, 2>;
    extern __shared__ __attribute__((aligned(1024))) uint8_t lds[];
    int tile_m, tile_n;
    tile_of_block(blockIdx.x, tiles_m * tiles_n, tiles_m, tiles_n, group_m, true, tile_m, tile_n);
    const int m0 = tile_m * BM, n0 = tile_n * BN, QK = K / BK;
    const int kb_begin = blockIdx.y * kb_per_split, kb_end = kb_begin + kb_per_split < QK ? kb_begin + kb_per_split : QK;
    f32x4 acc[G::TM][G::TN];
    tile_mainloop_any<BM, BN, WAVES_M, WAVES_N>(A, B, SA, SB, M, ldm, N, QK, m0, n0, kb_begin, kb_end, lds, acc);
    if constexpr (PARTIAL) {
        const int mp = (M + 15) / 16 * 16, ld_ws = (N + 15) / 16 * 16;
        store_tile_f32_staged<BM, BN, WAVES_M, WAVES_N>(acc, (float *)out + ((size_t)blockIdx.y * mp + m0) * ld_ws + n0, ld_ws, mp - m0,
                                                        ld_ws - n0, lds);
    } else {
        store_tile_bf16<BM, BN, WAVES_M, WAVES_N, default_store_passes<BM, WAVES_M>(), true, true>(acc, (uint16_t *)out, M, N, m0, n0, lds);
    }
}

// Sum of K parts in order, one bf16 rounding, into a C of any width and alignment: ws holds [part][rows_ws][ld] sums (ld a
// multiple of 8), C is the first `rows` x n of them. A thread sums eight columns of a row.
__global__ __launch_bounds__(256) void reduce_splitk_any_c(const float *__restrict__ ws, int ld, size_t part_stride, int splits, int n,
                                                           int rows, uint16_t *__restrict__ C) {
    const int pieces = (n + 7) / 8;
    const int per_block = pieces < 256 ? 256 / pieces : 1;
    const int trow = pieces < 256 ? (int)threadIdx.x / pieces : 0;
    const int piece = pieces < 256 ? (int)threadIdx.x - trow * pieces : (int)(blockIdx.y * 256 + threadIdx.x);
    const int r = (int)blockIdx.x * per_block + trow, col = piece * 8;
    if (trow >= per_block || piece >= pieces || r >= rows) return;
    const float *p = ws + (size_t)r * ld + col;
    f32x4 s0 = *(const f32x4 *)p, s1 = *(const f32x4 *)(p + 4);
    constexpr int BATCH = 4;
    for (int q0 = 1; q0 < splits; q0 += BATCH) {
        f32x4 v[BATCH][2];
#pragma unroll
        for (int q = 0; q < BATCH; q++)
            if (q0 + q < splits) {
                v[q][0] = *(const f32x4 *)(p + (size_t)(q0 + q) * part_stride);
                v[q][1] = *(const f32x4 *)(p + (size_t)(q0 + q) * part_stride + 4);
            }
#pragma unroll
        for (int q = 0; q < BATCH; q++)
            if (q0 + q < splits)
#pragma unroll
                for (int e = 0; e < 4; e++) {
                    s0[e] += v[q][0][e];
                    s1[e] += v[q][1][e];
                }
    }
    const u32x4_lds w = {pack_bf16x2(s0[0], s0[1]), pack_bf16x2(s0[2], s0[3]), pack_bf16x2(s1[0], s1[1]), pack_bf16x2(s1[2], s1[3])};
    uint16_t *out = C + (size_t)r * n + col;
    if (col + 8 <= n) {
        *(u32x4_any *)out = w;
    } else {
#pragma unroll
        for (int e = 0; e < 7; e++)
            if (col + e < n) out[e] = (uint16_t)(w[e / 2] >> (16 * (e % 2)));
    }
}

}  // namespace rf

// Few-rows form of the block-scaled fp8 GEMM: M up to a few dozen rows, any M and N, operands at any alignment.
//
// A decode step multiplies a handful of rows by a whole weight matrix: the launch is the streaming of B (N * K bytes), and
// at 5 to 130 KB of it per compute unit what counts is how soon all of it has been asked for and how little follows.
//   * a workgroup owns a strip of 32 to 128 columns and the K range of its split; its waves take K blocks in turn, so K is
//     split between the waves as well: each wave streams its own K blocks with no barrier, and one exchange through LDS at
//     the end adds the waves' sums in wave order;
//   * loads go to registers (16 bytes a lane; a wave asks for up to DEPTH K blocks, 6 to 20 KB each, before it uses the
//     first), then through a private LDS region of the wave, from which the transpose reads take MFMA fragments. Loads
//     into registers may start at any byte, which LDS-DMA may not: a row of A is M bytes ([K][M]) and is fetched as
//     16-byte pieces whatever M is; pieces that reach past M bring bytes of the next K row, whose results belong to rows
//     of C that do not exist and are not stored. So nothing is staged or padded for any M or N;
//   * pieces of the matrix's last K rows could reach past its end: every load's offset is cut to the last 16 bytes of the
//     matrix, and in its last K block the bytes are shifted back into place;
//   * SPLIT: the workgroups of a strip hand their sums over in memory, and the one that arrives last adds them in split
//     order and writes C. Nobody waits. With 2 to 16 KB per workgroup this chain (write-through store, counter, read
//     back) is a microsecond shorter than a second kernel and spares its launch (32 x 1536 x 7168: 8.7 -> 7.6 us), unlike
//     for the 98 KB tiles of the tiled kernels.
// Measured with operand sets that rotate out of L2, M x N x K, best tiled plan (with its staging, where M or N is ragged) ->
// here: 1 x 7168 x 2048 11.5 -> 6.2 us, 16 x 7168 x 2048 9.2 -> 6.2, 7 x 3072 x 1536 10.1 -> 3.7, 1 x 1536 x 7168 12.4 -> 6.9,
// 32 x 1536 x 7168 8.7 -> 7.5, 16 x 4608 x 7168 11.2 -> 10.1 (33 MB of weights: 5.1 TB/s beyond the 3.5 us of launch and
// hand-over), 64 x 5003 x 2048 23.4 -> 8.2. What is left is launch, one or two trips to memory and the hand-over.
// Numerics are those of the tiled kernels: per K block the products are summed inside the MFMA from zero and folded with
// acc = fma(a_scale * b_scale, partial, acc); a wave's K blocks in order, then the waves in order, then the splits in
// order, one bf16 rounding.
#pragma once
#include "fp8_gemm_kernels.h"

namespace rf {

typedef uint32_t u32x4_any __attribute__((ext_vector_type(4), aligned(1), may_alias));
typedef uint32_t u32x4_lds __attribute__((ext_vector_type(4), may_alias));

// TM 16-row tiles of A (and of C) per workgroup, TN 16-column tiles, NW waves, DEPTH K blocks asked for at a time.
template <int TM_, int TN_, int NW_, int DEPTH_>
struct FewRowsGeom {
    static constexpr int TM = TM_, TN = TN_, NW = NW_, DEPTH = DEPTH_;
    static constexpr int BM = 16 * TM, BN = 16 * TN;
    static constexpr int REGION = BK * (BM + BN);                     // one K block of A and of B, private to a wave
    static constexpr int EXCHANGE = NW * TM * TN * 1024;              // the waves' sums, over the regions
    static constexpr int LDS_BYTES = NW * REGION > EXCHANGE ? NW * REGION : EXCHANGE;
    // waves per SIMD: two workgroups per CU, where LDS has room
    static constexpr int WAVES_PER_SIMD = (LDS_BYTES < 80 * 1024 ? 2 : 1) * NW / 4;
    static_assert(LDS_BYTES <= 160 * 1024, "the waves' regions fit the CU's LDS");
    static_assert((TM & (TM - 1)) == 0 && (TN & (TN - 1)) == 0, "powers of two: the chunk swizzle stays inside a row");
};

// Byte offset of 16-byte chunk c of row k in a region whose rows are 16 * T bytes. The 32 lanes the LDS serves together
// in a transpose read point at 8 rows of two 32-row groups; rows of one chunk are spread by moving every second
// 32-row group by 8 rows (128 bytes), wider rows by the chunk swizzle of the tiled kernels.
template <int T>
__device__ __forceinline__ uint32_t fewrows_at(int k, int c) {
    if constexpr (T == 1) return (uint32_t)((k ^ (((k >> 5) & 1) << 3)) << 4);
    else return (uint32_t)(k * 16 * T + ((c ^ swizzle_of_row<16 * T>(k)) << 4));
}

// 16 bytes from base + off of a matrix that ends at base + end (end >= 16): past the end the bytes are undefined but
// nothing is read there. SHIFT false: the caller knows that off + 16 <= end.
template <bool SHIFT, bool STREAM = false>
__device__ __forceinline__ u32x4_lds load16(const uint8_t *base, uint32_t off, uint32_t end) {
    if constexpr (STREAM) return __builtin_nontemporal_load((const u32x4_any *)(base + off));
    if constexpr (!SHIFT) return *(const u32x4_any *)(base + off);
    const uint32_t at = off < end - 16 ? off : end - 16;
    return *(const u32x4_any *)(base + at);
}
// Moves the bytes of a cut load back to where they would have been.
__device__ __forceinline__ u32x4_lds shift_back(u32x4_lds v, uint32_t off, uint32_t end) {
    const uint32_t d = off < end - 16 ? 0 : off - (end - 16);         // 16 and more: every byte is past the end
    const uint32_t x0 = d & 8 ? v[2] : v[0], x1 = d & 8 ? v[3] : v[1];
    const uint32_t y0 = d & 4 ? x1 : x0, y1 = d & 4 ? (d & 8 ? 0 : v[2]) : x1, y2 = d & 4 ? v[3] : v[2], y3 = v[3];
    u32x4_lds r;
    r[0] = __builtin_amdgcn_alignbyte(y1, y0, d & 3);
    r[1] = __builtin_amdgcn_alignbyte(y2, y1, d & 3);
    r[2] = __builtin_amdgcn_alignbyte(y3, y2, d & 3);
    r[3] = __builtin_amdgcn_alignbyte(0, y3, d & 3);
    return r;
}

// What one wave does with one K block: loads into registers, the private LDS region, fragments, MFMAs.
template <int TM, int TN, bool BYTES, bool STREAM = false>
struct FewRowsWave {
    static constexpr int BM = 16 * TM, BN = 16 * TN;
    static constexpr int NLA = 2 * TM, NLB = 2 * TN;                  // 16-byte loads per lane and K block
    static_assert(128 % BN == 0, "a strip lies in one b_scale block");
    // One K block on its way: raw bytes of A and B, scales.
    struct Block {
        u32x4_lds a[NLA], b[NLB];
        float sa[TM], sb;
    };
    const uint8_t *A, *B;
    const float *SA, *SB;
    uint8_t *region;
    int ldm, N, K, QN, nb, lane, first;
    int zero = 0;                                                     // see gemm_fp8_blockscale_grouped_strips
    uint32_t off_a0, off_b0;
    int row_s[TM];

    // Tile m0, n0 of a problem of M rows that starts at column `first` of an A with ldm columns.
    __device__ __forceinline__ FewRowsWave(const uint8_t *A_, const uint8_t *B_, const float *SA_, const float *SB_, int M,
                                           int first_, int ldm_, int N_, int K_, int m0, int n0, uint8_t *region_, int lane_)
        : A(A_ + first_), B(B_), SA(SA_ + first_), SB(SB_), region(region_), ldm(ldm_), N(N_), K(K_), QN((N_ + 127) / 128),
          nb(n0 >> 7), lane(lane_), first(first_) {
        // Load i of a lane: 16-byte chunk lane % T of K row lane / T + i * 64 / T of the block
        int m = m0 + 16 * (lane % TM), n = n0 + 16 * (lane % TN);
        if (m >= M) m = m0;                                           // a whole chunk past M or N: any bytes will do
        if (n >= N) n = n0;
        off_a0 = (uint32_t)(lane / TM) * (uint32_t)ldm + (uint32_t)m;
        off_b0 = (uint32_t)(lane / TN) * (uint32_t)N + (uint32_t)n;
#pragma unroll
        for (int j = 0; j < TM; j++) {
            const int row = m0 + 16 * j + (lane & 15);
            row_s[j] = row < M ? row : M - 1;
        }
    }
    __device__ __forceinline__ uint32_t off_a(int i) const { return off_a0 + (uint32_t)(i * (64 / TM)) * (uint32_t)ldm; }
    __device__ __forceinline__ uint32_t off_b(int i) const { return off_b0 + (uint32_t)(i * (64 / TN)) * (uint32_t)N; }
    __device__ __forceinline__ uint32_t dst_a(int i) const { return fewrows_at<TM>(lane / TM + i * (64 / TM), lane % TM); }
    __device__ __forceinline__ uint32_t dst_b(int i) const {
        return BK * BM + fewrows_at<TN>(lane / TN + i * (64 / TN), lane % TN);
    }
    // Bytes from a K block's first row (column `skip` of it) to the end of the matrix, needed to cut the loads of the last
    // rows (below 2^32 always suffices: a K block's own offsets are).
    __device__ __forceinline__ uint32_t rest(int kb, int ld, int skip) const {
        const unsigned long long r = (unsigned long long)(K - kb * BK) * (unsigned)ld - (unsigned)skip;
        return r < 0xffffffffull ? (uint32_t)r : 0xffffffffu;
    }
    __device__ __forceinline__ void fetch(Block &x, int kb) const {
        const uint8_t *pb = B + (size_t)kb * BK * N, *pa = A + (size_t)kb * BK * ldm;
        const uint32_t end_b = rest(kb, N, 0), end_a = rest(kb, ldm, first);
#pragma unroll
        for (int q = 0; q < NLB; q++) x.b[q] = load16<BYTES, STREAM>(pb, off_b(q), end_b);
#pragma unroll
        for (int q = 0; q < NLA; q++) x.a[q] = load16<true>(pa, off_a(q), end_a);
#pragma unroll
        for (int j = 0; j < TM; j++) x.sa[j] = SA[(size_t)kb * ldm + row_s[j]];
        x.sb = SB[(size_t)kb * QN + nb + zero];
    }
    __device__ __forceinline__ i32x8 fragment(uint32_t at, int pitch) const {       // four transpose reads, 8 rows apart
        i32x8 f;
#pragma unroll
        for (int t = 0; t < 4; t++) {
            const i32x2 v = __builtin_amdgcn_ds_read_tr8_b64_v2i32((RF_LDS i32x2 *)(region + at + t * 8 * pitch));
            f[2 * t] = v[0];
            f[2 * t + 1] = v[1];
        }
        return f;
    }
    // rows 8 t further on lie at a fixed distance except in regions of one-chunk rows, whose every second 32-row group
    // is moved by 8 rows: row ^ 8 there
    __device__ __forceinline__ i32x8 fragment_1(uint32_t base, int krow, int L) const {
        i32x8 f;
#pragma unroll
        for (int t = 0; t < 4; t++) {
            const i32x2 v = __builtin_amdgcn_ds_read_tr8_b64_v2i32(
                (RF_LDS i32x2 *)(region + base + fewrows_at<1>(krow + 8 * t, 0) + 8 * (L & 1)));
            f[2 * t] = v[0];
            f[2 * t + 1] = v[1];
        }
        return f;
    }
    // The bytes of the block into the region. Its registers are free afterwards, but for the scales.
    __device__ __forceinline__ void stage(Block &x, int kb) const {
        if (kb == K / BK - 1) {                                       // only the matrix's last rows have cut loads
            const uint32_t end_b = rest(kb, N, 0), end_a = rest(kb, ldm, first);
            if constexpr (BYTES)
#pragma unroll
                for (int q = 0; q < NLB; q++) x.b[q] = shift_back(x.b[q], off_b(q), end_b);
#pragma unroll
            for (int q = 0; q < NLA; q++) x.a[q] = shift_back(x.a[q], off_a(q), end_a);
        }
#pragma unroll
        for (int q = 0; q < NLB; q++) *(u32x4_lds *)(region + dst_b(q)) = x.b[q];
#pragma unroll
        for (int q = 0; q < NLA; q++) *(u32x4_lds *)(region + dst_a(q)) = x.a[q];
    }
    // The products of the staged block: use(j, c, p) for every 16 x 16 tile, p summed from zero.
    template <typename Use>
    __device__ __forceinline__ void multiply(Use use) const {
        const int L = lane & 15, krow = 32 * (lane >> 4) + (L >> 1);
        i32x8 bf[TN], af[TM];
#pragma unroll
        for (int c = 0; c < TN; c++)
            bf[c] = TN == 1 ? fragment_1(BK * BM, krow, L) : fragment(BK * BM + fewrows_at<TN>(krow, c) + 8 * (L & 1), BN);
#pragma unroll
        for (int c = 0; c < TM; c++)
            af[c] = TM == 1 ? fragment_1(0, krow, L) : fragment(fewrows_at<TM>(krow, c) + 8 * (L & 1), BM);
#pragma unroll
        for (int j = 0; j < TM; j++)
#pragma unroll
            for (int c = 0; c < TN; c++)
                use(j, c, __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(bf[c], af[j], (f32x4){0.f, 0.f, 0.f, 0.f}, 0, 0, 0, 0,
                                                                           0, 0));
    }
};

// Stores a lane's C[m][n .. n + 3] of tile t of a workgroup's tile.
template <int TN>
__device__ __forceinline__ void fewrows_store(uint16_t *C, int M, int N, int m0, int n0, int t, int lane, const f32x4 &s) {
    const int m = m0 + 16 * (t / TN) + (lane & 15), n = n0 + 16 * (t % TN) + 4 * (lane >> 4);
    if (m >= M) return;
    uint16_t *out = C + (size_t)m * N + n;
    const uint32_t lo = pack_bf16x2(s[0], s[1]), hi = pack_bf16x2(s[2], s[3]);
    if (n + 4 <= N && ((uintptr_t)out & 7) == 0) {
        *(uint2 *)out = make_uint2(lo, hi);
    } else {
        if (n < N) out[0] = (uint16_t)lo;
        if (n + 1 < N) out[1] = (uint16_t)(lo >> 16);
        if (n + 2 < N) out[2] = (uint16_t)hi;
        if (n + 3 < N) out[3] = (uint16_t)(hi >> 16);
    }
}

// Grid: x = column strips * row blocks (row blocks innermost: they share the strip's B), y = K splits of kb_per_split
// blocks, every split at least one. A [K][ldm] (M of the ldm columns belong to this problem), SA [K/128][ldm], B [K][N],
// C [M][N]. Any M, N >= 1, any alignment of A, B and C; ldm and N below 2^25 (32-bit offsets inside a K block). BYTES
// false needs N % 16 == 0 and a 16-byte aligned B. SPLIT (gridDim.y > 1): counters holds a zero per item (gridDim.x) and
// is zero again afterwards, slots gridDim.x * gridDim.y * TM * TN KiB, 16-byte aligned.
template <int TM, int TN, int NW, int DEPTH, bool SPLIT, bool BYTES>
__global__ __launch_bounds__(NW * 64, (FewRowsGeom<TM, TN, NW, DEPTH>::WAVES_PER_SIMD)) void gemm_fp8_blockscale_fewrows(
    const uint8_t *__restrict__ A, const uint8_t *__restrict__ B, const float *__restrict__ SA,
    const float *__restrict__ SB, uint16_t *__restrict__ C, int M, int ldm, int N, int K, int kb_per_split, int row_blocks,
    unsigned *__restrict__ counters, float *__restrict__ slots) {
    using G = FewRowsGeom<TM, TN, NW, DEPTH>;
    using W = FewRowsWave<TM, TN, BYTES>;
    extern __shared__ __attribute__((aligned(1024))) uint8_t lds[];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
    // neighbouring strips on one XCD: a 32-column piece of a row of B is a quarter of a cache line
    const int xcd = blockIdx.x % NUM_XCD, idx = blockIdx.x / NUM_XCD, per = gridDim.x / NUM_XCD, rem = gridDim.x % NUM_XCD;
    const int item = xcd * per + (xcd < rem ? xcd : rem) + idx;
    const int n0 = item / row_blocks * G::BN, m0 = item % row_blocks * G::BM;
    const int QK = K / BK;
    const int kb_begin = blockIdx.y * kb_per_split, kb_end = kb_begin + kb_per_split < QK ? kb_begin + kb_per_split : QK;
    const int count = (kb_end - kb_begin - wave + NW - 1) / NW;       // this wave's K blocks: kb_begin + wave + NW * i
    W w(A, B, SA, SB, M, 0, ldm, N, K, m0, n0, lds + wave * G::REGION, lane);
    if constexpr (DEPTH == 1) asm("" : "+v"(w.zero));             // see gemm_fp8_blockscale_grouped_strips
    auto kb_of = [&](int i) { return kb_begin + wave + NW * i; };
    f32x4 acc[TM][TN];
#pragma unroll
    for (int j = 0; j < TM; j++)
#pragma unroll
        for (int i = 0; i < TN; i++) acc[j][i] = (f32x4){0.f, 0.f, 0.f, 0.f};
    auto products = [&](const float (&s)[TM]) {
        w.multiply([&](int j, int c, const f32x4 &p) {
#pragma unroll
            for (int e = 0; e < 4; e++) acc[j][c][e] = __builtin_fmaf(s[j], p[e], acc[j][c][e]);
        });
    };
    auto scales_of = [&](const typename W::Block &x, float (&s)[TM]) {
#pragma unroll
        for (int j = 0; j < TM; j++) s[j] = x.sa[j] * x.sb;
    };
    static_assert(DEPTH >= 1 && DEPTH <= 4, "one to four K blocks at a time");
    if constexpr (DEPTH == 1) {
        // The next K block is asked for as soon as this one's bytes are in LDS, and travels while this one is multiplied: for
        // waves with two and more K blocks and too many registers in a block to ask for all of them. us against one block
        // after the other (same tiles): 128 x 7168 x 2048 10.7 -> 9.7, 200 x 3072 x 1536 8.1 -> 7.5, 400 x 2003 x 7168 28.5 -> 25.8;
        // against the best plan before: 48 x 7168 x 2048 8.5 -> 7.4, 77 x 2048 x 2048 6.0 -> 5.1.
        auto step = [&](typename W::Block &x, int i, auto more) {
            w.stage(x, kb_of(i));
            float s[TM];
            scales_of(x, s);
            __builtin_amdgcn_sched_barrier(0);
            if constexpr (decltype(more)::value) w.fetch(x, kb_of(i + 1));
            __builtin_amdgcn_sched_barrier(0);
            products(s);
            __builtin_amdgcn_sched_barrier(0);
        };
        if (count > 0) {
            typename W::Block x;
            w.fetch(x, kb_of(0));
            int i = 0;
            for (; i + 1 < count; i++) step(x, i, IntTag<1>{});
            step(x, i, IntTag<0>{});
        }
    } else {
        // up to DEPTH K blocks asked for, then used in order; straight-line code for every count, so that each wait is for a
        // known number of younger loads
        auto batch = [&](auto count_c, int i) {
            constexpr int n = decltype(count_c)::value;
            typename W::Block x[n];
#pragma unroll
            for (int d = 0; d < n; d++) w.fetch(x[d], kb_of(i + d));
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int d = 0; d < n; d++) {
                w.stage(x[d], kb_of(i + d));
                float s[TM];
                scales_of(x[d], s);
                products(s);
                __builtin_amdgcn_sched_barrier(0);
            }
        };
        int i = 0;
        for (; i + DEPTH <= count; i += DEPTH) batch(IntTag<DEPTH>{}, i);
        if (DEPTH > 3 && count - i == 3) batch(IntTag<3>{}, i);
        else if (DEPTH > 2 && count - i == 2) batch(IntTag<2>{}, i);
        else if (count - i == 1) batch(IntTag<1>{}, i);
    }

    // the waves' sums through LDS, tile (j, c) of wave w at ((w * TM + j) * TN + c) * 1 KiB, lane l at + 16 l
    __syncthreads();
#pragma unroll
    for (int j = 0; j < TM; j++)
#pragma unroll
        for (int c = 0; c < TN; c++) *(f32x4 *)(lds + ((wave * TM + j) * TN + c) * 1024 + lane * 16) = acc[j][c];
    __syncthreads();
    auto store = [&](int t, const f32x4 &s) { fewrows_store<TN>(C, M, N, m0, n0, t, lane, s); };
    const int splits = gridDim.y;
    float *mine = slots + ((size_t)item * splits + blockIdx.y) * (TM * TN * 256) + lane * 4;
    for (int t = wave; t < TM * TN; t += NW) {
        f32x4 s = *(const f32x4 *)(lds + t * 1024 + lane * 16);
#pragma unroll
        for (int u = 1; u < NW; u++) {
            const f32x4 v = *(const f32x4 *)(lds + (u * TM * TN + t) * 1024 + lane * 16);
            s[0] += v[0]; s[1] += v[1]; s[2] += v[2]; s[3] += v[3];
        }
        if constexpr (SPLIT) {
            // system scope: written through, so that the acknowledgement below means "where every XCD's loads look"
            asm volatile("global_store_dwordx4 %0, %1, off sc0 sc1\n\ts_nop 1" :: "v"(mine + t * 256), "v"(s) : "memory");
        } else {
            store(t, s);
        }
    }
    if constexpr (SPLIT) {
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        __syncthreads();
        RF_LDS unsigned *mailbox = (RF_LDS unsigned *)lds;            // every wave has read the sums exchanged there
        if (threadIdx.x == 0) {
            const unsigned w = arrival_weight(blockIdx.y, (unsigned)splits);
            *mailbox = __hip_atomic_fetch_add(counters + item, w, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) + w;
        }
        __syncthreads();
        if (*mailbox != 0u) return;                                   // not the last
        const float *first = slots + (size_t)item * splits * (TM * TN * 256) + lane * 4;
        for (int t = wave; t < TM * TN; t += NW) {
            f32x4 s = {0.f, 0.f, 0.f, 0.f};
            for (int q0 = 0; q0 < splits; q0 += 8) {
                uint64_t v[8][2];
#pragma unroll
                for (int q = 0; q < 8; q++)
                    if (q0 + q < splits) {
                        const uint64_t *p = (const uint64_t *)(first + ((size_t)(q0 + q) * TM * TN + t) * 256);
                        v[q][0] = __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
                        v[q][1] = __hip_atomic_load(p + 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
                    }
#pragma unroll
                for (int q = 0; q < 8; q++)
                    if (q0 + q < splits) {
                        const f32x2 lo = __builtin_bit_cast(f32x2, v[q][0]), hi = __builtin_bit_cast(f32x2, v[q][1]);
                        s[0] += lo[0]; s[1] += lo[1]; s[2] += hi[0]; s[3] += hi[1];
                    }
            }
            store(t, s);
        }
    }
}

// Grouped forms for groups of a few rows each (an expert layer in decode): what counts is streaming every group's weights,
// N * K bytes each. A is read where the caller has it, at any byte and with a group starting at any column, so nothing is
// staged; the sums are those of the tiled forms to the bit, K blocks in order.
// Grid as for gemm_fp8_blockscale_grouped, a work item being a strip of columns and a block of 16 TM rows (row blocks of a
// strip side by side). table.row_start[g]: column of A at which group g starts (any number), out_row_start: its rows of C
// and their number. N % 16 == 0, B 16-byte aligned.
//
// First form: every wave has columns of its own and walks all of K with DEPTH K blocks on their way in registers; the waves
// share nothing, so there is no barrier. Strips of 128 columns (TN = 8): a load instruction then covers eight whole cache
// lines (an L1 miss fetches a line whatever part of it is asked for), and all strips of a launch are resident at once. Narrower
// strips ran at half the rate: 48 rows over 32 groups, 2048 x 7168 (366 MB of weights), columns per wave 16: 228 us, 32: 139,
// 64: 100, 128: 72 us with two K blocks on their way against 96.7 us for the tiled form with its staging copy.
// Bound by the streaming of B, whose rate depends on how much of a row is read at a time and on what the reads leave in the
// Infinity Cache (a plain read of the same matrices: 128 columns by one workgroup 4.96 TB/s, 256 5.7, 512 6.4; neighbouring
// strips dealt to different XCDs 5.4, 6.0, 6.6; with the non-temporal hint besides 5.9, 6.5). So items are dealt, the waves of
// a workgroup hold neighbouring strips (four where there are enough of them: 36 groups of 7168 x 2048 89.5 -> 82.3 us, 30 of
// 4096 x 2048 48 -> 45.3), and more weights than the Infinity Cache keeps are read with the hint (STREAM): the 366 MB
// above 72.5 -> 67.0 us = 5.5 TB/s. With fewer than about one strip per compute unit bound by the chain of 56 loads (0.95 us each).
template <int TM, int TN, int NW, int DEPTH, int WAVES_PER_SIMD, bool STREAM>
__global__ __launch_bounds__(NW * 64, WAVES_PER_SIMD) void gemm_fp8_blockscale_grouped_strips(
    const uint8_t *__restrict__ A, const uint8_t *__restrict__ B, const float *__restrict__ SA,
    const float *__restrict__ SB, uint16_t *__restrict__ C, int M_total, int N, int K, int groups, const GroupTable table) {
    using W = FewRowsWave<TM, TN, false, STREAM>;
    extern __shared__ __attribute__((aligned(1024))) uint8_t lds[];
    int grp, local;
    if (!grouped_work_item<true>(table, groups, grp, local)) return;
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
    const int out0 = table.out_row_start[grp], rows = table.out_row_start[grp + 1] - out0;
    const int row_blocks = (rows + 16 * TM - 1) / (16 * TM);
    const int m0 = local % row_blocks * (16 * TM), n0 = (local / row_blocks * NW + wave) * (16 * TN);
    if (n0 >= N) return;                                              // waves share nothing
    const int QK = K / BK, QN = (N + 127) / 128;
    W w(A, B + (size_t)grp * K * N, SA, SB + (size_t)grp * QK * QN, rows, table.row_start[grp], M_total, N, K, m0, n0,
        lds + wave * (BK * 16 * (TM + TN)), lane);
    // b_scale's index in a vector register: a scalar load on its way would make every wait for LDS a wait for memory
    asm("" : "+v"(w.zero));
    f32x4 acc[TM][TN];
#pragma unroll
    for (int j = 0; j < TM; j++)
#pragma unroll
        for (int c = 0; c < TN; c++) acc[j][c] = (f32x4){0.f, 0.f, 0.f, 0.f};
    typename W::Block x[DEPTH];
    auto fetch = [&](typename W::Block &b, int kb) { w.fetch(b, kb < QK ? kb : QK - 1); };   // (past the end: not used)
    auto step = [&](typename W::Block &b, int kb, auto more) {
        w.stage(b, kb);
        float s[TM];
#pragma unroll
        for (int j = 0; j < TM; j++) s[j] = b.sa[j] * b.sb;
        __builtin_amdgcn_sched_barrier(0);
        if constexpr (decltype(more)::value) fetch(b, kb + DEPTH);
        __builtin_amdgcn_sched_barrier(0);
        w.multiply([&](int j, int c, const f32x4 &p) {
#pragma unroll
            for (int e = 0; e < 4; e++) acc[j][c][e] = __builtin_fmaf(s[j], p[e], acc[j][c][e]);
        });
        __builtin_amdgcn_sched_barrier(0);
    };
#pragma unroll
    for (int d = 0; d < DEPTH; d++) fetch(x[d], d);
    int kb = 0;
    for (; kb + DEPTH < QK; kb += DEPTH)
#pragma unroll
        for (int d = 0; d < DEPTH; d++) step(x[d], kb + d, IntTag<1>{});
#pragma unroll
    for (int d = 0; d < DEPTH; d++)
        if (kb + d < QK) step(x[d], kb + d, IntTag<0>{});
#pragma unroll
    for (int j = 0; j < TM; j++)
#pragma unroll
        for (int c = 0; c < TN; c++) fewrows_store<TN>(C + (size_t)out0 * N, rows, N, m0, n0, j * TN + c, lane, acc[j][c]);
}

// Second form, for launches of few strips: the waves of a workgroup take K blocks in turn. After every round of NW K blocks
// they leave the blocks' products and scales in their regions, and the wave that holds an output tile folds them in K order;
// the next rounds' loads stay in flight across the round's two barriers. 8 groups of 2 rows, 2048 x 7168: 76 us (tiled) and
// 54 us (first form) -> 36 us; with four strips per compute unit the barriers cost more than the parallel chain saves.
template <int TM, int TN, int NW, int DEPTH, int WAVES_PER_SIMD>
__global__ __launch_bounds__(NW * 64, WAVES_PER_SIMD) void gemm_fp8_blockscale_grouped_ksplit(
    const uint8_t *__restrict__ A, const uint8_t *__restrict__ B, const float *__restrict__ SA,
    const float *__restrict__ SB, uint16_t *__restrict__ C, int M_total, int N, int K, int groups, const GroupTable table) {
    using W = FewRowsWave<TM, TN, false>;
    constexpr int REGION = BK * 16 * (TM + TN), SCALES = TM * TN * 1024;
    static_assert(SCALES + TM * 64 <= REGION, "a round's products and scales take the place of its operands");
    constexpr int TILES = (TM * TN + NW - 1) / NW;                    // output tiles a wave folds: wave, wave + NW, ...
    extern __shared__ __attribute__((aligned(1024))) uint8_t lds[];
    int grp, local;
    if (!grouped_work_item(table, groups, grp, local)) return;
    const int out0 = table.out_row_start[grp], rows = table.out_row_start[grp + 1] - out0;
    const int row_blocks = (rows + 16 * TM - 1) / (16 * TM);
    const int m0 = local % row_blocks * (16 * TM), n0 = local / row_blocks * (16 * TN);
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
    const int QK = K / BK, QN = (N + 127) / 128, rounds = (QK + NW - 1) / NW;
    uint8_t *region = lds + wave * REGION;
    W w(A, B + (size_t)grp * K * N, SA, SB + (size_t)grp * QK * QN, rows, table.row_start[grp], M_total, N, K, m0, n0, region,
        lane);
    asm("" : "+v"(w.zero));
    typename W::Block x[DEPTH];
    // a wave without a K block in the last round asks for the last one and does not use it
    auto fetch = [&](typename W::Block &b, int r) {
        const int kb = r * NW + wave;
        w.fetch(b, kb < QK ? kb : QK - 1);
    };
    f32x4 acc[TILES];
#pragma unroll
    for (int i = 0; i < TILES; i++) acc[i] = (f32x4){0.f, 0.f, 0.f, 0.f};
    constexpr int H = NW < 4 ? NW : 4;
    auto fold = [&](f32x4 &sum, int t) {
        const uint8_t *at = lds + t * 1024 + lane * 16, *at_s = lds + SCALES + t / TN * 64 + (lane & 15) * 4;
#pragma unroll
        for (int b0 = 0; b0 < NW; b0 += H) {
            f32x4 p[H];
            float s[H];
#pragma unroll
            for (int b = 0; b < H; b++) {
                p[b] = *(const f32x4 *)(at + (b0 + b) * REGION);
                s[b] = *(const float *)(at_s + (b0 + b) * REGION);
            }
#pragma unroll
            for (int b = 0; b < H; b++)
#pragma unroll
                for (int e = 0; e < 4; e++) sum[e] = __builtin_fmaf(s[b], p[b][e], sum[e]);
        }
    };
    auto step = [&](typename W::Block &b, int r, auto more) {
        const int kb = r * NW + wave;
        float s[TM];
        if (kb < QK) {
            w.stage(b, kb);
#pragma unroll
            for (int j = 0; j < TM; j++) s[j] = b.sa[j] * b.sb;
        }
        __builtin_amdgcn_sched_barrier(0);
        if constexpr (decltype(more)::value) fetch(b, r + DEPTH);
        __builtin_amdgcn_sched_barrier(0);
        auto leave = [&](int j, int c, const f32x4 &p) { *(f32x4 *)(region + (j * TN + c) * 1024 + lane * 16) = p; };
        if (kb < QK) {
            w.multiply(leave);
        } else {                                                      // -0 * 0 = -0, and x + -0 = x for every x
#pragma unroll
            for (int j = 0; j < TM; j++) {
                s[j] = -0.f;
#pragma unroll
                for (int c = 0; c < TN; c++) leave(j, c, (f32x4){0.f, 0.f, 0.f, 0.f});
            }
        }
        if (lane < 16)
#pragma unroll
            for (int j = 0; j < TM; j++) *(float *)(region + SCALES + j * 64 + lane * 4) = s[j];
        __syncthreads();
#pragma unroll
        for (int i = 0; i < TILES; i++)
            if (wave + i * NW < TM * TN) fold(acc[i], wave + i * NW);
        __syncthreads();
    };
#pragma unroll
    for (int d = 0; d < DEPTH; d++) fetch(x[d], d);
    int r = 0;
    for (; r + DEPTH < rounds; r += DEPTH)
#pragma unroll
        for (int d = 0; d < DEPTH; d++) step(x[d], r + d, IntTag<1>{});
#pragma unroll
    for (int d = 0; d < DEPTH; d++)
        if (r + d < rounds) step(x[d], r + d, IntTag<0>{});
#pragma unroll
    for (int i = 0; i < TILES; i++)
        if (wave + i * NW < TM * TN)
            fewrows_store<TN>(C + (size_t)out0 * N, rows, N, m0, n0, wave + i * NW, lane, acc[i]);
}

}  // namespace rf

// Block quantisers that produce the GEMM's operands on the GPU, in the launcher's layouts.
//
// The reference has no quantiser: its harness draws fp8 bytes and scales directly
// (tests/gemm/gemm_test.cpp:64-99), and the recipe that real callers use is only stated in words: per
// (row, 128-wide K block) for activations and per 128x128 block for weights, scale = amax / 448, value =
// e4m3fn(x / scale) with round-to-nearest-even. These kernels implement exactly that recipe and write
//   a[k*M + m]  (fp8, the [K][M] layout of the launcher),  as[kb*M + m]
//   b[k*N + n]  (fp8, [K][N]),                             bs[kb*QN + nb]
// so the step before the GEMM needs no host work and no transpose pass: the transposition happens in LDS on the
// way out. Both are pure streaming kernels (4 or 2 bytes read, 1 byte written per element): HBM-bound.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace rf {

typedef unsigned quant_u32x4 __attribute__((ext_vector_type(4)));
typedef unsigned quant_u32x4_any __attribute__((ext_vector_type(4), aligned(1)));
typedef unsigned quant_u32_any __attribute__((aligned(1)));
// 16 bytes of output, written through to memory (sc1) instead of left dirty in the XCD's L2: the GEMM that reads them
// runs on all XCDs, so they have to leave this L2 anyway, and written through they do so while the kernel still runs
// (6144 x 7168 from bf16: 26.2-27.0 -> 25.1-25.2 us, from fp32 36.0 -> 35.7 us).
// (The statement carries its own wait states: a store of more than 8 bytes reads its data registers a little after it
// has been issued, and the compiler's hazard check does not look inside it.)
__device__ __forceinline__ void store16_through(void *p, const uint4 &v) {
    const quant_u32x4 w = {v.x, v.y, v.z, v.w};
    asm volatile("global_store_dwordx4 %0, %1, off sc1\n\ts_nop 1" :: "v"(p), "v"(w) : "memory");
}

template <int V> struct IntConst { static constexpr int value = V; };
typedef unsigned short u16x2 __attribute__((ext_vector_type(2)));

// fp32 -> OCP e4m3fn code, round to nearest even, anything that rounds above 448 (and NaN) becomes NaN (0x7F).
// Integer/exact-float arithmetic only, so that it agrees bit for bit with a CPU implementation; no branches.
__device__ __forceinline__ uint32_t f32_to_e4m3fn_code(float f) {
    const uint32_t u = __builtin_bit_cast(uint32_t, f);
    const uint32_t sign = (u >> 24) & 0x80u, abits = u & 0x7fffffffu;
    const int e = (int)(abits >> 23) - 127;                   // floor(log2 |f|) for normal inputs
    int q = e - 3;                                            // exponent of the rounding quantum: 3 mantissa bits
    q = q < -9 ? -9 : q;                                      // subnormal range of e4m3: quantum 2^-9
    q = q > 120 ? 120 : q;                                    // Inf / NaN: keep the factor below finite
    const float inv_quantum = __builtin_bit_cast(float, (uint32_t)(127 - q) << 23);
    const float r = __builtin_rintf(__builtin_bit_cast(float, abits) * inv_quantum);   // exact product, RNE to integer
    // r is in [0,16] for finite inputs; code = exponent field (q+10) and mantissa r-8, which also covers the subnormal
    // codes (q = -9) and the carry r == 16 into the next exponent
    const bool finite = abits < 0x7f800000u;
    const int code = ((q + 10) << 3) + (int)(finite ? r : 0.f) - 8;
    return sign | (uint32_t)((code > 126 || !finite) ? 0x7F : code);
}

// Four fp32 values -> four e4m3fn codes packed in one word (value j in byte j), same results as f32_to_e4m3fn_code.
// Uses the conversion instruction of gfx950 (v_cvt_pk_fp8_f32: OCP e4m3fn, round to nearest even, values that round
// above 448 and infinities become NaN). Compared over all 2^32 inputs it differs from the integer encoder only for
// NaNs with a clear sign bit (it returns 0xFF, the encoder keeps the sign: 0x7F), so a group that contains a NaN goes
// through the integer encoder.
__device__ __forceinline__ uint32_t f32x4_to_e4m3fn_codes(float x0, float x1, float x2, float x3) {
    int w = __builtin_amdgcn_cvt_pk_fp8_f32(x0, x1, 0, false);
    w = __builtin_amdgcn_cvt_pk_fp8_f32(x2, x3, w, true);
    if (x0 != x0 || x1 != x1 || x2 != x2 || x3 != x3)
        w = (int)(f32_to_e4m3fn_code(x0) | (f32_to_e4m3fn_code(x1) << 8) | (f32_to_e4m3fn_code(x2) << 16) |
                  (f32_to_e4m3fn_code(x3) << 24));
    return (uint32_t)w;
}

// Plain elementwise cast fp32 -> e4m3fn (no scaling), four values per thread.
__global__ __launch_bounds__(256) void cast_f32_to_e4m3fn(const float *__restrict__ x, uint8_t *__restrict__ out, size_t n) {
    const size_t i = ((size_t)blockIdx.x * 256 + threadIdx.x) * 4;
    if (i + 4 <= n) {
        const float4 v = *(const float4 *)(x + i);
        *(uint32_t *)(out + i) = f32x4_to_e4m3fn_codes(v.x, v.y, v.z, v.w);
    } else {
        for (size_t j = i; j < n; j++) out[j] = (uint8_t)f32_to_e4m3fn_code(x[j]);
    }
}

__device__ __forceinline__ float bf16_bits_to_f32(uint32_t h) { return __builtin_bit_cast(float, h << 16); }

// Maximum over each aligned group of 16 lanes, left in all of them, for N unsigned values at once: four DPP steps
// (swap within pairs, within quads, rotate the 16-lane row by 4 and by 8) instead of LDS-crossbar shuffles, each one
// v_max_u32 with a DPP operand. Written as asm because the compiler emits move + max for the builtin form. A DPP
// operand must not be read within two instructions of the VALU write that produced it, and the compiler's hazard
// recogniser does not look inside asm statements (it may also place a register copy right in front of one): every
// step carries its own two wait states.
template <int N>
__device__ __forceinline__ void max_over_16_lanes(uint32_t (&a)[N]) {
#pragma unroll
    for (int i = 0; i < N; i++)
        asm volatile("s_nop 1\n\tv_max_u32_dpp %0, %0, %0 quad_perm:[1,0,3,2] row_mask:0xf bank_mask:0xf" : "+v"(a[i]));
#pragma unroll
    for (int i = 0; i < N; i++)
        asm volatile("s_nop 1\n\tv_max_u32_dpp %0, %0, %0 quad_perm:[2,3,0,1] row_mask:0xf bank_mask:0xf" : "+v"(a[i]));
#pragma unroll
    for (int i = 0; i < N; i++)
        asm volatile("s_nop 1\n\tv_max_u32_dpp %0, %0, %0 row_ror:4 row_mask:0xf bank_mask:0xf" : "+v"(a[i]));
#pragma unroll
    for (int i = 0; i < N; i++)
        asm volatile("s_nop 1\n\tv_max_u32_dpp %0, %0, %0 row_ror:8 row_mask:0xf bank_mask:0xf" : "+v"(a[i]));
    asm volatile("s_nop 1" ::: "memory");     // the compiler may follow up with a DPP or lane-crossing read of a[N-1]
}

// The same for one float with "a NaN never wins" comparisons (the rare path of rows that contain a NaN).
__device__ __forceinline__ float max_over_16_lanes_nan_safe(float a) {
    auto step = [&](auto ctrl) {
        const float o = __builtin_bit_cast(
            float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, a), decltype(ctrl)::value, 0xf, 0xf, false));
        a = o > a ? o : a;
    };
    step(IntConst<0xB1>{});      // quad_perm [1,0,3,2]
    step(IntConst<0x4E>{});      // quad_perm [2,3,0,1]
    step(IntConst<0x124>{});     // row_ror 4
    step(IntConst<0x128>{});     // row_ror 8
    return a;
}

// a / 448 for a in [2^-100, FLT_MAX]: product with RN(1/448) plus one correction step through the exact remainder.
// Compared with the IEEE division over every float in that range on the CPU: identical (below 2^-100 the remainder
// underflows and it is not).
__device__ __forceinline__ float div_by_448(float a) {
    constexpr float C = 1.0f / 448.0f;
    const float q = a * C;
    const float r = __builtin_fmaf(-q, 448.0f, a);
    return __builtin_fmaf(r, C, q);
}

// Codes of x[j] / s[j], j = 0..3, packed in one word. The value to encode is fl32(x / scale). A correctly rounded division costs
// ~11 instructions per element. Instead, with r = rcp(scale) (the hardware reciprocal, within a few ulp of 1 / scale),
// x * (r * (1 + 2^-20)) and x * (r * (1 - 2^-20)) (rup, rdown) are, in magnitude, above and below the exact quotient and
// its fp32 rounding (the factors' rounding errors and the reciprocal's error are below 2^-21 together). The fp8 conversion is
// monotonic, so if the two products convert to the same code, fl32(x / scale) converts to that code too. When they differ
// (a rounding boundary is that close: about 1 element in 10^5 for fp32 sources, far more often for bf16 ones) the group of
// four is redone with the exact quotient; when a row contains a NaN or an infinity, or its scale lies outside (2^-60, 2^60)
// (fast false), with the IEEE division and the NaN-aware encoder.
template <bool IN_BF16>
__device__ __forceinline__ uint32_t codes_of_quotients(const float (&x)[4], const float (&s)[4], const float (&rup)[4],
                                                       const float (&rdown)[4], bool fast) {
    // bf16 sources go straight to the exact quotient: x and amax have 8-bit mantissas, so x / scale often IS a rounding
    // boundary, one such lane in 64 sends the whole wave to the exact path, and with 256 values per wave and group that is
    // nearly every time; the bracket would only be computed on top of it.
    int hi = 0, lo = 1;
    if constexpr (!IN_BF16) {
        float yu[4], yd[4];
#pragma unroll
        for (int j = 0; j < 4; j++) {
            yu[j] = x[j] * rup[j];
            yd[j] = x[j] * rdown[j];
        }
        // (the first conversion of a word keeps the upper half of its old value, which the second one overwrites: any
        // register will do as the old value)
        hi = __builtin_amdgcn_cvt_pk_fp8_f32(yu[0], yu[1], __builtin_bit_cast(int, yu[0]), false);
        hi = __builtin_amdgcn_cvt_pk_fp8_f32(yu[2], yu[3], hi, true);
        lo = __builtin_amdgcn_cvt_pk_fp8_f32(yd[0], yd[1], __builtin_bit_cast(int, yd[0]), false);
        lo = __builtin_amdgcn_cvt_pk_fp8_f32(yd[2], yd[3], lo, true);
    }
    if (__builtin_expect(!fast, 0)) return f32x4_to_e4m3fn_codes(x[0] / s[0], x[1] / s[1], x[2] / s[2], x[3] / s[3]);
    if (__builtin_expect(hi == lo, !IN_BF16)) return (uint32_t)hi;
    // The exact quotient decides: the refinement steps of the f32 division expansion without its range scaling, which the
    // limits on the scale make unnecessary (identical to the IEEE quotient on 2.9e9 CPU cases, ties of bf16-like operands
    // and reciprocals off by an ulp included).
    float q[4];
#pragma unroll
    for (int j = 0; j < 4; j++) {
        const float d = s[j];
        float r = __builtin_amdgcn_rcpf(d);
        r = __builtin_fmaf(__builtin_fmaf(-d, r, 1.0f), r, r);
        float t = x[j] * r;
        t = __builtin_fmaf(__builtin_fmaf(-d, t, x[j]), r, t);
        q[j] = __builtin_copysignf(__builtin_fmaf(__builtin_fmaf(-d, t, x[j]), r, t), x[j]);   // -0 / d stays -0
    }
    const int c = __builtin_amdgcn_cvt_pk_fp8_f32(q[0], q[1], __builtin_bit_cast(int, q[0]), false);
    return (uint32_t)__builtin_amdgcn_cvt_pk_fp8_f32(q[2], q[3], c, true);
}

// scale = amax / 448, exactly as the IEEE division gives it; 1 for a block of zeros
__device__ __forceinline__ float scale_of_amax(float a) {
    float sc = a > 0.f ? div_by_448(a) : 1.0f;
    if (__builtin_expect(a > 0.f && !(a >= 0x1p-100f && a <= 0x1.fffffep127f), 0)) sc = a / 448.0f;
    return sc;
}
// scales for which codes_of_quotients' shortcut holds
__device__ __forceinline__ bool scale_is_fast(float s) { return s > 0x1p-60f && s < 0x1p60f; }

// One workgroup (NT threads) per 128 x 128 block: rows r0.. of X (ld = K elements), K block kb.
// PER_ROW: one scale per row (activations). Otherwise one scale for the whole block (weights).
// IN_BF16: X holds bf16 instead of fp32.
// A thread loads KPT consecutive k of one row at a time (4 or 8), so a row is spread over LPR = 32 (16) neighbouring lanes; it holds RPT rows, in runs of four consecutive rows (a run becomes one 32-bit LDS store
// per k): run g of thread t starts at row g * (128 / NG) + 4 * (t / LPR).
//
// GROUPED (activations of several groups, for the grouped GEMM): the R rows written are the rows of a padded layout in
// which group g starts at row pad_start[g], a multiple of 16, and holds src_start[g+1] - src_start[g] rows of X (from
// row src_start[g]) followed by rows of zeros with scale 1 up to the next group's start. Group starts are multiples
// of 16 and a thread's rows come in runs of four from a multiple of four, so a run lies in one group.
constexpr int kQuantMaxGroups = 256;
struct QuantGroups {
    int pad_start[kQuantMaxGroups + 1];     // first row of each group in the padded layout; [groups] = R
    int src_start[kQuantMaxGroups + 1];     // first row of each group in X; [groups] = rows of X
    int groups;
    // the group that holds the first row of each 128-row block of the padded layout, for the first kQuantBlockTable
    // blocks (later blocks search the table): a search is eight dependent scalar loads, about as long as a block's work
    unsigned short block_group[512];
};
constexpr int kQuantBlockTable = 512;
template <bool PER_ROW, bool IN_BF16, bool GROUPED, int NT, int KPT>
__device__ __forceinline__ void quantize_block128_body(const void *__restrict__ X, int R, int K,
                                                       uint8_t *__restrict__ out, float *__restrict__ scales,
                                                       int scale_ld, bool vector_store, const QuantGroups &tab) {
    constexpr int LPR = 128 / KPT, W = KPT * (IN_BF16 ? 2 : 4) / 4, RPT = 128 * 128 / NT / KPT, NG = RPT / 4;
    static_assert(RPT >= 4 && RPT % 4 == 0, "whole runs of four rows");
    constexpr int PITCH = 128 + 4;                            // LDS row (one k, 128 rows of X), padded against conflicts
    __shared__ __attribute__((aligned(16))) uint8_t tile[128 * PITCH];
    __shared__ float wave_max[NT / 64];
    const int t = threadIdx.x, lane_k = t % LPR, rsub = t / LPR;
    auto row_of = [&](int i) { return (i >> 2) * (128 / NG) + 4 * rsub + (i & 3); };
    // K blocks vary fastest over the grid: workgroups that run together read neighbouring pieces of the same rows
    const int rb = blockIdx.y, r0 = rb * 128, kb = blockIdx.x, k0 = kb * 128;
    // All loads are issued before the first one is used: rows past R read row R-1 again (their results are never
    // stored, and they are kept out of a block-wide maximum below) instead of sitting behind a branch each.
    // GROUPED: source row of each run of four rows and the first padded row past its group's true rows. The groups
    // that reach into this block are found with table reads that are the same for all lanes (the block starts in
    // group g0; at most 8 more groups of at least 16 padded rows follow inside it).
    int run_shift[NG], run_limit[NG];
    if constexpr (GROUPED) {
        int lo = 0, hi = tab.groups;                          // last g with pad_start[g] <= r0 (uniform)
        if (rb < kQuantBlockTable) {
            lo = tab.block_group[rb];
        } else {
            while (hi - lo > 1) {
                const int mid = (lo + hi) >> 1;
                if (tab.pad_start[mid] <= r0) lo = mid; else hi = mid;
            }
        }
#pragma unroll
        for (int u = 0; u < NG; u++) { run_shift[u] = 0; run_limit[u] = 0; }
        for (int g = lo; g < tab.groups && tab.pad_start[g] < r0 + 128; g++) {
            const int ps = tab.pad_start[g], ss = tab.src_start[g], rows = tab.src_start[g + 1] - ss;
#pragma unroll
            for (int u = 0; u < NG; u++)
                if (r0 + row_of(4 * u) >= ps) { run_shift[u] = ss - ps; run_limit[u] = ps + rows; }
        }
    }
    const int src_rows = GROUPED ? tab.src_start[tab.groups] : R;
    uint32_t raw[RPT][W];                                     // W words per load
#pragma unroll
    for (int i = 0; i < RPT; i++) {
        const int r = r0 + row_of(i);
        int rc = r < R ? r : R - 1;
        if constexpr (GROUPED) {
            rc = r + run_shift[i >> 2];
            rc = rc < src_rows ? rc : src_rows - 1;
            rc = rc > 0 ? rc : 0;
        }
        const size_t off = (size_t)rc * K + k0 + KPT * lane_k;
        typedef uint32_t words __attribute__((ext_vector_type(W)));
        const words x = IN_BF16 ? *(const words *)((const uint16_t *)X + off) : *(const words *)((const float *)X + off);
#pragma unroll
        for (int e = 0; e < W; e++) {
            raw[i][e] = x[e];
            if constexpr (GROUPED) {
                if (r >= run_limit[i >> 2]) raw[i][e] = 0u;   // padding row: zeros, scale 1
            }
        }
    }
    float v[RPT][KPT];
#pragma unroll
    for (int i = 0; i < RPT; i++) {
        const uint32_t (&q)[W] = raw[i];
#pragma unroll
        for (int e = 0; e < W; e++) {
            if constexpr (IN_BF16) {
                v[i][2 * e] = bf16_bits_to_f32(q[e] & 0xffffu);
                v[i][2 * e + 1] = bf16_bits_to_f32(q[e] >> 16);
            } else {
                v[i][e] = __builtin_bit_cast(float, q[e]);
            }
        }
    }
    // amax: NaNs never win a comparison, like a scalar "if (|x| > amax)" loop. For everything but NaNs the order of
    // |x| is the order of its bit pattern as an unsigned integer, and NaN patterns lie above infinity: the maximum is
    // taken on the raw bits (two bf16 per instruction), and a row whose maximum lands above infinity contains a NaN
    // and takes the comparison loop instead.
    uint32_t amax_bits[RPT];
#pragma unroll
    for (int i = 0; i < RPT; i++) {
        const uint32_t (&q)[W] = raw[i];
        if constexpr (IN_BF16) {
            u16x2 m = {0, 0};
#pragma unroll
            for (int e = 0; e < W; e++) m = __builtin_elementwise_max(m, __builtin_bit_cast(u16x2, q[e] & 0x7fff7fffu));
            amax_bits[i] = (uint32_t)(m[0] > m[1] ? m[0] : m[1]) << 16;
        } else {
            uint32_t m = 0;
#pragma unroll
            for (int e = 0; e < W; e++) { const uint32_t x = q[e] & 0x7fffffffu; m = x > m ? x : m; }
            amax_bits[i] = m;
        }
    }
    max_over_16_lanes(amax_bits);                             // all 16 lanes of a row group hold it
    float amax[RPT];
    bool has_nan[RPT];
#pragma unroll
    for (int i = 0; i < RPT; i++) {
        if constexpr (LPR == 32) { const uint32_t o = __shfl_xor(amax_bits[i], 16, 64); amax_bits[i] = o > amax_bits[i] ? o : amax_bits[i]; }
        amax[i] = __builtin_bit_cast(float, amax_bits[i]);
        has_nan[i] = amax_bits[i] > 0x7f800000u;              // the same in all lanes of the row
        if (__builtin_expect(has_nan[i], 0)) {
            float a = 0.f;
#pragma unroll
            for (int e = 0; e < KPT; e++) { const float x = __builtin_fabsf(v[i][e]); a = x > a ? x : a; }
            a = max_over_16_lanes_nan_safe(a);
            if constexpr (LPR == 32) { const float o = __shfl_xor(a, 16, 64); a = o > a ? o : a; }
            amax[i] = a;
        }
    }
    float s[RPT];
    if constexpr (PER_ROW) {
#pragma unroll
        for (int i = 0; i < RPT; i++) {
            s[i] = scale_of_amax(amax[i]);
            const int r = r0 + row_of(i);
            if (lane_k == 0 && r < R) scales[(size_t)kb * scale_ld + r] = s[i];
        }
    } else {
        float a = 0.f;
#pragma unroll
        for (int i = 0; i < RPT; i++) a = (amax[i] > a && r0 + row_of(i) < R) ? amax[i] : a;
#pragma unroll
        for (int off = LPR; off < 64; off <<= 1) { const float o = __shfl_xor(a, off, 64); a = o > a ? o : a; }
        if ((t & 63) == 0) wave_max[t >> 6] = a;
        __syncthreads();
        a = wave_max[0];
#pragma unroll
        for (int w = 1; w < NT / 64; w++) a = wave_max[w] > a ? wave_max[w] : a;
        const float sb = scale_of_amax(a);
#pragma unroll
        for (int i = 0; i < RPT; i++) s[i] = sb;
        if (t == 0) scales[(size_t)kb * scale_ld + rb] = sb;
    }
    // quantise and transpose through LDS: tile[k][row]
    float rup[RPT], rdown[RPT];
    bool fast[RPT / 4];
#pragma unroll
    for (int i = 0; i < RPT; i++) {
        const float rinv = __builtin_amdgcn_rcpf(s[i]);
        rup[i] = rinv * (1.0f + 0x1p-20f);
        rdown[i] = rinv * (1.0f - 0x1p-20f);
    }
#pragma unroll
    for (int g = 0; g < NG; g++) {
        fast[g] = true;
#pragma unroll
        for (int j = 0; j < 4; j++) fast[g] = fast[g] && scale_is_fast(s[4 * g + j]) && !has_nan[4 * g + j];
    }
#pragma unroll
    for (int g = 0; g < NG; g++)
#pragma unroll
        for (int e = 0; e < KPT; e++) {
            float x[4], sc[4], up[4], down[4];
#pragma unroll
            for (int j = 0; j < 4; j++) {
                x[j] = v[4 * g + j][e];
                sc[j] = s[4 * g + j];
                up[j] = rup[4 * g + j];
                down[j] = rdown[4 * g + j];
            }
            *(uint32_t *)(tile + (KPT * lane_k + e) * PITCH + row_of(4 * g)) = codes_of_quotients<IN_BF16>(x, sc, up, down, fast[g]);
        }
    __syncthreads();
    // out[(k0 + k) * R + r0 + ..]: 128 bytes per k, 16 per thread; at any byte where R is ragged (vector stores need no
    // alignment), single bytes where a piece reaches past R
    constexpr int KPP = NT / 8;                               // k per pass
#pragma unroll
    for (int p = 0; p < 128 / KPP; p++) {
        const int k = p * KPP + (t >> 3), c = (t & 7) * 16;
        const uint32_t *src = (const uint32_t *)(tile + k * PITCH + c);
        const uint4 w = {src[0], src[1], src[2], src[3]};
        uint8_t *dst = out + (size_t)(k0 + k) * R + r0 + c;
        if (vector_store) {
            if (r0 + c < R) {
                // whole 128-byte lines (R a multiple of 128) are written through; pieces of lines are left to L2 to
                // merge (written through, the grouped layout's rows, which start at multiples of 16, took 8 % longer)
                if (!GROUPED && R % 128 == 0) store16_through(dst, w);
                else *(uint4 *)dst = w;
            }
        } else if (r0 + c + 16 <= R) {
            *(quant_u32x4_any *)dst = quant_u32x4_any{w.x, w.y, w.z, w.w};
        } else {
            const uint32_t words[4] = {w.x, w.y, w.z, w.w};
#pragma unroll
            for (int j = 0; j < 16; j++)
                if (r0 + c + j < R) dst[j] = (uint8_t)(words[j >> 2] >> (8 * (j & 3)));
        }
    }
}

// Threads per workgroup and k per thread: 16-byte loads, and as many threads as whole runs of four rows allow. The work per
// compute unit is the same for any count, but its waves then hold less of it each and overlap their neighbours' loads
// with their own arithmetic. us with 256 threads -> with these (5.1 TB/s copy rate in brackets):
//   fp32, 1024 threads: 6144 x 7168 47.7 -> 43.4 (43.2), 2048 x 2048 9.0 -> 5.9, 6001 x 7168 50.7 -> 44.9
//   bf16, 512 threads:  6144 x 7168 30.2 -> 27.8 (25.9), 2048 x 2048 6.4 -> 5.0, 6001 x 7168 32.3 -> 29.9
// (bf16 with 1024 threads and 8-byte loads: 28.2, 5.0.)
template <bool IN_BF16>
struct QuantShape {
    static constexpr int KPT = IN_BF16 ? 8 : 4, NT = 4096 / KPT;
};
template <bool PER_ROW, bool IN_BF16>
__global__ __launch_bounds__(QuantShape<IN_BF16>::NT) void quantize_block128(const void *__restrict__ X, int R, int K,
                                                                             uint8_t *__restrict__ out,
                                                                             float *__restrict__ scales, int scale_ld,
                                                                             bool vector_store) {
    QuantGroups none;                                         // not read
    quantize_block128_body<PER_ROW, IN_BF16, false, QuantShape<IN_BF16>::NT, QuantShape<IN_BF16>::KPT>(
        X, R, K, out, scales, scale_ld, vector_store, none);
}
template <bool IN_BF16>
__global__ __launch_bounds__(QuantShape<IN_BF16>::NT) void quantize_block128_grouped(const void *__restrict__ X, int R, int K,
                                                                                     uint8_t *__restrict__ out,
                                                                                     float *__restrict__ scales,
                                                                                     const QuantGroups tab) {
    quantize_block128_body<true, IN_BF16, true, QuantShape<IN_BF16>::NT, QuantShape<IN_BF16>::KPT>(X, R, K, out, scales, R, true,
                                                                                                   tab);
}

// Activations that do not fill the chip with 128 x 128 blocks: one workgroup of 256 threads per 16 rows x 128 k, eight k of
// one row per thread. A 128-row block of a handful of rows loads and encodes 128 rows and stores single bytes. us with
// 128-row blocks -> here, from bf16, on sources that rotate out of the caches (one source, which stays there, in brackets):
// 7 x 1536 4.2 -> 2.3 (the rate of back-to-back launches), 512 x 7168 5.6 -> 4.8 (4.1 -> 3.7), 2048 x 2048 6.0 -> 5.1 (4.2 ->
// 4.0). Its stores are 16-byte pieces of rows of the output, which L2 merges as long as they stay there: beyond seven to ten
// million elements the 128-row blocks are faster where they store whole lines (4096 x 2048 7.9 against 8.5 here, 1024 x 7168
// 7.5 against 8.1, 2048 x 7168 12.4 against 13.4), later where rows are ragged (1400 x 7168 11.2 against 10.7) and about as
// fast from fp32 (1024 x 7168 9.8, 9.9; 2048 x 7168 16.5, 16.7). Between one launch and the next GEMM it runs at half the copy
// rate: 2048 x 2048 is 12.6 MB, 2.5 us at 5.1 TB/s, beside 2.3 us that the shortest launch takes.
template <bool IN_BF16, bool GROUPED>
__device__ __forceinline__ void quantize_rows16_body(const void *__restrict__ X, int R, int K, uint8_t *__restrict__ out,
                                                     float *__restrict__ scales, const QuantGroups &tab, int kb, int piece) {
    constexpr int PITCH = 16 + 4;
    __shared__ __attribute__((aligned(16))) uint8_t tile[128 * PITCH];
    const int t = threadIdx.x, row = t >> 4, lane_k = t & 15;
    const int r0 = piece * 16, r = r0 + row, k0 = kb * 128;
    int from = r < R ? r : R - 1;                             // rows past R: any row, not stored
    bool padding = false;
    if constexpr (GROUPED) {                                  // group starts are multiples of 16: one group per workgroup
        int lo = 0, hi = tab.groups;                          // last g with pad_start[g] <= r0 (uniform)
        while (hi - lo > 1) {
            const int mid = (lo + hi) >> 1;
            if (tab.pad_start[mid] <= r0) lo = mid; else hi = mid;
        }
        from = r - tab.pad_start[lo] + tab.src_start[lo];
        padding = from >= tab.src_start[lo + 1];
        if (padding) from = tab.src_start[lo + 1] - 1;        // the group has rows, or no padded row would be in it
    }
    const size_t off = (size_t)from * K + k0 + 8 * lane_k;
    uint32_t q[8];
    if constexpr (IN_BF16) {
        const uint4 a = *(const uint4 *)((const uint16_t *)X + off);
        const uint32_t h[4] = {a.x, a.y, a.z, a.w};
#pragma unroll
        for (int e = 0; e < 4; e++) {
            q[2 * e] = h[e] << 16;
            q[2 * e + 1] = h[e] & 0xffff0000u;
        }
    } else {
        const uint4 a = *(const uint4 *)((const float *)X + off), b = *(const uint4 *)((const float *)X + off + 4);
        q[0] = a.x; q[1] = a.y; q[2] = a.z; q[3] = a.w; q[4] = b.x; q[5] = b.y; q[6] = b.z; q[7] = b.w;
    }
    uint32_t m[1] = {0};
    float v[8];
#pragma unroll
    for (int e = 0; e < 8; e++) {
        if (GROUPED && padding) q[e] = 0u;
        v[e] = __builtin_bit_cast(float, q[e]);
        const uint32_t x = q[e] & 0x7fffffffu;
        m[0] = x > m[0] ? x : m[0];
    }
    max_over_16_lanes(m);                                     // on bit patterns, NaNs above infinity (see above)
    float amax = __builtin_bit_cast(float, m[0]);
    const bool has_nan = m[0] > 0x7f800000u;
    if (__builtin_expect(has_nan, 0)) {
        amax = 0.f;
#pragma unroll
        for (int e = 0; e < 8; e++) { const float x = __builtin_fabsf(v[e]); amax = x > amax ? x : amax; }
        amax = max_over_16_lanes_nan_safe(amax);
    }
    const float s = scale_of_amax(amax), rinv = __builtin_amdgcn_rcpf(s);
    const float up = rinv * (1.0f + 0x1p-20f), down = rinv * (1.0f - 0x1p-20f);
    const bool fast = scale_is_fast(s) && !has_nan;
    if (lane_k == 0 && r < R) scales[(size_t)kb * R + r] = s;
#pragma unroll
    for (int h = 0; h < 2; h++) {
        const uint32_t w = codes_of_quotients<IN_BF16>({v[4 * h], v[4 * h + 1], v[4 * h + 2], v[4 * h + 3]}, {s, s, s, s},
                                                       {up, up, up, up}, {down, down, down, down}, fast);
#pragma unroll
        for (int e = 0; e < 4; e++) tile[(8 * lane_k + 4 * h + e) * PITCH + row] = (uint8_t)(w >> (8 * e));
    }
    __syncthreads();
    if (R < 16) {
        // the K block of the output is 128 * R consecutive bytes
        for (int f = 4 * t; f < 128 * R; f += 1024) {
            uint32_t w = 0;
#pragma unroll
            for (int e = 0; e < 4; e++) w |= (uint32_t)tile[(f + e) / R * PITCH + (f + e) % R] << (8 * e);
            *(quant_u32_any *)(out + (size_t)k0 * R + f) = w;
        }
    } else if (t < 128) {
        const uint32_t *src = (const uint32_t *)(tile + t * PITCH);
        uint8_t *dst = out + (size_t)(k0 + t) * R + r0;
        const uint32_t words[4] = {src[0], src[1], src[2], src[3]};
        if (r0 + 16 <= R) {
            *(quant_u32x4_any *)dst = quant_u32x4_any{words[0], words[1], words[2], words[3]};
        } else {
#pragma unroll
            for (int j = 0; j < 16; j++)
                if (r0 + j < R) dst[j] = (uint8_t)(words[j >> 2] >> (8 * (j & 3)));
        }
    }
}
// DEALT: eight pieces, 128 rows of a K block, at a time to every XCD (grid: 64 workgroups for eight such units), so that a
// line of the output is written by one L2. In the plain order that is so where the number of K blocks is a multiple of
// eight; where it is not, eight L2s held parts of each line and wrote them one by one: 3001 x 2304 11.9 -> 8.6 us, 6000 x 1536
// 10.7 -> 10.0. (Where it is, the plain order is the faster one: 4096 x 2048 7.8, dealt 8.1.)
template <bool IN_BF16, bool DEALT>
__global__ __launch_bounds__(256) void quantize_rows16(const void *__restrict__ X, int R, int K, uint8_t *__restrict__ out,
                                                       float *__restrict__ scales) {
    QuantGroups none;                                         // not read
    int kb = blockIdx.x, piece = blockIdx.y;
    if constexpr (DEALT) {
        const int xcd = blockIdx.x % NUM_XCD, j = blockIdx.x / NUM_XCD, unit = j / 8 * NUM_XCD + xcd, blocks = K / BK;
        kb = unit % blocks;
        piece = unit / blocks * 8 + j % 8;
        if (piece * 16 >= R) return;
    }
    quantize_rows16_body<IN_BF16, false>(X, R, K, out, scales, none, kb, piece);
}
template <bool IN_BF16>
__global__ __launch_bounds__(256) void quantize_rows16_grouped(const void *__restrict__ X, int R, int K, uint8_t *__restrict__ out,
                                                               float *__restrict__ scales, const QuantGroups tab) {
    quantize_rows16_body<IN_BF16, true>(X, R, K, out, scales, tab, blockIdx.x, blockIdx.y);
}

}  // namespace rf

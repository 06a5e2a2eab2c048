// Host side of libgemm.so: the C ABI declared in include/rf_gemm.h.
//
// Takes the place of the reference's launcher (src/gemm/gemm_launcher.cpp): `run` keeps its
// signature and abort-on-error behaviour; dispatch is shape-generic (a heuristic over a small
// variant table tuned for gfx950) instead of a switch over 29 hard-coded shapes, and no transpose
// pre-pass or transposed copies exist.
#include <hip/hip_runtime.h>
#include <algorithm>
#include <cmath>

#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <mutex>
#include <string>
#include <vector>

#include "../../include/rf_gemm.h"
#include "fp8_gemm_kernels.h"
#include "fp8_gemm_persistent.h"
#include "fp8_gemm_skinny.h"
#include "fp8_gemm_fewrows.h"
#include "fp8_gemm_any.h"
#include "grown_buffer.h"
#include "plan_limits.h"
#include "quantize_kernels.h"

// Scratch memory of rf_fp8_gemm_static, the entry point that allocates nothing: split-K partial sums and staging
// copies live here instead of in buffers from hipMalloc. Every device the library runs on holds its own copy at its
// own address until the process ends; host code never uses this name as an address (see ensure_device_info).
constexpr size_t kStaticScratchBytes = (size_t)32 << 20;
static __device__ __align__(256) uint8_t scratch[kStaticScratchBytes];
// Counters of a launch: arrivals at tiles that several workgroups finish (few-rows kernels with a K split, stream-K), and
// the draws from the grouped GEMM's queues, in words of their own. One set per buffer set (StreamBuffers) and one for
// rf_fp8_gemm_static. They are zero when the library is loaded, and every launch that uses them leaves them at zero: nothing
// is allocated or cleared on the way to a launch, also not under graph capture (a counter buffer allocated and zeroed by the
// first launch that ran eagerly put a kernel of 16384 words in front of every captured one).
constexpr int kMaxTileCounters = 16384, kQueueCounters = 64;
constexpr int kMaxStreamBuffers = 32;    // per device; one more stream takes over the least recently used set
struct CounterSet {
    unsigned tile[kMaxTileCounters], queue[kQueueCounters];
};
static_assert(rf::NUM_XCD <= kQueueCounters, "a counter per queue");
static __device__ CounterSet counter_sets[kMaxStreamBuffers + 1];

namespace {

thread_local std::string g_last_error;

// A launch without the trip through the call configuration that the <<<>>> form makes (push, stub, pop): 0.10 us of host time less, medians
// of 600 times 100 calls of either in turn (an rf_fp8_gemm of 7 x 3072 x 1536 4.24 -> 4.14 us with its caller's 1 us; quantize_a and that
// GEMM in a loop, which runs at its host time, 7.99 -> 7.78). Failures are left to hipGetLastError, as with that form.
template <typename... P, typename... A>
void enqueue(void (*kernel)(P...), dim3 grid, dim3 block, size_t lds, hipStream_t stream, A... args) {
    [&](P... p) {
        void *values[] = {(void *)&p...};
        (void)hipLaunchKernel((const void *)kernel, grid, block, values, lds, stream);
    }(args...);
}

int fail(int code, const std::string &msg) {
    g_last_error = msg;
    return code;
}
#define RF_HIP(expr)                                                                                   \
    do {                                                                                               \
        hipError_t e_ = (expr);                                                                        \
        if (e_ != hipSuccess)                                                                          \
            return fail(RF_ERR_HIP, std::string(#expr) + ": " + hipGetErrorString(e_));               \
    } while (0)

// ---- variant table -------------------------------------------------------------------------
typedef void (*tile_kernel_t)(const uint8_t *, const uint8_t *, const float *, const float *, void *, int, int, int,
                              int, int, int, int, int);
typedef void (*streamk_kernel_t)(const uint8_t *, const uint8_t *, const float *, const float *, uint16_t *, int, int,
                                 int, int, int, int, unsigned *, float *);
typedef void (*persistent_kernel_t)(const uint8_t *, const uint8_t *, const float *, const float *, uint16_t *, int, int,
                                    int, int, int, int, int);
typedef void (*fewrows_kernel_t)(const uint8_t *, const uint8_t *, const float *, const float *, uint16_t *, int, int, int,
                                 int, int, int, unsigned *, float *);
typedef void (*any_c_kernel_t)(const uint8_t *, const uint8_t *, const float *, const float *, uint16_t *, int, int, int, int,
                               int, int, int, int);
typedef void (*any_tile_kernel_t)(const uint8_t *, const uint8_t *, const float *, const float *, void *, int, int, int, int, int, int,
                                  int, int);
struct Variant {
    int bm, bn, waves_m, waves_n, lds;
    tile_kernel_t direct, partial;
    streamk_kernel_t streamk;            // null: the variant has no stream-K form
    persistent_kernel_t persistent;      // null: no persistent form
    int lds_persistent;
    persistent_kernel_t persistent_half_tail = nullptr;   // null: no form that ends with half tiles
    int k_groups = 1;                    // > 1: wave groups of one workgroup split K between them (needs K/128 % k_groups == 0)
    fewrows_kernel_t fewrows[2][2] = {{nullptr, nullptr}, {nullptr, nullptr}};   // [K split][any alignment of B]; null: a tiled variant
    any_c_kernel_t any_c = nullptr;      // the direct form for a C of any width and alignment
    any_tile_kernel_t any_tile[2] = {nullptr, nullptr};   // [K split]: operands at any alignment (fp8_gemm_any.h)
    bool is_fewrows() const { return fewrows[0][0] != nullptr; }
    bool is_any_tile() const { return any_tile[0] != nullptr; }
    bool takes_any_shape() const { return is_fewrows() || is_any_tile(); }
    int lds_bytes() const { return lds; }
    int threads() const { return waves_m * waves_n * 64 * k_groups; }
};
#define RF_ANY_C(BM, BN, WM, WN, NS) nullptr, 1, {}, rf::gemm_fp8_blockscale_tile_any_c<BM, BN, WM, WN, NS>
#define RF_VARIANT(BM, BN, WM, WN)                                                         \
    Variant { BM, BN, WM, WN, rf::TileGeom<BM, BN, WM, WN>::LDS_BYTES,                     \
              rf::gemm_fp8_blockscale_tile<BM, BN, WM, WN, false>,                         \
              rf::gemm_fp8_blockscale_tile<BM, BN, WM, WN, true>,                          \
              rf::gemm_fp8_blockscale_streamk<BM, BN, WM, WN>,                             \
              rf::gemm_fp8_blockscale_persistent<BM, BN, WM, WN>,                          \
              rf::PersistentGeom<BM, BN, WM, WN>::LDS_BYTES, RF_ANY_C(BM, BN, WM, WN, 2) }
// tiles with sides that are not powers of two, same inner loop: one workgroup per tile only
#define RF_VARIANT_TILE_ONLY(BM, BN, WM, WN)                                               \
    Variant { BM, BN, WM, WN, rf::TileGeom<BM, BN, WM, WN>::LDS_BYTES,                     \
              rf::gemm_fp8_blockscale_tile<BM, BN, WM, WN, false>,                         \
              rf::gemm_fp8_blockscale_tile<BM, BN, WM, WN, true>, nullptr, nullptr, 0, RF_ANY_C(BM, BN, WM, WN, 2) }
// the same with three LDS stages: two K blocks in flight instead of one. A K block of these tiles is 0.4 us of MFMAs,
// less than a load takes to come back from L2 or the Infinity Cache on a busy chip, so with two stages the loop ran at
// the latency of its loads: 1024 x 4608 x 7168 45.6 -> 39.0 us, 256 x 7168 x 2304 15.6 -> 13.1 us; the plan of 21
// of the 163 tabled shapes, and variant 28 of 37. The two-stage forms stay: they fit more workgroups per CU (64 x 128: three instead of
// two), which the smallest problems prefer. (128 x 128 with four waves and three stages never won; with eight it is variant 28.)
#define RF_VARIANT_TILE_ONLY_NS3(BM, BN, WM, WN)                                           \
    Variant { BM, BN, WM, WN, rf::TileGeom<BM, BN, WM, WN, 3>::LDS_BYTES,                  \
              rf::gemm_fp8_blockscale_tile<BM, BN, WM, WN, false, 3>,                      \
              rf::gemm_fp8_blockscale_tile<BM, BN, WM, WN, true, 3>, nullptr, nullptr, 0, RF_ANY_C(BM, BN, WM, WN, 3) }
// few-rows kernels (fp8_gemm_fewrows.h): any shape, any alignment, K splits reduced inside the launch
#define RF_VARIANT_FEWROWS(TM, TN, NW, DEPTH)                                              \
    Variant { 16 * TM, 16 * TN, 1, NW, rf::FewRowsGeom<TM, TN, NW, DEPTH>::LDS_BYTES,      \
              nullptr, nullptr, nullptr, nullptr, 0, nullptr, 1,                           \
              {{rf::gemm_fp8_blockscale_fewrows<TM, TN, NW, DEPTH, false, false>,          \
                rf::gemm_fp8_blockscale_fewrows<TM, TN, NW, DEPTH, false, true>},          \
               {rf::gemm_fp8_blockscale_fewrows<TM, TN, NW, DEPTH, true, false>,           \
                rf::gemm_fp8_blockscale_fewrows<TM, TN, NW, DEPTH, true, true>}} }
// tiles whose operands pass through registers, at any alignment (fp8_gemm_any.h)
#define RF_VARIANT_ANY_TILE(BM, BN, WM, WN)                                                \
    Variant { BM, BN, WM, WN, rf::AnyGeom<BM, BN, WM, WN>::LDS_BYTES, nullptr, nullptr, nullptr, nullptr, 0, nullptr, 1, {}, nullptr, \
              {rf::gemm_fp8_blockscale_tile_any<BM, BN, WM, WN, false>, rf::gemm_fp8_blockscale_tile_any<BM, BN, WM, WN, true>} }
const Variant kVariants[] = {
    Variant{256, 256, 2, 4, rf::TileGeom<256, 256, 2, 4>::LDS_BYTES, rf::gemm_fp8_blockscale_tile<256, 256, 2, 4, false>,
            rf::gemm_fp8_blockscale_tile<256, 256, 2, 4, true>, rf::gemm_fp8_blockscale_streamk<256, 256, 2, 4>,
            rf::gemm_fp8_blockscale_persistent<256, 256, 2, 4>, rf::PersistentGeom<256, 256, 2, 4>::LDS_BYTES,
            rf::gemm_fp8_blockscale_persistent<256, 256, 2, 4, true>, 1, {},
            rf::gemm_fp8_blockscale_tile_any_c<256, 256, 2, 4, 2>},   // 0: 8 waves, wave tile 128(m) x 64(n), 128 KiB LDS
    RF_VARIANT(128, 128, 2, 2),   // 1: 4 waves, wave tile 64 x 64, 64 KiB LDS (2 workgroups per CU)
    RF_VARIANT(256, 128, 2, 2),   // 2: 4 waves, wave tile 128 x 64, 96 KiB LDS
    RF_VARIANT(128, 256, 2, 4),   // 3: 8 waves, wave tile 64 x 64, 96 KiB LDS
    RF_VARIANT(128, 64, 2, 1),    // 4: 2 waves, wave tile 64 x 64, 48 KiB LDS (3 workgroups per CU)
    RF_VARIANT_TILE_ONLY(192, 192, 2, 4),   // 5: 8 waves, wave tile 96 x 48, 98 KiB LDS (6144 x 4608 = 768 tiles = 3 x 256)
    RF_VARIANT_TILE_ONLY(128, 192, 2, 4),   // 6: 8 waves, wave tile 64 x 48, 82 KiB LDS (N = 576, 1536: no padded columns)
    RF_VARIANT_TILE_ONLY(64, 128, 2, 2),    // 7: 4 waves, wave tile 32 x 64, 49 KiB LDS (3 workgroups per CU; short M)
    RF_VARIANT_TILE_ONLY_NS3(128, 192, 2, 4),   // 8: variant 6 with three stages, 123 KiB LDS
    RF_VARIANT_TILE_ONLY_NS3(64, 128, 2, 2),    // 9: variant 7 with three stages, 74 KiB LDS (2 workgroups per CU)
    RF_VARIANT_TILE_ONLY_NS3(128, 256, 2, 4),   // 10: variant 3 with three stages, 149 KiB LDS
    RF_VARIANT_TILE_ONLY_NS3(192, 192, 2, 4),   // 11: variant 5 with three stages, 147 KiB LDS
    // 12: the 64 x 128 three-stage tile with K split between two wave groups of one workgroup (8 waves, 150 KiB LDS):
    // the split-K plan of a short, wide-K shape in one launch, with no partial sums in memory
    Variant{64, 128, 2, 2, rf::InWgSplitGeom<64, 128, 2, 2, 3, 2>::LDS_BYTES,
            rf::gemm_fp8_blockscale_tile_ksplit_in_wg<64, 128, 2, 2, 3, 2>, nullptr, nullptr, nullptr, 0, nullptr, 2},
    // 13: the 128 x 128 two-stage tile with K split between two wave groups (8 waves, 130 KiB LDS)
    Variant{128, 128, 2, 2, rf::InWgSplitGeom<128, 128, 2, 2, 2, 2>::LDS_BYTES,
            rf::gemm_fp8_blockscale_tile_ksplit_in_wg<128, 128, 2, 2, 2, 2>, nullptr, nullptr, nullptr, 0, nullptr, 2},
    RF_VARIANT_FEWROWS(1, 2, 8, 3),   // 14: 16 rows x 32 columns
    RF_VARIANT_FEWROWS(1, 4, 8, 2),   // 15: 16 x 64
    RF_VARIANT_FEWROWS(1, 8, 8, 1),   // 16: 16 x 128
    RF_VARIANT_FEWROWS(2, 2, 8, 2),   // 17: 32 x 32
    RF_VARIANT_FEWROWS(2, 4, 8, 2),   // 18: 32 x 64
    RF_VARIANT_FEWROWS(4, 2, 8, 2),   // 19: 64 x 32
    RF_VARIANT_FEWROWS(4, 4, 8, 1),   // 20: 64 x 64
    RF_VARIANT_FEWROWS(4, 4, 4, 1),   // 21: 64 x 64, four waves: two workgroups per CU (200 x 5003 x 2048, 316 workgroups:
                                      // one round of the chip instead of two, 23.2 -> 19.8 us)
    // tiles of which a wave has one K block on its way while it multiplies another (16, 20 and 21 above work like that too)
    RF_VARIANT_FEWROWS(1, 2, 8, 1),   // 22: 16 x 32
    RF_VARIANT_FEWROWS(1, 4, 8, 1),   // 23: 16 x 64
    RF_VARIANT_FEWROWS(2, 2, 8, 1),   // 24: 32 x 32
    RF_VARIANT_FEWROWS(2, 4, 8, 1),   // 25: 32 x 64
    RF_VARIANT_FEWROWS(2, 4, 4, 1),   // 26: 32 x 64, four waves
    RF_VARIANT_FEWROWS(2, 8, 4, 1),   // 27: 32 x 128, four waves
    // 28: 8 waves, wave tile 32 x 64, three stages, 100 KiB LDS. At a wave per SIMD the reads of fragments, the barrier and the
    // loads of a K block wait for each other; with two they hide. us, variant 1 (four waves, two stages), the best plan before,
    // this: 512 x 7168 x 2048 15.1, 14.1, 11.7; 1024 x 1536 x 7168 23.9, 23.2, 22.3; 2048 x 1536 x 7168 35.3, 32.6, 29.1. The plan of 37
    // of the 163 tabled shapes, 10 % faster there. (Four stages: the same within 2 %. Sixteen waves on 128 x 256 tiles: 49 against
    // 44 with eight on 1024 x 4608 x 7168.)
    RF_VARIANT_TILE_ONLY_NS3(128, 128, 4, 2),
    RF_VARIANT_ANY_TILE(128, 128, 4, 2),   // 29: 8 waves, wave tile 32 x 64
    RF_VARIANT_ANY_TILE(128, 256, 2, 4),   // 30: 8 waves, wave tile 64 x 64
};
constexpr int kFewRows64x64 = 20, kFirstFewRows = 14, kAnyTile128 = 29;
constexpr int kNumVariants = sizeof(kVariants) / sizeof(kVariants[0]);

// ---- process-wide state ---------------------------------------------------------------------
struct TunedPlan {
    int m, n, k, variant, split_k, group_m, stream_k;
};

// Buffers, counters and kernel attributes belong to a device: one State per device, chosen by the device that is
// current at the call. Plans and the lock are shared by the process.
//
// Temporary device memory (split-K partial sums, stream-K slots, staging copies of ragged operands) is
// kept per (device, stream): two launches on different streams of one device never share a buffer, so they may overlap,
// and launches on one stream are ordered by the stream. A buffer that has to grow is replaced, and the old one is kept
// until rf_gemm_destroy: work enqueued earlier may still use it, and waiting for that work here would block the host
// (and, with a timing callback of run() pending, deadlock against it).
struct StreamBuffers {
    hipStream_t stream = nullptr;
    uint8_t *pad = nullptr;              // staging for shapes the tiled kernels do not take as they are (see launch_padded)
    size_t pad_bytes = 0;
    float *ws = nullptr;                 // split-K partial sums / stream-K slots
    size_t ws_bytes = 0;
    rf::RefusedGrowth ws_refused;
    uint64_t last_use = 0;
};
struct State {
    std::vector<StreamBuffers> buffers;  // set i has counters[i]
    std::vector<void *> retired;         // outgrown buffers, freed by rf_gemm_destroy
    uint64_t tick = 0;
    bool attrs_set = false, grouped_attrs_set = false;
    int num_cu = 0;
    CounterSet *counters = nullptr;      // this device's copy of counter_sets, the last one for rf_fp8_gemm_static
    uint8_t *static_scratch = nullptr;   // this device's copy of the file-scope scratch array (rf_fp8_gemm_static)
    std::mutex ev_mu;                    // guards free_events only: the timing callback takes no other lock
    std::vector<std::pair<hipEvent_t, hipEvent_t>> free_events;
};
struct Shared {
    std::mutex mu;
    std::vector<TunedPlan> user_plans;   // rf_gemm_load_plans / RF_GEMM_PLANS: looked up before the built-in table
    int plan_generation = 0;             // counts changes of user_plans
    bool env_plans_checked = false;
};
constexpr int kMaxDevices = 64;
Shared &shared() {
    static Shared s;
    return s;
}
State &state() {
    static State states[kMaxDevices];
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= kMaxDevices) dev = 0;
    return states[dev];
}

// Plan file: one plan per line, "M N K variant split_k group_m stream_k"; braces and commas count as blanks (so a
// tuned_plans.inc written by the tuner is a plan file too), '#' and "//" start a comment. Appends to `out`.
int parse_plans(const char *path, std::vector<TunedPlan> &out) {
    FILE *f = fopen(path, "r");
    if (!f) return fail(RF_ERR_BAD_CONFIG, std::string("cannot open plan file ") + path);
    char line[512];
    int lineno = 0;
    std::vector<TunedPlan> plans;
    while (fgets(line, sizeof line, f)) {
        lineno++;
        if (char *c = strstr(line, "//")) *c = 0;
        if (char *c = strchr(line, '#')) *c = 0;
        for (char *c = line; *c; c++)
            if (*c == '{' || *c == '}' || *c == ',') *c = ' ';
        TunedPlan p;
        char extra;
        const int got = sscanf(line, " %d %d %d %d %d %d %d %c", &p.m, &p.n, &p.k, &p.variant, &p.split_k, &p.group_m,
                               &p.stream_k, &extra);
        if (got <= 0) continue;                       // blank or comment line
        if (got != 7 || p.m < 1 || p.n < 1 || p.k < rf::BK || p.k % rf::BK != 0 || p.variant < 0 ||
            p.variant >= kNumVariants || p.split_k < 1 || p.group_m < 1 || p.stream_k < RF_SCHEDULE_TILES ||
            p.stream_k > RF_SCHEDULE_SKINNY_K || (p.stream_k != RF_SCHEDULE_TILES && p.split_k != 1)) {
            fclose(f);
            return fail(RF_ERR_BAD_CONFIG, std::string(path) + ":" + std::to_string(lineno) +
                                               ": expected \"M N K variant split_k group_m stream_k\" with valid values");
        }
        plans.push_back(p);
    }
    fclose(f);
    out.insert(out.end(), plans.begin(), plans.end());
    return RF_OK;
}

int ensure_device_info(State &s) {
    if (s.attrs_set) return RF_OK;
    if (!shared().env_plans_checked) {
        // a file named by RF_GEMM_PLANS is loaded once, before the first plan is chosen; a bad file is an error
        if (const char *path = getenv("RF_GEMM_PLANS")) {
            int rc = parse_plans(path, shared().user_plans);
            if (rc != RF_OK) return rc;
            shared().plan_generation++;
        }
        shared().env_plans_checked = true;
    }
    int dev = 0;
    RF_HIP(hipGetDevice(&dev));
    hipDeviceProp_t prop;
    RF_HIP(hipGetDeviceProperties(&prop, dev));
    if (strncmp(prop.gcnArchName, "gfx950", 6) != 0)
        return fail(RF_ERR_HIP, std::string("libgemm.so is built for gfx950 only, device is ") + prop.gcnArchName);
    s.num_cu = prop.multiProcessorCount;
    for (const Variant &v : kVariants) {
        for (auto &pair : v.fewrows)
            for (fewrows_kernel_t f : pair)
                if (f) RF_HIP(hipFuncSetAttribute((const void *)f, hipFuncAttributeMaxDynamicSharedMemorySize, v.lds_bytes()));
        for (any_tile_kernel_t f : v.any_tile)
            if (f) RF_HIP(hipFuncSetAttribute((const void *)f, hipFuncAttributeMaxDynamicSharedMemorySize, v.lds_bytes()));
        if (v.direct)
            RF_HIP(hipFuncSetAttribute((const void *)v.direct, hipFuncAttributeMaxDynamicSharedMemorySize, v.lds_bytes()));
        if (v.any_c)
            RF_HIP(hipFuncSetAttribute((const void *)v.any_c, hipFuncAttributeMaxDynamicSharedMemorySize, v.lds_bytes()));
        if (v.partial)
            RF_HIP(hipFuncSetAttribute((const void *)v.partial, hipFuncAttributeMaxDynamicSharedMemorySize, v.lds_bytes()));
        if (v.streamk)
            RF_HIP(hipFuncSetAttribute((const void *)v.streamk, hipFuncAttributeMaxDynamicSharedMemorySize, v.lds_bytes()));
        if (v.persistent)
            RF_HIP(hipFuncSetAttribute((const void *)v.persistent, hipFuncAttributeMaxDynamicSharedMemorySize,
                                       v.lds_persistent));
        if (v.persistent_half_tail)
            RF_HIP(hipFuncSetAttribute((const void *)v.persistent_half_tail, hipFuncAttributeMaxDynamicSharedMemorySize,
                                       v.lds_persistent));
    }
    RF_HIP(hipFuncSetAttribute((const void *)rf::gemm_fp8_blockscale_skinny<1>, hipFuncAttributeMaxDynamicSharedMemorySize,
                               rf::SkinnyGeom<1>::LDS_BYTES));
    RF_HIP(hipFuncSetAttribute((const void *)rf::gemm_fp8_blockscale_skinny<2>, hipFuncAttributeMaxDynamicSharedMemorySize,
                               rf::SkinnyGeom<2>::LDS_BYTES));
    RF_HIP(hipFuncSetAttribute((const void *)rf::gemm_fp8_blockscale_skinny<3>, hipFuncAttributeMaxDynamicSharedMemorySize,
                               rf::SkinnyGeom<3>::LDS_BYTES));
    RF_HIP(hipFuncSetAttribute((const void *)rf::gemm_fp8_blockscale_skinny<4>, hipFuncAttributeMaxDynamicSharedMemorySize,
                               rf::SkinnyGeom<4>::LDS_BYTES));
    // the device address of this device's copy of the scratch array (the array's name is only a host-side handle)
    void *scratch_ptr = nullptr;
    RF_HIP(hipGetSymbolAddress(&scratch_ptr, HIP_SYMBOL(scratch)));
    s.static_scratch = (uint8_t *)scratch_ptr;
    RF_HIP(hipGetSymbolAddress(&scratch_ptr, HIP_SYMBOL(counter_sets)));
    s.counters = (CounterSet *)scratch_ptr;
    s.attrs_set = true;
    return RF_OK;
}

// hipMalloc that also works while the calling thread records a stream into a HIP graph: an allocation is not part
// of the recorded work, so the capture mode is relaxed around it (under the default mode the call would fail and
// invalidate the capture).
hipError_t device_malloc(void **p, size_t bytes) {
    hipStreamCaptureMode mode = hipStreamCaptureModeRelaxed;
    hipError_t e = hipThreadExchangeStreamCaptureMode(&mode);
    if (e != hipSuccess) return e;
    e = hipMalloc(p, bytes);
    (void)hipThreadExchangeStreamCaptureMode(&mode);
    return e;
}

// Where a launch finds its temporary device memory: the growable buffers of its (device, stream), or, for
// rf_fp8_gemm_static, consecutive pieces of the device's static scratch array (nothing is allocated; a launch that
// needs more than the array holds fails).
int buffers_of(State &s, hipStream_t stream, StreamBuffers **out);
struct Mem {
    State &s;
    StreamBuffers *sb = nullptr;         // growable buffers of `stream`, bound at the first use (never in static mode)
    uint8_t *fixed = nullptr;            // static mode: this device's scratch array
    size_t fixed_used = 0;
    hipStream_t stream = nullptr;
    // Most launches need no temporary memory at all (one kernel, no K split, no staging): the stream's buffer set is
    // looked up, and past kMaxStreamBuffers streams taken over from another stream, only when a buffer is asked for.
    int bind() { return sb ? RF_OK : buffers_of(s, stream, &sb); }

    template <typename T>
    int grow(T *&buf, size_t &have, size_t need) {
        // the old buffer may still be read by launches enqueued earlier: it is kept until rf_gemm_destroy
        RF_HIP(rf::grow_buffer(buf, have, need, s.retired, device_malloc));
        return RF_OK;
    }
    int take_fixed(size_t bytes, void **out, const char *what) {
        const size_t at = (fixed_used + 255) / 256 * 256;
        if (at + bytes > kStaticScratchBytes)
            return fail(RF_ERR_BAD_CONFIG, std::string("rf_fp8_gemm_static: this shape needs ") + std::to_string(at + bytes) +
                                               " bytes of scratch memory (" + what + "), the static array holds " +
                                               std::to_string(kStaticScratchBytes));
        *out = fixed + at;
        fixed_used = at + bytes;
        return RF_OK;
    }
    // bytes the static array still has to give (after rounding the next piece up to 256)
    size_t fixed_left() const {
        const size_t at = (fixed_used + 255) / 256 * 256;
        return at < kStaticScratchBytes ? kStaticScratchBytes - at : 0;
    }
    int pad(size_t bytes, uint8_t **out) {
        if (fixed) return take_fixed(bytes, (void **)out, "staging copy of ragged or unaligned operands");
        int rc = bind();
        if (rc != RF_OK) return rc;
        rc = grow(sb->pad, sb->pad_bytes, bytes);
        *out = sb->pad;
        return rc;
    }
    int workspace(size_t bytes, float **out) {
        if (fixed) return take_fixed(bytes, (void **)out, "split-K partial sums");
        int rc = bind();
        if (rc != RF_OK) return rc;
        rc = grow(sb->ws, sb->ws_bytes, bytes);
        *out = sb->ws;
        return rc;
    }
    // Whether there is a workspace of that size, for a plan that another can take the place of (not for the static mode).
    bool try_workspace(size_t bytes) {
        float *ws = nullptr;
        int rc = bind();
        if (rc == RF_OK) {
            if (bytes <= sb->ws_bytes) return true;
            if (!sb->ws_refused.ask(bytes)) return false;
            rc = workspace(bytes, &ws);
            sb->ws_refused.answer(bytes, rc == RF_OK);
        }
        if (rc == RF_OK) return true;
        (void)hipGetLastError();
        g_last_error.clear();
        return false;
    }
    int counters(CounterSet **out) {
        if (fixed) {
            *out = s.counters + kMaxStreamBuffers;
            return RF_OK;
        }
        int rc = bind();
        if (rc != RF_OK) return rc;
        *out = s.counters + (sb - s.buffers.data());
        return RF_OK;
    }
};

// The buffer set of (current device, stream); the caller holds the lock. A set prepared by rf_gemm_init and not yet
// bound to a stream is taken first. Past kMaxStreamBuffers streams the least recently used set changes hands: the new
// stream is made to wait (on the device, through an event) for what the old stream has enqueued so far, so the host
// does not wait. A stream that is being captured into a graph cannot take a set over (the wait would become part of
// the graph, and the old stream's later work would not be ordered against the graph's replays): RF_ERR_BAD_CONFIG.
constexpr uintptr_t kUnboundStream = 1;  // not a valid stream handle
int buffers_of(State &s, hipStream_t stream, StreamBuffers **out) {
    StreamBuffers *unbound = nullptr, *lru = nullptr;
    for (StreamBuffers &b : s.buffers) {
        if (b.stream == stream) {
            b.last_use = ++s.tick;
            *out = &b;
            return RF_OK;
        }
        if ((uintptr_t)b.stream == kUnboundStream) unbound = &b;
        if (!lru || b.last_use < lru->last_use) lru = &b;
    }
    StreamBuffers *b = unbound;
    if (!b && (int)s.buffers.size() < kMaxStreamBuffers) {
        if (s.buffers.capacity() < (size_t)kMaxStreamBuffers) s.buffers.reserve(kMaxStreamBuffers);
        s.buffers.emplace_back();
        b = &s.buffers.back();
    }
    if (!b) {
        hipStreamCaptureStatus st = hipStreamCaptureStatusNone;
        const hipError_t qe = hipStreamIsCapturing(stream, &st);
        if (qe != hipSuccess || st != hipStreamCaptureStatusNone) {
            if (qe != hipSuccess) (void)hipGetLastError();
            return fail(RF_ERR_BAD_CONFIG, "more than " + std::to_string(kMaxStreamBuffers) + " streams have used temporary "
                        "device memory on this device, and a stream that is being captured cannot take over another "
                        "stream's buffers: use rf_fp8_gemm_static under capture, or fewer streams");
        }
        hipEvent_t ev = nullptr;
        RF_HIP(hipEventCreateWithFlags(&ev, hipEventDisableTiming));
        hipError_t e = hipEventRecord(ev, lru->stream);
        if (e == hipSuccess) e = hipStreamWaitEvent(stream, ev, 0);
        (void)hipEventDestroy(ev);                               // released once the wait has been satisfied
        if (e != hipSuccess) {
            // the old stream no longer exists (or is being captured): wait for the device instead
            (void)hipGetLastError();
            RF_HIP(hipDeviceSynchronize());
        }
        b = lru;
    }
    b->stream = stream;
    b->last_use = ++s.tick;
    *out = b;
    return RF_OK;
}

inline int ceil_div(int a, int b) { return (a + b - 1) / b; }

struct Variant;
bool persistent_ok(const Variant &v, int m, int n, int k);

bool tiled_path_ok(const void *a, const void *b, const void *c, int m, int n) {
    return m >= 16 && n >= 16 && m % 16 == 0 && n % 16 == 0 && ((uintptr_t)a % 16) == 0 && ((uintptr_t)b % 16) == 0 &&
           ((uintptr_t)c % 16) == 0;
}

bool persistent_ok(const Variant &v, int m, int n, int k) {
    return v.persistent && m >= v.bm && m % 16 == 0 && n % v.bn == 0 && (k / rf::BK) % 2 == 0 && rf::persistent_offsets_fit(m, n, k);
}

// Persistent schedule that finishes the last, partial round with half tiles: one workgroup per CU, at least one whole
// round, and a last round that two half tiles per left-over tile still fit into (see the kernel).
bool half_tail_ok(const Variant &v, int m, int n, int k, int num_cu) {
    if (!v.persistent_half_tail || !persistent_ok(v, m, n, k)) return false;
    const long t = (long)ceil_div(m, v.bm) * ceil_div(n, v.bn);
    const long r = t % num_cu;
    return t >= num_cu && r > 0 && (r + 7) / 8 * 8 + r <= num_cu;
}

// Skinny-K schedule (fp8_gemm_skinny.h): one to four K blocks, whole 16-row m-tiles and whole 64-column wave tiles.
bool skinny_ok(int m, int n, int k) {
    return k >= rf::BK && k <= 4 * rf::BK && k % rf::BK == 0 && m >= 16 && m % 16 == 0 && n >= 64 && n % 64 == 0;
}

// Bands of rows the skinny-K schedule deals to the XCDs (see skinny_work), as a power of two; -1: none, workgroups as they
// come. With g bands an XCD fetches 1/g of A and g/8 of B; B counts four times, since everybody waits for it at the start
// while A streams ahead of its use. us, none -> one band / two: 512 x 7168 x 384 7.2 -> 4.9 / 5.1; 1024 x 7168 x 256 6.9 -> 5.5 / 5.5;
// 4096 x 7168 x 256 14.9 -> 13.5 / 13.5; 6144 x 7168 x 256 21.2 -> 19.9 / 23.2; 6144 x 3072 x 512 17.4 -> 16.6 / 15.3; 8192 x 3072 x 384
// 17.0 -> 16.8 / 15.9. None where that is the faster way:
//   rows of C whose length is a power of two up to 8 KB put the few columns an XCD would have onto few channels of its L2
//     (8192 x 2048 x 256 8.1 -> 9.6 with one band); rows of 16 KB need two bands (6144 x 8192 x 256 24.7 -> 23.1 / 20.9)
//   K = 128: A and B are small next to C (3072 x 1536 x 128 4.4 -> 4.7, 4096 x 8192 x 128 12.1 -> 13.9; but 4096 x 7168 x 128 12.0 -> 11.5)
//   few strips whose shares come in eighths: each XCD has an eighth of the rows anyway (4096 x 576 x 384 4.8 -> 5.0; with shares
//     that do not, 6144 x 576 x 384 8.2 -> 7.2)
int skinny_bands_log2(int m, int n, int qk, int strips, int per_strip) {
    const bool power = (n & (n - 1)) == 0;
    if ((power && n <= 4096) || (qk == 1 && (power || n <= 4096)) || (strips <= 8 && per_strip % 8 == 0)) return -1;
    int best = power ? 1 : 0;
    for (int l = best + 1; l <= 3; l++)
        if ((double)m / (1 << l) + 0.5 * n * (1 << l) < (double)m / (1 << best) + 0.5 * n * (1 << best)) best = l;
    return best;
}

// Few-rows kernels keep offsets inside a K block in 32 bits.
bool fewrows_ok(long ldm, int n) { return ldm < (1 << 25) && n < (1 << 25); }

// Stream-K: at least one tile per workgroup (then a split tile has exactly two contributors, which is all the kernel
// handles) and no more tiles than arrival counters.
bool stream_k_ok(const Variant &v, int m, int n, int num_cu) {
    const long t = (long)ceil_div(m, v.bm) * ceil_div(n, v.bn);
    return v.streamk && t >= num_cu && t <= kMaxTileCounters;
}

// Plans measured on one MI355X by the tuner (python -m radeonflow_kernels_amd.tuner.gemm_tuner --all --emit).
// The role of the reference's DISPATCH_GEMM table (src/gemm/gemm_launcher.cpp:229-259), except that a shape
// outside the table is not an error: it gets the heuristic below.
const TunedPlan kTunedPlans[] = {
    {0, 0, 0, 0, 1, 1, 0},
#include "tuned_plans.inc"
};

constexpr int kTunedOnCUs = 256;

// Estimated time in microseconds of the best few-rows plan for a shape, and that plan. Its constants are searched on 22280
// plans measured on operand sets that rotate out of the L2 caches: M = 1 ... 512, 23 pairs of N and K from 200 to 8192 and 128
// to 7168, every few-rows variant with 1 to 14 splits (tuner/fewrows_model.py: --measure takes them, --fit searches; the model
// stands there too). The plan it picks is 2.3 % slower than the best one measured on average and 19 % at worst (least
// squares on the times: 3.9 % and 28 %); its figure is 13 % off. Variants 15 and 17 to 19 are not tried: with them the best
// measured plans are 0.2 % faster.
//   2.56                                       launch, and the way back
//   + 0.64 + 0.192 per KiB of sums handed over when K is split
//   + rounds * (b + 0.253 * batches of loads of a wave + c * K blocks of a wave * workgroups sharing a CU), times `any`
//     where rows of B start at any byte (any_bytes); variants that load the next K block while they multiply: one batch
//   + d * MB of A and B that all workgroups fetch + 0.0505 * MB of A and B
// `any` is 1.27 but for three variants: a row of 16 and 27's 128 columns is one cache line where it is aligned and two where it is not, and of 21 two
// workgroups share a CU and its L1. Searched on 12 pairs of ragged N from 1000 to 5003 and K from 384 to 7168, M = 1 ... 500
// (tuner/fewrows_model.py --ragged): the plan taken, any_tile_plan's among the choice, is 1.4 % behind the fastest on average and 12 % at
// worst, with 1.27 for all 2.5 % and 17 % (40 x 2003 x 7168 12.2 us on variant 16, 10.9 on 25).
double fewrows_plan(int m, int n, int k, int num_cu, bool any_bytes, rf_gemm_config *out) {
    struct Fit { int variant, per_cu, depth; double b, c, d, any = 1.27; };
    constexpr int kAll = 1 << 20;
    const Fit fits[] = {{14, 2, 3, 0.0238, 0.6526, 0.0811},    {16, 1, kAll, 0.017, 1.6541, 0.0325, 1.5},  {20, 1, kAll, 0.2932, 1.9032, 0.0785},
                        {21, 2, kAll, 1.3762, 1.0315, 0.0158, 1.5}, {22, 2, kAll, 0.0007, 0.6572, 0.086},  {23, 1, kAll, 0.0704, 1.4481, 0.0227},
                        {24, 2, kAll, 0.0049, 0.9508, 0.0676}, {25, 1, kAll, 0.0106, 1.7903, 0.0289}, {26, 2, kAll, 0.3722, 0.7608, 0.0427},
                        {27, 1, kAll, 1.0902, 1.385, 0.0109, 1.5}};
    const double operands = 0.0505e-6 * k * ((double)m + n);
    const int splits_tried[] = {1, 2, 3, 4, 5, 6, 8, 12, 14}, qk = k / rf::BK;
    double best = 1e30;
    for (const Fit &f : fits) {
        const Variant &v = kVariants[f.variant];
        const long items = (long)ceil_div(m, v.bm) * ceil_div(n, v.bn);
        for (int sp : splits_tried) {
            if (sp > qk || (sp > 1 && (items * sp > 4L * num_cu || items > kMaxTileCounters))) break;
            const int kb = ceil_div(qk, sp), parts = ceil_div(qk, kb), own = ceil_div(kb, v.waves_n);
            const long wgs = items * parts, rounds = (wgs + (long)num_cu * f.per_cu - 1) / ((long)num_cu * f.per_cu);
            const double mb = (double)wgs * kb * (v.bm + v.bn) * rf::BK * 1e-6 * 256 / num_cu;
            const double t = 2.5568 + (parts > 1 ? 0.6363 + 0.1919 * parts * v.bm * v.bn / 1024.0 : 0.0) +
                             rounds * (any_bytes ? f.any : 1.0) *
                                 (f.b + 0.2531 * ceil_div(own, f.depth) + f.c * own * (wgs > num_cu ? f.per_cu : 1)) +
                             f.d * mb + operands;
            if (t < best) {
                best = t;
                *out = {f.variant, sp, 8, RF_SCHEDULE_TILES};
            }
        }
    }
    return best;
}
// Rows up to which the few-rows kernels are considered; the second one where B (or C) needs staging or N is small, on devices
// with kTunedOnCUs units only (others keep the first, and with it the plans of their padded shapes). The estimate is fitted up to
// 512 rows and comes out 9 % low beyond, which is added where nothing but M can be ragged. A staged B costs a tiled plan up to
// three launches, which variant 21 beats up to a few thousand rows while N is small: few rows against the best of 25 tiled plans
// with their staging (fewrows_model.py --meet), us: 1000 x 1000 x 1024 8.5, 15.8; 1500 x 1000 x 2048 17.6, 22.8; 3000 x 1000 x 384
// 11.0, 13.9; 700 x 5003 x 1024 24.1, 21.3; 2000 x 2003 x 1024 24.4, 18.6. A small N leaves most compute units without one of
// the large tiles, so that those split K and sum in a second launch. Before -> with the few-rows kernels in the choice, us:
// 528 x 256 x 2048 10.1 -> 7.7, 1833 x 256 x 2048 13.2 -> 9.1, 1919 x 512 x 2048 17.0 -> 11.6, 848 x 576 x 1024 7.9 -> 6.1,
// 779 x 1024 x 1024 10.1 -> 7.7, 665 x 1536 x 384 6.4 -> 5.4; of 130 shapes with N = 200 ... 1536 and 513 to 4096 rows 27 are
// faster by 2 to 47 %, none slower by more than the 2 % that runs differ by.
constexpr int kFewRowsMaxM = 512, kFewRowsMaxMWide = 4096, kFewRowsSmallN = 1536;

// What a shape or its pointers need before the tiled kernels can run on it (see launch_padded): copies of A and a_scale, or of B
// (and of C on the way back). kTiledOnly: no few-rows plan.
// kBytesA, kBytesB: rows of that operand do not all start at a multiple of four bytes.
// kFewRowsOnly: the few-rows plan (m and n as they are). kCutC: rows of C are not whole cache lines.
// kCopyB: B is copied (kStageB without it: only C is unaligned). kNoSplitTiles: without split_tile_plan, whose plans want memory.
enum { kStageA = 1, kStageB = 2, kTiledOnly = 4, kBytesA = 8, kBytesB = 16, kFewRowsOnly = 32, kCutC = 64, kCopyB = 128, kNoSplitTiles = 256 };
static_assert(kNoSplitTiles == 1 << (rf::kStageBits - 1), "the last flag");

// The flags of a shape and its pointers (0: aligned).
int stage_flags(int m, int n, uintptr_t a, uintptr_t b, uintptr_t c) {
    const bool copy_b = n % 16 != 0 || b % 16 != 0;
    return (m % 16 != 0 || a % 16 != 0 ? kStageA : 0) | (copy_b || c % 16 != 0 ? kStageB : 0) | (copy_b ? kCopyB : 0) |
           (m % 4 != 0 || a % 4 != 0 ? kBytesA : 0) | (n % 4 != 0 || b % 4 != 0 ? kBytesB : 0) | (n % 64 != 0 || c % 128 != 0 ? kCutC : 0);
}

// The three estimates below decide what a call takes whose operands would have to be staged. Their constants are fitted (relative
// error) to plans of 430 random shapes measured on operand sets and C in rotation, as those of fewrows_plan are
// (tuner/staged_model.py: --measure takes them, --fit fits).

// Estimated time in microseconds of the best any-alignment tile plan for a shape, and that plan. 1809 plans, 8 % off:
//   1.84 + rounds * (f + K blocks * (c + c_a where rows of A start at any byte + c_b where rows of B do))
//   + 0.21 per million outputs, 0.56 more where rows of C are not whole lines (two tiles then write each line at their border) and
//     0.17 where those of B, and with a ragged N those of C, start at any byte
//   + 3.02 + 1.03 per million sums when K is split
double any_tile_plan(int m, int n, int k, int num_cu, int stage, rf_gemm_config *out) {
    struct Fit { int variant; double f, c, c_a, c_b; };
    const Fit fits[] = {{29, 2.54, 0.580, 0.093, 0.105}, {30, 3.835, 0.792, 0.093, 0.285}};
    const int splits_tried[] = {1, 2, 3, 4, 6, 8}, qk = k / rf::BK;
    const double mn = (double)m * n * 1e-6;
    double best = 1e30;
    for (const Fit &f : fits) {
        const Variant &v = kVariants[f.variant];
        const long tiles = (long)ceil_div(m, v.bm) * ceil_div(n, v.bn);
        const double per_block = f.c + (stage & kBytesA ? f.c_a : 0.0) + (stage & kBytesB ? f.c_b : 0.0);
        for (int sp : splits_tried) {
            if (sp > qk) break;
            const int kb = ceil_div(qk, sp), parts = ceil_div(qk, kb);
            if (parts > 1 && mn * parts > 40.0) break;      // no more than was measured, 150 MB of sums
            const long rounds = (tiles * parts + num_cu - 1) / num_cu;
            const double t = 1.837 + rounds * (f.f + kb * per_block) + (parts > 1 ? 3.021 + 1.029 * parts * mn : 0.0) +
                             mn * (0.21 + (stage & kCutC ? 0.562 : 0.0) + (stage & kBytesB ? 0.168 : 0.0));
            if (t < best) {
                best = t;
                *out = {f.variant, sp, 8, RF_SCHEDULE_TILES};
            }
        }
    }
    return best;
}

// Estimated time in microseconds of the skinny-K schedule on staged copies: `mn` million outputs in qk K blocks, the copy of A and
// the one of B, and C's way back, which costs less beyond the 15 million outputs (30 MB) that the L2 caches hold. 154 shapes, 7 % off.
// With it the plan taken of this schedule and any_tile_plan's is 0.9 % slower than the faster one on average and 22 % at worst.
// Shapes with ragged N, or only B or C unaligned, had none, and all of them took any_tile_plan's: 4256 x 8000 x 256 with B at an odd byte
// 46.8 -> 22.9 us, 6144 x 7168 x 256 with C 8 bytes off 74.2 -> 49.5, 8192 x 7160 x 256 97.5 -> 65.9, 6000 x 4090 x 128 46.9 -> 33.5; but
// 1264 x 5632 x 256 with C 8 bytes off stays (11.3, the schedule 15.6).
double skinny_staged_us(int qk, double mn, int stage) {
    double t = 2.137 + 1.033 * qk + (0.265 + 0.098 * qk) * mn;
    if (stage & kStageA) t += 2.591;
    if (stage & kCopyB) t += 2.948;
    if ((stage & kStageB) && (stage & kCutC)) t += 1.522 + 0.921 * std::min(mn, 15.0) + 0.369 * std::max(mn - 15.0, 0.0);
    return t;
}

// The same of one round of 128 x 128 tiles over three or four K blocks, nothing staged. 30 shapes, 2 % off.
double one_round_us(int qk, double mn) { return 3.458 + 0.526 * qk + 0.434 * mn; }

// A plan of one workgroup per tile and K part in estimated microseconds, where K is long and the chip is not full of the largest tile:
//   start + rounds * (f + K blocks of a part * (c + g * share of the units at work + b * cut B + a * cut A)) + out per million outputs
//   + in per million bytes of A and B + split + sum per million sums when K is split
// (the more units are at work the longer each waits for L2 and the longer a K block; cut: the share of that operand's rows that start
// inside a cache line, of which a tile then reads one more). Two sets of constants: operands that come from the Infinity Cache (calls that
// repeat, a layer or two) and from memory (the layers of a model in turn), where a K block of many units takes up to 1.5 times as
// long. Fitted (tuner/long_k_model.py: --measure takes the times, --fit fits; estimates and choice stand there too) to the plans
// within 1.5 times the fastest of 441 shapes (48 to 2464 rows, N = 256 to 8192, K = 1024 to 8192, 40 % of them the benchmark's pairs of N
// and K), every variant below with 1 to 8 parts on operand sets in rotation. Cached 6.9 % off (root mean square, 35 % at worst) over all
// 9922 plans of these shapes and from memory 7.0 % (41 %); fitted to two thirds of the shapes, 6.9 and 7.1 % on the others. The model in
// select_config_uncached, which ranks plans first, counts a K split's sums at twice what they cost against a K block, and a K block the
// same on half the chip as on all of it. `*out` is replaced (split_tile_plan) where another plan is below both estimates: with the second
// alone a fifth of the plans that changed were over 2 % slower cached, up to 1.45 times (272 x 8192 x 7168 29.4 us, 42.4 with four parts).
// That is 7 % of the shapes in the range. 291 of them, none fitted, plan after against plan before: cached 10 % faster (geometric mean; nine by over
// 2 % slower, 7.3 % at worst), from memory 18 % (one, 7.3 %). 160 calls with odd rows: 7 and 17 % faster (three, 5.8 %).
// us, cached and from memory: 1232 x 1616 x 7552 38.1 -> 31.0, 53.0 -> 33.2 (28 in one part, 11 in four); 304 x 1632 x 2176 12.8 -> 11.3, 12.8 ->
// 11.4; 544 x 4096 x 7168 28.6 -> 29.1, 41.8 -> 31.8 (28 in one part, 10 in three).
// Left out: the 64 x 128 tile in one part, which takes plans from variant 12 that are up to 9 % faster. In 64 bits' terms the results are
// as exact as before (relative error 1.660e-3 to 1.664e-3 on either side, the bf16 of C).
struct SplitTileFit { int variant; double f, c, g, b, a; };
struct SplitTileCosts { SplitTileFit of[7]; double start, out, in, split, sum; };
constexpr SplitTileCosts kSplitTileCached = {
    {{9, 0.0, 0.366, 0.0, 0.07, 0.028}, {12, 0.185, 0.592, 0.147, 0.19, 0.059}, {28, 0.194, 0.333, 0.132, 0.069, 0.039}, {8, 0.765, 0.496, 0.077, 0.033, 0.039},
     {10, 0.759, 0.59, 0.077, 0.073, 0.058}, {11, 0.875, 0.738, 0.021, 0.036, 0.018}, {0, 1.138, 1.033, 0.023, 0.049, 0.104}},
    4.531, 0.403, 0.0, 2.274, 1.177};
constexpr SplitTileCosts kSplitTileMemory = {
    {{9, 0.169, 0.397, 0.041, 0.047, 0.028}, {12, 0.0, 0.63, 0.444, 0.172, 0.066}, {28, 0.073, 0.375, 0.23, 0.072, 0.056}, {8, 0.497, 0.574, 0.217, 0.025, 0.072},
     {10, 0.712, 0.692, 0.076, 0.086, 0.088}, {11, 0.76, 0.847, 0.056, 0.038, 0.042}, {0, 1.004, 1.207, 0.0, 0.095, 0.087}},
    3.922, 0.531, 0.054, 2.283, 1.173};
// Share of the rows of `bytes` bytes, one after the other, that do not start at a multiple of 128.
double cut_rows(int bytes) { return 1.0 - std::min(bytes & -bytes, 128) / 128.0; }
// 0 for a variant that is not estimated.
double split_tile_us(const SplitTileCosts &costs, int variant, int m, int n, int k, int splits, int num_cu) {
    const Variant &v = kVariants[variant];
    const int qk = k / rf::BK;
    const double wgs = (double)ceil_div(m, v.bm) * ceil_div(n, v.bn) * splits, mn = (double)m * n * 1e-6;
    const double rounds = std::ceil(wgs / num_cu), blocks = v.k_groups > 1 ? qk / v.k_groups : ceil_div(qk, splits);
    for (const SplitTileFit &f : costs.of)
        if (f.variant == variant)
            return costs.start + rounds * (f.f + blocks * (f.c + f.g * wgs / num_cu / rounds + f.b * cut_rows(n) + f.a * cut_rows(m))) + costs.out * mn + costs.in * 1e-6 * k * ((double)m + n) +
                   (splits > 1 ? costs.split + costs.sum * mn * splits : 0.0);
    return 0.0;
}
// The sizes it was fitted to and checked on; plans beyond them stay as the first model has them.
bool long_k_range(int m, int n, int k) {
    return m >= 48 && m <= 2608 && n >= 256 && n <= 8192 && k >= 1024 && k <= 8192 && (double)n * k <= 6.0e7;
}
// Returns the cached figure of the plan that it leaves in *out, 0 for one that is not estimated here. K splits whose sums take more than
// `most` bytes are not tried. What part of the plan before's figure another's has to stay below: from memory 0.94; cached, by what the estimates of
// 763 such pairs are off by (time over estimate, new plan against plan before): up to 512 rows K splits come out too low, 1.03 to 1.09,
// beyond them not (variant 28 0.91, 10 0.97, 11 1.0), 9 in place of 12 too low at any size, 1.04 to 1.08. Up to 512 rows 103 of 348 pairs
// change at 0.93 and five are over 2 % slower (54 of 198 at 0.97), beyond 512 rows 247 of 415 and 13 at 1.0 (72 and one at 0.93). Of 62 pairs
// with 9 in place of 12 eleven were slower at 0.93 and 1.0, up to 9.7 %, none of 21 at 0.88; of 56 with 28 in place of 12 three at 1.0 (1600 x
// 384 x 3072 12.4 -> 13.6 us), one of 39 at 0.96. Where rows of B are a multiple of 1024 bytes apart 12 takes up to 20 % longer than its figure:
// 32 shapes that change there are 8 % faster, 1.7 % slower at worst (551 x 2048 x 4096 20.6 -> 18.8 us).
double split_tile_plan(int m, int n, int k, int num_cu, rf_gemm_config *out, size_t most = SIZE_MAX) {
    const int qk = k / rf::BK, parts = ceil_div(qk, ceil_div(qk, out->split_k));
    const double cached = split_tile_us(kSplitTileCached, out->variant, m, n, k, parts, num_cu);
    const int first = out->variant;
    double kept = cached, best = 0.94 * split_tile_us(kSplitTileMemory, out->variant, m, n, k, parts, num_cu);
    for (const SplitTileFit &f : kSplitTileMemory.of) {
        const Variant &v = kVariants[f.variant];
        // (up to 512 rows variant 28 in more parts is not tried: the few-rows kernels were weighed against its plan of the first model)
        if (f.variant == 28 && m <= kFewRowsMaxM) continue;
        const double tiles = (double)ceil_div(m, v.bm) * ceil_div(n, v.bn);
        const double limit = (f.variant == 9 ? (first == 12 ? 0.88 : 0.93) : m <= kFewRowsMaxM ? 0.93 : first != 12 ? 1.0 : n % 1024 == 0 ? 1.06 : 0.96) * cached;
        for (int sp : {1, 2, 3, 4, 5, 6, 8}) {
            if (sp > qk || ceil_div(qk, ceil_div(qk, sp)) != sp || (v.k_groups > 1 && (sp > 1 || qk % v.k_groups != 0))) continue;
            if (sp == 1 && f.variant == 9) continue;
            if (sp > 1 && (tiles * sp > 600 || (double)m * n * sp > 45.0e6)) continue;      // no more than was measured
            if (sp > 1 && (size_t)m * n * sizeof(float) * sp > most) continue;
            const double us = split_tile_us(kSplitTileCached, f.variant, m, n, k, sp, num_cu);
            if (us >= limit) continue;
            const double t = split_tile_us(kSplitTileMemory, f.variant, m, n, k, sp, num_cu);
            if (t < best) {
                best = t;
                kept = us;
                *out = {f.variant, sp, 8, RF_SCHEDULE_TILES};
            }
        }
    }
    return kept;
}

// Plan for a shape (m, n multiples of 16, the padded sizes when something is staged).
void select_config_uncached(int m, int n, int k, int num_cu, int stage, const std::vector<TunedPlan> &user_plans,
                            rf_gemm_config *out) {
    out->split_k = 1;
    out->group_m = 8;
    out->stream_k = 0;
    auto fewrows_usable = [&](const TunedPlan &p) {
        const Variant &v = kVariants[p.variant];
        return !(stage & kTiledOnly) && p.stream_k == RF_SCHEDULE_TILES && fewrows_ok(m, n) &&
               (p.split_k == 1 || (long)ceil_div(m, v.bm) * ceil_div(n, v.bn) <= kMaxTileCounters);
    };
    auto usable = [&](const TunedPlan &p) {
        return p.m == m && p.n == n && p.k == k && p.variant < kNumVariants && p.split_k <= k / rf::BK &&
               (!kVariants[p.variant].is_fewrows() || fewrows_usable(p)) &&
               (!kVariants[p.variant].is_any_tile() || (p.stream_k == RF_SCHEDULE_TILES && fewrows_ok(m, n))) &&
               (kVariants[p.variant].k_groups == 1 || (p.split_k == 1 && (k / rf::BK) % kVariants[p.variant].k_groups == 0)) &&
               (p.stream_k != RF_SCHEDULE_PERSISTENT || persistent_ok(kVariants[p.variant], m, n, k)) &&
               (p.stream_k != RF_SCHEDULE_STREAM_K || stream_k_ok(kVariants[p.variant], m, n, num_cu)) &&
               (p.stream_k != RF_SCHEDULE_PERSISTENT_HALF_TAIL || half_tail_ok(kVariants[p.variant], m, n, k, num_cu)) &&
               (p.stream_k != RF_SCHEDULE_SKINNY_K || skinny_ok(m, n, k));
    };
    const TunedPlan *hit = nullptr;
    for (const TunedPlan &p : user_plans)
        if (!hit && usable(p)) hit = &p;
    // the compiled-in table was measured on a device with kTunedOnCUs compute units: round counts, and with them the
    // best tile and split, change with the unit count, so another device takes the cost model below (which counts
    // rounds for the device at hand) unless the caller has loaded plans measured there
    auto take = [&](const TunedPlan &p) { *out = {p.variant, p.split_k, p.group_m, p.stream_k}; };
    if (hit) return take(*hit);
    if (num_cu == kTunedOnCUs)
        for (const TunedPlan &p : kTunedPlans)
            if (!hit && usable(p)) hit = &p;
    if (hit && (!(stage & (kStageA | kStageB)) || kVariants[hit->variant].takes_any_shape())) return take(*hit);
    // Up to four K blocks and a large C: the launch is a streaming store, which the skinny-K schedule does best. Against the best
    // tiled plan, us: K = 128, 592 x 7168 5.1, 5.4 and 1328 x 4096 5.8, 6.5, but 592 x 4096 (2.4 million outputs) 4.4, 3.9; K = 256,
    // 848 x 7168 6.2, 6.8 and 2016 x 3072 5.9, 7.0, but 592 x 7168 6.3, 6.3 and 2048 x 2048 6.5, 5.6; K = 384, 1328 x 3072 6.3, 6.9
    // and 848 x 7168 7.3, 7.7. With K = 512 and more than sixteen strips the tiles are as fast or faster up to 20 million outputs
    // (2016 x 7168 13.5, 13.3) and again beyond 60 (8048 x 8192 57.5, 54.2; between them 3008 x 7168 18.7, 20.8). Three or four K blocks whose C is one
    // round of 128 x 128 tiles: those (variant 28), 592 x 4096 x 512 7.7 -> 6.3, 1328 x 2048 x 512 7.2 -> 6.7, 848 x 4096 x 384 6.9 -> 6.2,
    // 3008 x 576 x 512 6.7 -> 6.1; 336 x 7168 x 384 5.7, 5.8.
    // Staged operands: the schedule has to beat the tiles that take them as they are, see below.
    const double mn = (double)m * n;
    const int qk = k / rf::BK;
    const bool staged = stage & (kStageA | kStageB);
    const int tiles_128 = ceil_div(m, 128) * ceil_div(n, 128);
    const bool one_round = !staged && num_cu == kTunedOnCUs && (qk == 3 || qk == 4) && tiles_128 <= num_cu && tiles_128 >= 96 &&
                           (qk == 4 || mn >= 2.0e6);
    const bool skinny = !one_round && skinny_ok(m, n, k) &&
                        (qk == 1 ? mn >= 4.1e6 : qk == 2 ? mn >= 6.0e6 : mn >= 2.0e6 && (qk == 3 || ceil_div(n, 256) <= 16));
    if (one_round) out->variant = 28;
    if (skinny) {
        if (hit) {
            take(*hit);
        } else {
            out->variant = 0;
            out->stream_k = RF_SCHEDULE_SKINNY_K;
        }
        if (!staged || num_cu != kTunedOnCUs) return;
    }
    // No measured entry: a cost model whose constants were searched on the tuner's measurements of the tabled shapes so
    // that its plan comes close to the best measured one. Searched on 213 shapes (the 163 of the table and 50 others,
    // 36 of them drawn at random with M = 16 ... 8192, N = 512 ... 8192, K = 128 ... 8192): 0.8 % slower than the best
    // measured plan on average, 10 % at worst. On shapes a search had not seen its constants were 1.7 to 1.9 % behind
    // on average and 8 to 16 % at worst (14, 60 and 36 shapes). The constants rank plans, they are not measured times.
    // Time in microseconds of a plan =
    //   rounds * (K blocks per workgroup * c + f)           one workgroup per tile and K split
    //   rounds * K blocks * c + f + (rounds - 1) * f_next   persistent: only the first tile starts cold
    //   the same over the whole rounds + f_next + K blocks * c + f of the three-stage 128x256 tile
    //                                                       persistent with a last round of half tiles (the half
    //                                                       tiles start cold: at K = 512 the plain persistent
    //                                                       schedule of 128x256 tiles is 15-20 % faster)
    //   + reduction cost when K is split
    // with rounds = ceil(workgroups / CUs). Candidates: the 256x256 tile and the 128x256, 192x192, 128x192 and 64x128
    // tiles with two and with three stages (192-wide tiles win where they divide the shape into fuller rounds or leave
    // no padded columns, e.g. N = 576, 1536 or 3072; the 64x128 tile where M is short or the whole problem is a few
    // microseconds); the others never won by more than a few percent.
    struct Candidate { int variant; double c, f; };
    // (variant 12 splits K between two wave groups of one workgroup: half the K blocks per group, one launch, no
    // reduction term. The 64 x 128 tile: the best plan of short shapes, M <= 512, with K = 512 ... 2304. Variant 28, the
    // 128 x 128 tile with eight waves and three stages, searched for by itself on 37 further shapes, the other constants as
    // they were: choice 1.4 % behind the best of all, 4.6 % without it. Not among them: variants 6 (c = 0.74, f = 4.3) and 13
    // (half of 1.06, 3.3), whose tiles 8 and 28 have at less of both)
    const Candidate cands[] = {{0, 0.905, 5.96}, {3, 0.679, 3.61}, {5, 0.80, 5.8},  {7, 0.85, 0.3},  {8, 0.52, 4.2},
                               {9, 0.73, 0.5},   {10, 0.53, 5.9},  {11, 0.71, 7.0}, {12, 0.93, 1.4}, {28, 0.44, 2.25}};
    const double f_next = 3.3, reduce_fixed = 6.03, reduce_per_elem = 1.27e-6, c_half_tile = 0.47, f_half_tile = 5.2;
    const int splits_tried[] = {1, 2, 3, 4, 6, 8, 12, 16};
    double best_cost = 1e30, cost_28 = 1e30;
    int split_28 = 1;
    if (!skinny && !one_round) for (const Candidate &cd : cands) {
        const Variant &v = kVariants[cd.variant];
        const long tiles = (long)ceil_div(m, v.bm) * ceil_div(n, v.bn);
        for (int sp : splits_tried) {
            if (sp > qk) break;
            if (v.k_groups > 1) {
                if (sp != 1 || qk % v.k_groups != 0) continue;
                const double t = (double)((tiles + num_cu - 1) / num_cu) * (qk / v.k_groups * cd.c + cd.f);
                if (t < best_cost) {
                    best_cost = t;
                    out->variant = cd.variant;
                    out->split_k = 1;
                    out->stream_k = RF_SCHEDULE_TILES;
                }
                continue;
            }
            const int kb_per = ceil_div(qk, sp), splits = ceil_div(qk, kb_per);
            const long rounds = (tiles * splits + num_cu - 1) / num_cu;
            for (int sched : {RF_SCHEDULE_TILES, RF_SCHEDULE_PERSISTENT}) {
                if (sched == RF_SCHEDULE_PERSISTENT && (splits != 1 || !persistent_ok(v, m, n, k))) continue;
                double t = sched == RF_SCHEDULE_PERSISTENT ? rounds * kb_per * cd.c + cd.f + (rounds - 1) * f_next
                                                           : rounds * (kb_per * cd.c + cd.f);
                if (splits > 1) t += reduce_fixed + reduce_per_elem * splits * (double)m * n;
                if (cd.variant == 28 && t < cost_28) {
                    cost_28 = t;
                    split_28 = sp;
                }
                if (t < best_cost) {
                    best_cost = t;
                    out->variant = cd.variant;
                    out->split_k = sp;
                    out->stream_k = sched;
                }
                if (sched == RF_SCHEDULE_PERSISTENT && half_tail_ok(v, m, n, k, num_cu)) {
                    t = (rounds - 1) * kb_per * cd.c + cd.f + (rounds - 1) * f_next + kb_per * c_half_tile + f_half_tile;
                    if (t < best_cost) {
                        best_cost = t;
                        out->variant = cd.variant;
                        out->split_k = 1;
                        out->stream_k = RF_SCHEDULE_PERSISTENT_HALF_TAIL;
                    }
                }
            }
        }
    }
    if (hit) take(*hit);                                    // a measured plan, but one that would run on staged copies
    // Few rows: the few-rows kernels, which need no staging, when they come out faster. The model above ranks tiled plans;
    // what their launches take is 3.1 us + 0.67 of its figure, and staging adds the copies' launches and bytes. B's term
    // counts C's way back for every plan, although plans of one K part and one workgroup per tile store into a ragged C
    // themselves. Counting it (1.0 us + 0.9 us per million outputs) per plan instead made 33 of 187 shapes 5 % faster on average,
    // but ten of them 1 to 31 % slower (664 x 3001 x 7168 43 -> 56 us: the figure of a K split is too high against that of one part).
    double t = 3.1 + 0.67 * best_cost;
    if (stage & kStageA) t += 3.2 + 2.0 * k * m / 4e6;
    if (stage & kStageB) t += 7.0 + 2.0 * k * n / 5e6 + 4.0 * m * n / 5e6;
    if (skinny) t = skinny_staged_us(qk, 1e-6 * mn, stage);
    if (one_round) t = one_round_us(qk, 1e-6 * mn);
    rf_gemm_config other;
    const int max_m = ((stage & kStageB) || n <= kFewRowsSmallN) && num_cu == kTunedOnCUs ? kFewRowsMaxMWide : kFewRowsMaxM;
    if (m <= max_m && fewrows_ok(m, n) && !(stage & kTiledOnly)) {
        const double few = fewrows_plan(m, n, k, num_cu, (stage & kStageB) != 0, &other) * (m > kFewRowsMaxM && !(stage & kStageB) ? 1.09 : 1.0);
        if (few < t) {
            t = few;
            *out = other;
        }
    }
    // Operands that would be staged: the tiles that take them as they are, on the compute unit count they were measured on.
    // On 166 shapes that the fit has not seen (100 to 8192 rows, M or N or both ragged) the plan taken is 1.2 % behind the best of few
    // rows, these tiles with every K split and the plans of the padded shape on average, 24 % at worst.
    if ((stage & (kStageA | kStageB)) && num_cu == kTunedOnCUs && fewrows_ok(m, n) && any_tile_plan(m, n, k, num_cu, stage, &other) < t) *out = other;
    if (!hit && num_cu == kTunedOnCUs && !(stage & (kStageB | kNoSplitTiles)) && out->stream_k == RF_SCHEDULE_TILES &&
        !kVariants[out->variant].takes_any_shape() && long_k_range(m, n, k) && ceil_div(m, 256) * ceil_div(n, 256) <= num_cu) {
        // The few-rows kernels again, against the cached figure of a plan of one K part (a tiled plan of long K has too low a `t` above). How far
        // below it they have to be, by pairs of times: 28 at 0.85 25 pairs change, one is over 2 % slower (at 0.92 five of 37); 12 at 0.88 52 and
        // one, at 0.93 89 and four; where rows of B are a multiple of 1024 bytes apart 12 takes up to 20 % longer than its figure: 46 and none,
        // 7 % faster. 169 shapes that change plan here, before against after: cached 5 % faster (geometric mean; two by over 2 % slower, 4.3 % at
        // worst), from memory 9 % (one, 2.6 %). us: 256 x 3824 x 2560 14.2 -> 12.6, 17.5 -> 13.1; 112 x 8192 x 2048 12.1 -> 10.2, 15.5 -> 12.6. Not
        // against plans with a K split: 128 x 7344 x 4608 18.1 (28, four parts), 22.0.
        // (Variant 28's best plan, which tuner/fewrows_model.py knows, has to be behind as well.)
        const double tiled = split_tile_plan(m, n, k, num_cu, out);
        if (m <= kFewRowsMaxM && out->split_k == 1 && !(stage & kTiledOnly) && fewrows_ok(m, n)) {
            const double few = fewrows_plan(m, n, k, num_cu, false, &other);
            const double share = out->variant == 28 ? 0.85 : out->variant == 12 && n % 1024 == 0 ? 1.0 : 0.88, share_28 = n % 1024 == 0 ? 1.0 : 0.85;
            const bool below_28 = split_28 == 1 ? few < share_28 * split_tile_us(kSplitTileCached, 28, m, n, k, 1, num_cu) : few < 3.1 + 0.67 * cost_28;
            if (few < share * tiled && below_28) *out = other;
        }
    }
}

// The same through a small table of plans already worked out (the models take 1 to 3 us of host time, as long as a small
// launch). Entries hold for one generation of the loaded plan files; the caller holds the lock.
void select_config(int m, int n, int k, int num_cu, int stage, rf_gemm_config *out) {
    struct Entry { int m, n, k, num_cu, stage, generation; rf_gemm_config cfg; };
    constexpr unsigned kEntries = 1024;
    static Entry table[kEntries];                           // zeroed: no entry has k == 0
    Entry &e = table[rf::plan_slot(m, n, k, stage, kEntries)];
    if (e.m != m || e.n != n || e.k != k || e.num_cu != num_cu || e.stage != stage || e.generation != shared().plan_generation) {
        e = {m, n, k, num_cu, stage, shared().plan_generation, {}};
        if (stage & kFewRowsOnly) fewrows_plan(m, n, k, num_cu, (stage & kStageB) != 0, &e.cfg);
        else select_config_uncached(m, n, k, num_cu, stage, shared().user_plans, &e.cfg);
    }
    *out = e.cfg;
}

// Bytes in which the workgroups of a few-rows launch with K in `parts` parts hand over their sums.
size_t fewrows_slot_bytes(const Variant &v, int m, int n, int parts) {
    return (size_t)ceil_div(m, v.bm) * v.bm * ceil_div(n, v.bn) * v.bn * sizeof(float) * parts;
}

// Whether the memory of a few-rows plan's K split is to be had: not on a stream under capture that would have to take over
// another stream's buffers, nor when device memory has run out. (Static mode: the caller cuts the split down beforehand.)
bool fewrows_split_fits(Mem &mem, const Variant &v, int m, int n, int k, int splits) {
    if (splits == 1 || mem.fixed) return true;
    const int qk = k / rf::BK;
    return mem.try_workspace(fewrows_slot_bytes(v, m, n, ceil_div(qk, ceil_div(qk, splits))));
}

// The same of a tiled plan's K split: without memory for its sums the plan is the one that split_tile_plan found. mp: the rows that are
// planned, m: those of c, stage: the plan's flags. In the static array, beside `staged` bytes of copies, that plan in the parts that fit
// is weighed once more against the others that fit: 942 x 1904 x 6016, A staged, 37.5 us cached and 46.0 from memory (28, one part) -> 28.5 and
// 32.4 (8, three parts instead of four of 10). 150 shapes whose plan does not fit, against the plan that split_tile_plan found: 9 % faster
// cached (geometric mean), 12 % from memory, one 2.7 % slower cached and the others within the 1 % that runs differ by.
void fit_tile_split(State &s, Mem &mem, int m, int mp, int n, int k, int stage, size_t staged, rf_gemm_config *cfg) {
    if (cfg->variant < 0 || cfg->split_k == 1 || cfg->stream_k != RF_SCHEDULE_TILES || kVariants[cfg->variant].takes_any_shape()) return;
    const int qk = k / rf::BK, parts = ceil_div(qk, ceil_div(qk, cfg->split_k));
    const size_t part = (size_t)m * n * sizeof(float), left = mem.fixed_left() > staged ? mem.fixed_left() - staged : 0;
    if (mem.fixed ? part * parts <= left : mem.try_workspace(part * parts)) return;
    rf_gemm_config first;
    select_config(mp, n, k, s.num_cu, stage | kNoSplitTiles, &first);
    const bool changed = first.variant != cfg->variant || first.split_k != cfg->split_k;
    *cfg = first;
    if (!mem.fixed || !changed) return;
    if (cfg->split_k > 1) cfg->split_k = (int)std::max<size_t>(1, std::min<size_t>(cfg->split_k, left / part));
    split_tile_plan(mp, n, k, s.num_cu, cfg, left);
}

// m rows out of ldm (the distance between two K rows of a and as); any shape and alignment. splits >= 1.
int launch_fewrows(Mem &mem, const Variant &v, const void *a, const void *b, const float *as, const float *bs, void *c, int m,
                   int ldm, int n, int k, int splits, hipStream_t stream) {
    const int qk = k / rf::BK, row_blocks = ceil_div(m, v.bm), items = ceil_div(n, v.bn) * row_blocks;
    const int kb_per_split = ceil_div(qk, splits);
    splits = ceil_div(qk, kb_per_split);                    // every split owns at least one K block
    CounterSet *counters = nullptr;
    float *slots = nullptr;
    if (splits > 1) {
        if (items > kMaxTileCounters) return fail(RF_ERR_BAD_CONFIG, "too many tiles for a K split of this variant");
        int rc = mem.counters(&counters);
        if (rc != RF_OK) return rc;
        rc = mem.workspace(fewrows_slot_bytes(v, m, n, splits), &slots);
        if (rc != RF_OK) return rc;
    }
    const bool any = n % 16 != 0 || (uintptr_t)b % 16 != 0;
    enqueue(v.fewrows[splits > 1][any], dim3(items, splits), dim3(v.threads()), v.lds_bytes(), stream,
            (const uint8_t *)a, (const uint8_t *)b, as, bs, (uint16_t *)c, m, ldm, n, k, kb_per_split, row_blocks,
            counters ? counters->tile : nullptr, slots);
    RF_HIP(hipGetLastError());
    return RF_OK;
}

// Bytes of a part's sums in a K split of an any-alignment tile plan: rows and columns rounded up to whole 16-byte pieces.
size_t any_tile_part_bytes(int m, int n) { return (size_t)ceil_div(m, 16) * 16 * ceil_div(n, 16) * 16 * sizeof(float); }

dim3 pad_grid_of_pieces(int pieces, int rows, int rounds);

// Any shape and alignment; rows of A and a_scale are ldm (>= m) long. splits >= 1.
int launch_any_tile(Mem &mem, const Variant &v, const void *a, const void *b, const float *as, const float *bs, void *c, int m, int ldm,
                    int n, int k, int splits, int group_m, hipStream_t stream) {
    const int qk = k / rf::BK, tiles_m = ceil_div(m, v.bm), tiles_n = ceil_div(n, v.bn), kb_per_split = ceil_div(qk, splits);
    splits = ceil_div(qk, kb_per_split);                    // every split owns at least one K block
    void *out = c;
    if (splits > 1) {
        float *ws = nullptr;
        const int rc = mem.workspace(any_tile_part_bytes(m, n) * splits, &ws);
        if (rc != RF_OK) return rc;
        out = ws;
    }
    enqueue(v.any_tile[splits > 1], dim3(tiles_m * tiles_n, splits), dim3(v.threads()), v.lds_bytes(), stream,
            (const uint8_t *)a, (const uint8_t *)b, as, bs, out, m, ldm, n, k, kb_per_split, tiles_m, tiles_n, group_m);
    RF_HIP(hipGetLastError());
    if (splits > 1) {
        const int np = ceil_div(n, 16) * 16;
        enqueue(rf::reduce_splitk_any_c, pad_grid_of_pieces(ceil_div(n, 8), m, 1), dim3(256), 0, stream, (const float *)out, np,
                any_tile_part_bytes(m, n) / sizeof(float), splits, n, m, (uint16_t *)c);
        RF_HIP(hipGetLastError());
    }
    return RF_OK;
}

// The launch proper; the caller holds the lock and has checked shape and pointers. m_store >= 0: c has only m_store
// (<= m) rows, the rest of the m rows of the operands are padding (one workgroup per tile schedules only).
int launch_locked(State &s, Mem &mem, const void *a, const void *b, const float *as, const float *bs, void *c, int m, int n,
                  int k, const rf_gemm_config *user_cfg, hipStream_t stream, int m_store = -1) {
    int rc = RF_OK;
    if (m_store < 0) m_store = m;
    const bool tiled_ok = tiled_path_ok(a, b, c, m, n);
    rf_gemm_config cfg;
    if (user_cfg) {
        cfg = *user_cfg;
        if (cfg.variant >= kNumVariants || cfg.variant < -1 || cfg.split_k < 1 || cfg.group_m < 1 ||
            cfg.split_k > k / rf::BK || (cfg.variant >= 0 && !kVariants[cfg.variant].takes_any_shape() && !tiled_ok) || (cfg.variant < 0 && cfg.split_k != 1) ||
            (cfg.stream_k != 0 && (cfg.variant < 0 || cfg.split_k != 1)))
            return fail(RF_ERR_BAD_CONFIG, "configuration not usable for this shape");
        if (cfg.variant >= 0 && kVariants[cfg.variant].takes_any_shape() && !fewrows_ok(m, n))
            return fail(RF_ERR_BAD_CONFIG, "the few-rows and any-alignment kernels need M and N below 2^25");
        if (cfg.variant >= 0 && kVariants[cfg.variant].k_groups > 1 &&
            (cfg.split_k != 1 || cfg.stream_k != RF_SCHEDULE_TILES || (k / rf::BK) % kVariants[cfg.variant].k_groups != 0))
            return fail(RF_ERR_BAD_CONFIG, "this variant splits K inside the workgroup: it needs split_k == 1, the tile "
                                           "schedule and a number of K blocks that its wave groups divide");
        if (cfg.stream_k == RF_SCHEDULE_STREAM_K) {
            const Variant &sv = kVariants[cfg.variant];
            if (!sv.streamk) return fail(RF_ERR_BAD_CONFIG, "this variant has no stream_k form");
            if (!stream_k_ok(sv, m, n, s.num_cu))
                return fail(RF_ERR_BAD_CONFIG, "stream_k needs at least as many tiles as compute units");
        } else if (cfg.stream_k == RF_SCHEDULE_PERSISTENT) {
            if (!persistent_ok(kVariants[cfg.variant], m, n, k))
                return fail(RF_ERR_BAD_CONFIG, "the persistent schedule needs M >= the tile height, M % 16 == 0, N a multiple of the tile width, K/128 even, and K * M and K * N below 2^32");
        } else if (cfg.stream_k == RF_SCHEDULE_PERSISTENT_HALF_TAIL) {
            if (!half_tail_ok(kVariants[cfg.variant], m, n, k, s.num_cu))
                return fail(RF_ERR_BAD_CONFIG, "the half-tile schedule needs the 256x256 tile, the persistent schedule's "
                                               "shape rules, at least one tile per compute unit and a last round that "
                                               "is at most half full");
        } else if (cfg.stream_k == RF_SCHEDULE_SKINNY_K) {
            if (cfg.variant != 0 || !skinny_ok(m, n, k))
                return fail(RF_ERR_BAD_CONFIG, "the skinny-K schedule needs variant 0, K = 128 ... 512, M a multiple of 16 and N a multiple of 64");
        } else if (cfg.stream_k != RF_SCHEDULE_TILES) {
            return fail(RF_ERR_BAD_CONFIG, "unknown schedule");
        }
    } else {
        if (tiled_ok) select_config(m, n, k, s.num_cu, 0, &cfg);
        else cfg = {-1, 1, 8, RF_SCHEDULE_TILES};
        // no memory for a few-rows plan's sums: the tiled plan, which often needs none
        if (cfg.variant >= 0 && kVariants[cfg.variant].is_fewrows() &&
            !fewrows_split_fits(mem, kVariants[cfg.variant], m, n, k, cfg.split_k))
            select_config(m, n, k, s.num_cu, kTiledOnly, &cfg);
        // no memory for a tiled plan's sums
        fit_tile_split(s, mem, m_store, m, n, k, kTiledOnly, 0, &cfg);
    }

    if (mem.fixed && cfg.variant >= 0) {
        // rf_fp8_gemm_static: the plan has to live inside what is left of the static array. A stream-K plan (only a
        // plan file can name one) is replaced by the cost model's plan; a K split whose partial sums do not fit is cut
        // down to the number of parts that do, a single part needing no scratch memory at all.
        if (cfg.stream_k == RF_SCHEDULE_STREAM_K) select_config_uncached(m, n, k, s.num_cu, kNoSplitTiles, std::vector<TunedPlan>(), &cfg);
        if (cfg.stream_k == RF_SCHEDULE_STREAM_K) cfg.stream_k = RF_SCHEDULE_TILES;
        if (cfg.split_k > 1) {
            const Variant &fv = kVariants[cfg.variant];
            // (of the rows of c, as the launches below have it)
            const size_t per_part = fv.is_fewrows() ? fewrows_slot_bytes(fv, m_store, n, 1)
                                    : fv.is_any_tile() ? any_tile_part_bytes(m_store, n) : (size_t)m_store * n * sizeof(float);
            const int qk_ = k / rf::BK, kb_per = ceil_div(qk_, cfg.split_k), parts = ceil_div(qk_, kb_per);
            const size_t fit = mem.fixed_left() / per_part;
            if ((size_t)parts > fit) cfg.split_k = fit < 2 ? 1 : (int)fit;
        }
    }
    if (m_store != m && (cfg.variant < 0 || cfg.stream_k == RF_SCHEDULE_STREAM_K))
        return fail(RF_ERR_BAD_CONFIG, "internal: this schedule cannot write fewer rows than it computes");
    if (cfg.variant < 0 && !user_cfg && fewrows_ok(m, n)) {
        // a small problem the tiled kernels do not take (reported as plan -1: no tile variant): the few-rows kernels do. A wave
        // of the bounds-checked kernel gathers bytes K block after K block, 13 to 27 us where these take 3 to 4
        // (M x N x K = 4 x 200 x 2048: 27.8 -> 3.7, 8 x 1000 x 384: 13.6 -> 3.1).
        select_config(m, n, k, s.num_cu, kFewRowsOnly | (n % 16 != 0 ? kStageB : 0), &cfg);
        if (!fewrows_split_fits(mem, kVariants[cfg.variant], m, n, k, cfg.split_k)) cfg.split_k = 1;
        return launch_fewrows(mem, kVariants[cfg.variant], a, b, as, bs, c, m, m, n, k, cfg.split_k, stream);
    }
    if (cfg.variant < 0) {
        dim3 grid(ceil_div(n, 16), ceil_div(m, 16));
        enqueue(rf::gemm_fp8_blockscale_checked, grid, dim3(64), 0, stream, (const uint8_t *)a,
                (const uint8_t *)b, as, bs, (uint16_t *)c, m, m, n, k);
        RF_HIP(hipGetLastError());
        return RF_OK;
    }

    const Variant &v = kVariants[cfg.variant];
    if (v.is_fewrows()) return launch_fewrows(mem, v, a, b, as, bs, c, m_store, m, n, k, cfg.split_k, stream);
    if (v.is_any_tile()) {
        if (cfg.stream_k != RF_SCHEDULE_TILES) return fail(RF_ERR_BAD_CONFIG, "the any-alignment tiles have one schedule");
        return launch_any_tile(mem, v, a, b, as, bs, c, m_store, m, n, k, cfg.split_k, cfg.group_m, stream);
    }
    const int tiles_m = ceil_div(m, v.bm), tiles_n = ceil_div(n, v.bn);
    const int qk = k / rf::BK;
    const int kb_per_split = ceil_div(qk, cfg.split_k);
    const int splits = ceil_div(qk, kb_per_split);          // every split owns at least one K block
    dim3 grid(tiles_m * tiles_n, splits);
    dim3 block(v.threads());
    if (cfg.stream_k == RF_SCHEDULE_PERSISTENT) {
        // as many resident workgroups as the LDS of a CU holds (small tiles: two or three per CU, so that one's
        // store drain overlaps another's compute)
        const int T = tiles_m * tiles_n;
        int per_cu = (160 * 1024) / v.lds_persistent;
        if (per_cu > 2048 / v.threads()) per_cu = 2048 / v.threads();
        const int P = s.num_cu * (per_cu < 1 ? 1 : per_cu);
        enqueue(v.persistent, dim3(T < P ? T : P), block, v.lds_persistent, stream,
                (const uint8_t *)a, (const uint8_t *)b, as, bs, (uint16_t *)c, m, n, k, tiles_m, tiles_n,
                cfg.group_m, m_store);
        RF_HIP(hipGetLastError());
        return RF_OK;
    }
    if (cfg.stream_k == RF_SCHEDULE_SKINNY_K) {
        // one strip of 256 columns per workgroup, and as many workgroups per strip as fill the chip once (each takes a
        // share of the strip's rows, in units of 64)
        const int strips = ceil_div(n, 256), units = ceil_div(m, 64);
        int per_strip = s.num_cu / strips;
        per_strip = per_strip < 1 ? 1 : per_strip > units ? units : per_strip;
        // From 40 million outputs on C is written band by band, all workgroups of a strip side by side, and not a stretch of rows each.
        // Time with rounds over without, 96 shapes of 7 to 60 million outputs, N = 2048 ... 8192, operands and C in rotation: beyond 42
        // million 0.98 on average (0.88 ... 1.02; 6272 x 7168 x 256 25.3 -> 22.3 us), 40 to 42 million 0.99, 32 to 39.5 million 1.00 at K = 128
        // and 1.03 at K = 256, below 1.00 and 1.01 (0.94 ... 1.07, as the rows divide among the workgroups). All of these C are smaller than
        // the Infinity Cache. The 64-row items of K = 384 and 512 spend more on each item (6144 x 7168 x 384 24.5 -> 25.0).
        const int rounds = qk <= 2 && (double)m * n >= 4.0e7 ? m / (per_strip * rf::SkinnyGeom<2>::IM) : 0;
        const int rest = ceil_div(m - rounds * per_strip * rf::SkinnyGeom<2>::IM, 64);
        const rf::SkinnyWork work = {strips, per_strip, skinny_bands_log2(m, n, qk, strips, per_strip), rounds, rest / per_strip, rest % per_strip};
#define RF_LAUNCH_SKINNY(QK)                                                                                            \
    enqueue(rf::gemm_fp8_blockscale_skinny<QK>, dim3(strips * per_strip), dim3(512),                         \
            rf::SkinnyGeom<QK>::LDS_BYTES, stream, (const uint8_t *)a, (const uint8_t *)b, as, bs,           \
            (uint16_t *)c, m, n, work, m_store)
        if (qk == 1) RF_LAUNCH_SKINNY(1);
        else if (qk == 2) RF_LAUNCH_SKINNY(2);
        else if (qk == 3) RF_LAUNCH_SKINNY(3);
        else RF_LAUNCH_SKINNY(4);
#undef RF_LAUNCH_SKINNY
        RF_HIP(hipGetLastError());
        return RF_OK;
    }
    if (cfg.stream_k == RF_SCHEDULE_PERSISTENT_HALF_TAIL) {
        enqueue(v.persistent_half_tail, dim3(s.num_cu), block, v.lds_persistent, stream, (const uint8_t *)a,
                (const uint8_t *)b, as, bs, (uint16_t *)c, m, n, k, tiles_m, tiles_n, cfg.group_m, m_store);
        RF_HIP(hipGetLastError());
        return RF_OK;
    }
    if (cfg.stream_k == RF_SCHEDULE_STREAM_K) {
        const int P = s.num_cu;
        CounterSet *counters = nullptr;
        float *ws = nullptr;
        rc = mem.counters(&counters);
        if (rc != RF_OK) return rc;
        rc = mem.workspace((size_t)2 * P * v.bm * v.bn * sizeof(float), &ws);
        if (rc != RF_OK) return rc;
        enqueue(v.streamk, dim3(P), block, v.lds_bytes(), stream, (const uint8_t *)a, (const uint8_t *)b, as,
                bs, (uint16_t *)c, m, n, k, tiles_m, tiles_n, cfg.group_m, counters->tile, ws);
        RF_HIP(hipGetLastError());
        return RF_OK;
    }
    if (splits == 1) {
        enqueue(v.direct, grid, block, v.lds_bytes(), stream, (const uint8_t *)a, (const uint8_t *)b, as, bs,
                c, m, n, k, kb_per_split, tiles_m, tiles_n, cfg.group_m, m_store);
        RF_HIP(hipGetLastError());
    } else {
        const size_t mn = (size_t)m_store * n;
        float *ws = nullptr;
        rc = mem.workspace(mn * splits * sizeof(float), &ws);
        if (rc != RF_OK) return rc;
        enqueue(v.partial, grid, block, v.lds_bytes(), stream, (const uint8_t *)a, (const uint8_t *)b, as,
                bs, (void *)ws, m, n, k, kb_per_split, tiles_m, tiles_n, cfg.group_m, m_store);
        RF_HIP(hipGetLastError());
        enqueue(rf::reduce_splitk_bf16, dim3((unsigned)((mn / 4 + 255) / 256)), dim3(256), 0, stream,
                (const float *)ws, (uint16_t *)c, mn, splits);
        RF_HIP(hipGetLastError());
    }
    return RF_OK;
}

// ---- shapes and pointers the tiled kernels do not take as they are ----
// M or N not a multiple of 16 (or below 16), or operands that are not 16-byte aligned. Token counts are arbitrary in
// practice. Where the few-rows kernels, which take such operands as they are, are not the faster ones, the operands that need
// it are copied into a staging buffer with rows padded to a multiple of 16 (zeros: padded rows and columns produce values
// nobody reads), the tiled kernels run on the padded shape under the automatic plan and store into the caller's C where they
// can (one K part, one workgroup per tile); otherwise C is copied back without the padding. b_scale needs no copy:
// ceil(N/128) does not change. The copies cost K*M (+ K*N when N is ragged) bytes.
// Below this many multiply-adds a ragged shape takes the few-rows kernel estimated fastest without a look at the plans (a
// launch of a few microseconds, whose plan the table and the cost model do not know better); a grouped call that would have
// to stage runs the bounds-checked kernel.
constexpr double kPadThresholdMacs = 2097152.0;

// The grouped GEMM's staging copy: the caller's [rows][m_total] matrix (A with T = bytes, a_scale with T = float), in
// which group g owns columns out_row_start[g] .. out_row_start[g+1]-1 (counted from column `first`), is copied to
// [rows][m_pad] with group g starting at column row_start[g], a multiple of 16; the columns between a group's end and the
// next start become zero. Bound by memory, but for few columns by latency: a workgroup writes the 16-byte pieces of whole
// rows side by side, kPadRows rounds of 256 / (pieces of a row) rows, so that all its threads have work at any width (256
// pieces of kPadRows rows when rows are longer), and every thread finds its group by a search in LDS instead of a walk
// over the kernel argument. A source piece starts at any byte and is one unaligned 16-byte load, cut at the end of the matrix.
// 1001 x 7168 bytes: 7.7 -> 6.8 us (rocprofv3), 48 rows in 32 groups x 7168: 10.6 -> 5.8 us, 2.8 us of either being what
// the shortest kernel takes. One round up to kPadOneRound bytes, whose workgroups hardly fill the chip, two beyond: the GEMM with
// its copy in two rounds -> one, us: 701 x 7168 x 2048 26.4 -> 25.7, 3001 x 7168 x 256 16.7 -> 16.0, 1990 x 2048 x 2048 21.8 -> 21.4;
// even at 1001 x 4608 x 7168 (7.3 MB), but 5001 x 7168 x 2048 (10.5 MB) 86.3 -> 87.2. (Four rounds: up to 5 % slower.)
constexpr double kPadOneRound = 8.0e6;
template <typename T, int kPadRows>
__device__ __forceinline__ void pad_group_rows_body(const T *__restrict__ src, int first, int m_total, int m_pad, int rows,
                                                    int groups, T *__restrict__ dst, const rf::GroupTable &table,
                                                    int block_row, int block_chunk) {
    constexpr int PER = 16 / sizeof(T);
    const int pieces = m_pad / PER;
    if (block_chunk * 256 >= pieces) return;
    __shared__ int row_start[rf::kMaxGroups + 1], out_row_start[rf::kMaxGroups + 1];
    if (groups > 1) {
        for (int g = threadIdx.x; g <= groups; g += 256) {
            row_start[g] = table.row_start[g];
            out_row_start[g] = table.out_row_start[g];
        }
        __syncthreads();
    }
    const int per_round = pieces < 256 ? 256 / pieces : 1;
    const int trow = pieces < 256 ? (int)threadIdx.x / pieces : 0;
    const int piece = pieces < 256 ? (int)threadIdx.x - trow * pieces : block_chunk * 256 + (int)threadIdx.x;
    if (trow >= per_round || piece >= pieces) return;
    const int col = piece * PER;
    int start = 0, from = 0, count = table.out_row_start[1];
    if (groups > 1) {                                                  // the last group that starts at or before col
        int lo = 0, hi = groups;
        while (hi - lo > 1) {
            const int mid = (lo + hi) >> 1;
            if (row_start[mid] <= col) lo = mid; else hi = mid;
        }
        start = row_start[lo];
        from = out_row_start[lo];
        count = out_row_start[lo + 1] - from;
    }
    int valid = count - (col - start);                                 // columns of this piece that exist in the source
    valid = valid < 0 ? 0 : valid > PER ? PER : valid;
    const int r_first = block_row * kPadRows * per_round + trow;
    const size_t at = (size_t)first + from + (col - start);            // column in the source
    rf::u32x4_lds w[kPadRows];
#pragma unroll
    for (int u = 0; u < kPadRows; u++) {
        const int r = r_first + u * per_round;
        w[u] = (rf::u32x4_lds){0u, 0u, 0u, 0u};
        if (r < rows && valid > 0) {
            if constexpr (sizeof(T) == 4) {
                const uint32_t *p = (const uint32_t *)src + (size_t)r * m_total + at;
#pragma unroll
                for (int e = 0; e < 4; e++) w[u][e] = e < valid ? p[e] : 0u;
            } else {
                const size_t off = (size_t)r * m_total + at, last = (size_t)rows * m_total - 16;     // rows >= 128
                w[u] = *(const rf::u32x4_any *)(src + (off < last ? off : last));
            }
        }
    }
#pragma unroll
    for (int u = 0; u < kPadRows; u++) {
        const int r = r_first + u * per_round;
        if (r >= rows) continue;
        if constexpr (sizeof(T) == 1) {
            const size_t off = (size_t)r * m_total + at, last = (size_t)rows * m_total - 16;
            if (off > last) w[u] = rf::shift_back(w[u], (uint32_t)(off - last), 16u);
#pragma unroll
            for (int e = 0; e < 4; e++) {
                const int nv = valid - 4 * e;
                if (nv < 4) w[u][e] = nv <= 0 ? 0u : w[u][e] & ((1u << (8 * nv)) - 1u);
            }
        }
        *(uint4 *)(dst + (size_t)r * m_pad + col) = make_uint4(w[u][0], w[u][1], w[u][2], w[u][3]);
    }
}

template <typename T, int kPadRows>
__global__ __launch_bounds__(256) void pad_group_rows(const T *__restrict__ src, int m_total, int m_pad, int rows,
                                                      int groups, T *__restrict__ dst, const rf::GroupTable table) {
    pad_group_rows_body<T, kPadRows>(src, 0, m_total, m_pad, rows, groups, dst, table, blockIdx.x, blockIdx.y);
}

// A and a_scale in one launch (they are staged together whenever M or the group sizes are ragged): the first
// blocks_a workgroups along x copy the bytes of A, the others the floats of a_scale.
template <int kPadRows>
__global__ __launch_bounds__(256) void pad_group_rows_a_and_scales(const uint8_t *__restrict__ a, const float *__restrict__ as,
                                                                   int first, int m_total, int m_pad, int k, int groups,
                                                                   uint8_t *__restrict__ a_dst, float *__restrict__ as_dst,
                                                                   int blocks_a, const rf::GroupTable table) {
    if ((int)blockIdx.x < blocks_a)
        pad_group_rows_body<uint8_t, kPadRows>(a, first, m_total, m_pad, k, groups, a_dst, table, blockIdx.x, blockIdx.y);
    else
        pad_group_rows_body<float, kPadRows>(as, first, m_total, m_pad, k / rf::BK, groups, as_dst, table, blockIdx.x - blocks_a,
                                   blockIdx.y);
}

// The way back: the first n columns of C's padded copy [rows][ld], ld a multiple of 16, to the caller's [rows][n]. The same
// split, a piece per thread; a piece is one aligned load and one 16-byte store at any element, the last piece of a row stored by elements.
// (hipMemcpy2DAsync took 120 us for 6160 x 5003, a width whose rows start at odd elements: 6160 x 5003 x 2048 202 -> 104 us.)
__global__ __launch_bounds__(256) void unpad_rows_bf16(const uint16_t *__restrict__ src, int ld, int n, int rows,
                                                       uint16_t *__restrict__ dst) {
    const int pieces = (n + 7) / 8;
    const int per_block = pieces < 256 ? 256 / pieces : 1;
    const int trow = pieces < 256 ? (int)threadIdx.x / pieces : 0;
    const int piece = pieces < 256 ? (int)threadIdx.x - trow * pieces : (int)(blockIdx.y * 256 + threadIdx.x);
    const int r = (int)blockIdx.x * per_block + trow, col = piece * 8;
    if (trow >= per_block || piece >= pieces || r >= rows) return;
    const rf::u32x4_lds w = *(const rf::u32x4_lds *)(src + (size_t)r * ld + col);
    uint16_t *out = dst + (size_t)r * n + col;
    if (col + 8 <= n) {
        *(rf::u32x4_any *)out = w;
    } else {
#pragma unroll
        for (int e = 0; e < 7; e++)
            if (col + e < n) out[e] = (uint16_t)(w[e / 2] >> (16 * (e % 2)));
    }
}

// grid of these copies for `rows` rows of `pieces` 16-byte pieces, `rounds` rows per thread
dim3 pad_grid_of_pieces(int pieces, int rows, int rounds) {
    const int per_block = rounds * (pieces < 256 ? 256 / pieces : 1);
    return dim3((unsigned)ceil_div(rows, per_block), (unsigned)ceil_div(pieces, 256));     // rows on x: no 65535 limit
}
dim3 pad_grid(int m_pad, int size, int rows, int rounds) { return pad_grid_of_pieces(m_pad / (16 / size), rows, rounds); }

void launch_unpad_rows(const void *src, int ld, int n, int rows, void *dst, hipStream_t stream) {
    enqueue(unpad_rows_bf16, pad_grid_of_pieces(ceil_div(n, 8), rows, 1), dim3(256), 0, stream, (const uint16_t *)src,
            ld, n, rows, (uint16_t *)dst);
}

// Stages A and a_scale with one launch: columns first, first + 1, ... of matrices of m_total columns.
void launch_pad_a_and_scales(const void *a, const float *as, int first, int m_total, int m_pad, int k, int groups,
                             uint8_t *a_dst, float *as_dst, const rf::GroupTable &table, hipStream_t stream) {
    const bool one = (double)m_pad * k <= kPadOneRound;
    const dim3 ga = pad_grid(m_pad, 1, k, one ? 1 : 2), gs = pad_grid(m_pad, 4, k / rf::BK, one ? 1 : 2);
    const auto kernel = one ? &pad_group_rows_a_and_scales<1> : &pad_group_rows_a_and_scales<2>;
    enqueue(kernel, dim3(ga.x + gs.x, ga.y > gs.y ? ga.y : gs.y), dim3(256), 0, stream,
            (const uint8_t *)a, as, first, m_total, m_pad, k, groups, a_dst, as_dst, (int)ga.x, table);
}

// table of one group of `cols` columns padded to `cols_pad`
rf::GroupTable one_group(int cols, int cols_pad) {
    rf::GroupTable t;
    t.row_start[0] = t.out_row_start[0] = t.tile_start[0] = 0;
    for (int g = 1; g <= rf::kMaxGroups; g++) {
        t.row_start[g] = cols_pad;
        t.out_row_start[g] = cols;
        t.tile_start[g] = 0;
    }
    return t;
}

// Stages one matrix of K rows of `cols` bytes.
void launch_pad_bytes(const void *src, int cols, int cols_pad, int k, uint8_t *dst, hipStream_t stream) {
    const bool one = (double)cols_pad * k <= kPadOneRound;
    const auto kernel = one ? &pad_group_rows<uint8_t, 1> : &pad_group_rows<uint8_t, 2>;
    enqueue(kernel, pad_grid(cols_pad, 1, k, one ? 1 : 2), dim3(256), 0, stream, (const uint8_t *)src, cols, cols_pad, k, 1,
            dst, one_group(cols, cols_pad));
}

// rf_fp8_gemm_static on a ragged or unaligned shape whose staging copies do not fit the static array as a whole: the
// rows of the problem are cut into pieces (row ranges of A, a_scale and C are independent GEMMs), each piece is staged,
// computed and, where C is staged too, copied back before the next one re-uses the same memory; the stream orders them.
// The staged copy of B (ragged N or an unaligned b) is shared by all pieces and has to fit beside them: when it takes
// more than half of the array, the 64 x 64 few-rows kernel computes the whole problem in place instead.
int launch_padded_in_pieces(State &s, Mem &mem, const void *a, const void *b, const float *as, const float *bs, void *c,
                            int m, int n, int k, hipStream_t stream) {
    auto pad16 = [](int x) { return x < 16 ? 16 : (x + 15) / 16 * 16; };
    auto align = [](size_t x) { return (x + 255) / 256 * 256; };
    const int np = pad16(n), qk = k / rf::BK;
    const bool copy_b = np != n || (uintptr_t)b % 16 != 0;
    const bool copy_c = np != n || (uintptr_t)c % 16 != 0;
    const size_t b_bytes = copy_b ? align((size_t)k * np) : 0;
    // per row of a piece: its bytes of A, of a_scale and (when C is staged) of C; a quarter of what is left after B is
    // kept for the piece's split-K partial sums (launch_locked cuts the split down to what fits)
    const size_t per_row = (size_t)k + (size_t)qk * sizeof(float) + (copy_c ? (size_t)np * 2 : 0);
    const size_t left = mem.fixed_left() > b_bytes ? mem.fixed_left() - b_bytes : 0;
    long rows_fit = (long)((left - left / 4) / per_row) / 16 * 16 - 16;
    if (b_bytes > mem.fixed_left() / 2 || rows_fit < 16) {
        if (fewrows_ok(m, n))
            return launch_fewrows(mem, kVariants[kFewRows64x64], a, b, as, bs, c, m, m, n, k, 1, stream);
        enqueue(rf::gemm_fp8_blockscale_checked, dim3(ceil_div(n, 16), ceil_div(m, 16)), dim3(64), 0, stream,
                (const uint8_t *)a, (const uint8_t *)b, as, bs, (uint16_t *)c, m, m, n, k);
        RF_HIP(hipGetLastError());
        return RF_OK;
    }
    int rc = RF_OK;
    const void *b2 = b;
    if (copy_b) {
        uint8_t *pb = nullptr;
        rc = mem.pad(b_bytes, &pb);
        if (rc != RF_OK) return rc;
        launch_pad_bytes(b, n, np, k, pb, stream);
        RF_HIP(hipGetLastError());
        b2 = pb;
    }
    const size_t base = mem.fixed_used;
    const int pieces = ceil_div(m, (int)(rows_fit < m ? rows_fit : m));
    const int rows_per = (ceil_div(m, pieces) + 15) / 16 * 16;           // even pieces, whole m-tiles
    for (int r0 = 0; r0 < m; r0 += rows_per) {
        const int rows = m - r0 < rows_per ? m - r0 : rows_per, rp = pad16(rows);
        mem.fixed_used = base;                                            // the pieces take turns in the same memory
        uint8_t *pa = nullptr, *psa = nullptr, *pc = nullptr;
        if ((rc = mem.pad(align((size_t)k * rp), &pa)) != RF_OK) return rc;
        if ((rc = mem.pad(align((size_t)qk * rp * sizeof(float)), &psa)) != RF_OK) return rc;
        if (copy_c && (rc = mem.pad(align((size_t)rp * np * 2), &pc)) != RF_OK) return rc;
        // columns r0 .. r0 + rows - 1 of the caller's [K][m] matrices, padded to rp columns
        launch_pad_a_and_scales(a, as, r0, m, rp, k, 1, pa, (float *)psa, one_group(rows, rp), stream);
        RF_HIP(hipGetLastError());
        rf_gemm_config cfg;
        select_config(rp, np, k, s.num_cu, kNoSplitTiles, &cfg);
        void *c_piece = copy_c ? (void *)pc : (void *)((uint16_t *)c + (size_t)r0 * n);
        rc = launch_locked(s, mem, pa, b2, (const float *)psa, bs, c_piece, rp, np, k, &cfg, stream, copy_c ? rp : rows);
        if (rc != RF_OK) return rc;
        if (copy_c) {
            launch_unpad_rows(pc, np, n, rows, (uint16_t *)c + (size_t)r0 * n, stream);
            RF_HIP(hipGetLastError());
        }
    }
    return RF_OK;
}

int launch_padded(State &s, Mem &mem, const void *a, const void *b, const float *as, const float *bs, void *c, int m, int n,
                  int k, hipStream_t stream) {
    auto pad16 = [](int x) { return x < 16 ? 16 : (x + 15) / 16 * 16; };
    auto align = [](size_t x) { return (x + 255) / 256 * 256; };
    int mp = pad16(m), np = pad16(n);
    const int qk = k / rf::BK;
    const bool copy_a = mp != m || (uintptr_t)a % 16 != 0, copy_b = np != n || (uintptr_t)b % 16 != 0;
    const bool copy_sa = mp != m;
    // The plan of the padded shape. With whole columns and an aligned c, the whole-tile schedules (one workgroup per
    // tile, persistent) write the m true rows straight into c (their stores are masked by row), and the tile kernels
    // have a form for any c; otherwise C is staged and copied back.
    rf_gemm_config cfg;
    const int stage = stage_flags(m, n, (uintptr_t)a, (uintptr_t)b, (uintptr_t)c);
    select_config(mp, np, k, s.num_cu, stage, &cfg);
    if (!(stage & kStageB))
        fit_tile_split(s, mem, m, mp, n, k, stage, (copy_a ? align((size_t)k * mp) : 0) + (copy_sa ? align((size_t)qk * mp * sizeof(float)) : 0), &cfg);
    // The skinny-K schedule in the static array: a C that is staged and does not fit would be computed and copied back range by
    // range, with launches for each, behind the tiles that write it in place: 8192 x 7160 x 256 138 us, 98; 2144 x 7860 x 256 47, 36.
    if (mem.fixed && cfg.stream_k == RF_SCHEDULE_SKINNY_K && (np != n || (uintptr_t)c % 16 != 0) && fewrows_ok(m, n) &&
        (size_t)mp * np * 2 + (size_t)k * ((size_t)mp + np) > mem.fixed_left())
        any_tile_plan(mp, np, k, s.num_cu, stage, &cfg);
    if (kVariants[cfg.variant].is_any_tile()) {
        const size_t part = any_tile_part_bytes(m, n);
        if (mem.fixed && cfg.split_k > 1) {                // as many K parts as the static array holds
            const size_t fit = mem.fixed_left() / part;
            if ((size_t)cfg.split_k > fit) cfg.split_k = fit < 2 ? 1 : (int)fit;
        } else if (cfg.split_k > 1) {                      // no memory for the sums: K in one part
            float *ws = nullptr;
            const int qk_ = k / rf::BK, parts = ceil_div(qk_, ceil_div(qk_, cfg.split_k));
            if (mem.workspace(part * parts, &ws) != RF_OK) {
                (void)hipGetLastError();
                g_last_error.clear();
                cfg.split_k = 1;
            }
        }
        return launch_any_tile(mem, kVariants[cfg.variant], a, b, as, bs, c, m, m, n, k, cfg.split_k, cfg.group_m, stream);
    }
    if (kVariants[cfg.variant].is_fewrows()) {
        if (mem.fixed && cfg.split_k > 1) {                // as many K parts as the static array holds
            const Variant &v = kVariants[cfg.variant];
            const size_t fit = mem.fixed_left() / fewrows_slot_bytes(v, m, n, 1);
            if ((size_t)cfg.split_k > fit) cfg.split_k = fit < 2 ? 1 : (int)fit;
        } else if (!fewrows_split_fits(mem, kVariants[cfg.variant], m, n, k, cfg.split_k)) {
            cfg.split_k = 1;                               // no memory for the sums: K in one part
        }
        return launch_fewrows(mem, kVariants[cfg.variant], a, b, as, bs, c, m, m, n, k, cfg.split_k, stream);
    }
    // whole K in one part, one workgroup per tile: the kernel stores into any c itself
    const bool any_c = (np != n || (uintptr_t)c % 16 != 0) && cfg.split_k == 1 && cfg.stream_k == RF_SCHEDULE_TILES &&
                       cfg.variant >= 0 && kVariants[cfg.variant].any_c;
    const bool copy_c = !any_c && (np != n || (uintptr_t)c % 16 != 0 || (mp != m && cfg.stream_k == RF_SCHEDULE_STREAM_K));
    if (!mem.fixed && !copy_c && cfg.variant >= 0) {
        // The staged rows become whole cache lines where that adds no tile and the schedule still holds (staged_length): a row of
        // a tile is then one or two lines, and not one more. Rows of A of 1024 bytes instead of 1008 (N x K = 4608 x 7168), of B of
        // 4608 instead of 4592, us: 128 x 192 tiles 41.4 -> 39.6, 128 x 256 46.5 -> 43.4 and 45.2 -> 43.4, 128 x 128 61.7 -> 57.7 and
        // 63.4 -> 57.7; 256 x 256, 2032 rows, 74.5 -> 72.2 and 78.7 -> 72.2.
        const Variant &v = kVariants[cfg.variant];
        const bool persistent = cfg.stream_k == RF_SCHEDULE_PERSISTENT || cfg.stream_k == RF_SCHEDULE_PERSISTENT_HALF_TAIL;
        if (copy_a && copy_sa) mp = rf::staged_length(mp, cfg.stream_k == RF_SCHEDULE_SKINNY_K ? 64 : v.bm, np, k, persistent);
        if (copy_b && any_c) np = rf::staged_length(np, v.bn, mp, k, false);      // (any_c: one workgroup per tile)
    }
    size_t off = 0;
    const size_t off_a = off;  off += copy_a ? align((size_t)k * mp) : 0;
    const size_t off_b = off;  off += copy_b ? align((size_t)k * np) : 0;
    const size_t off_sa = off; off += copy_sa ? align((size_t)qk * mp * sizeof(float)) : 0;
    const size_t off_c = off;  off += copy_c ? align((size_t)mp * np * 2) : 0;
    if (mem.fixed && off > mem.fixed_left()) return launch_padded_in_pieces(s, mem, a, b, as, bs, c, m, n, k, stream);
    uint8_t *pad = nullptr;
    int rc = off ? mem.pad(off, &pad) : RF_OK;
    if (rc != RF_OK && !mem.fixed && fewrows_ok(m, n)) {   // no memory for the copies: the tiles that need none, K in one part
        (void)hipGetLastError();
        g_last_error.clear();
        return launch_any_tile(mem, kVariants[kAnyTile128], a, b, as, bs, c, m, m, n, k, 1, 8, stream);
    }
    if (rc != RF_OK) return rc;
    const void *a2 = a, *b2 = b;
    const float *as2 = as;
    void *c2 = c;
    if (copy_a && copy_sa) {
        launch_pad_a_and_scales(a, as, 0, m, mp, k, 1, pad + off_a, (float *)(pad + off_sa), one_group(m, mp), stream);
        a2 = pad + off_a;
        as2 = (const float *)(pad + off_sa);
    } else if (copy_a) {                                   // M is fine, only the pointer is not aligned
        launch_pad_bytes(a, m, mp, k, pad + off_a, stream);
        a2 = pad + off_a;
    }
    if (copy_b) {
        launch_pad_bytes(b, n, np, k, pad + off_b, stream);
        b2 = pad + off_b;
    }
    if (copy_c) c2 = pad + off_c;
    RF_HIP(hipGetLastError());
    if (any_c) {
        const Variant &v = kVariants[cfg.variant];
        const int tiles_m = ceil_div(mp, v.bm), tiles_n = ceil_div(np, v.bn);
        enqueue(v.any_c, dim3(tiles_m * tiles_n), dim3(v.threads()), v.lds_bytes(), stream, (const uint8_t *)a2,
                (const uint8_t *)b2, as2, bs, (uint16_t *)c, mp, np, k, tiles_m, tiles_n, cfg.group_m, m, n);
        RF_HIP(hipGetLastError());
        return RF_OK;
    }
    rc = launch_locked(s, mem, a2, b2, as2, bs, c2, mp, np, k, &cfg, stream, copy_c ? mp : m);
    if (rc != RF_OK) return rc;
    if (copy_c) {
        launch_unpad_rows(c2, np, n, m, c, stream);
        RF_HIP(hipGetLastError());
    }
    return RF_OK;
}

int launch(const void *a, const void *b, const float *as, const float *bs, void *c, int m, int n, int k,
           const rf_gemm_config *user_cfg, hipStream_t stream, bool static_memory = false) {
    g_last_error.clear();
    if (m < 1 || n < 1 || k < rf::BK || k % rf::BK != 0)
        return fail(RF_ERR_BAD_SHAPE, "unsupported shape M=" + std::to_string(m) + " N=" + std::to_string(n) +
                                          " K=" + std::to_string(k) + " (need M,N>=1, K a positive multiple of 128)");
    if (!a || !b || !as || !bs || !c) return fail(RF_ERR_NULL_POINTER, "null device pointer");
    State &s = state();
    std::lock_guard<std::mutex> lock(shared().mu);
    int rc = ensure_device_info(s);
    if (rc != RF_OK) return rc;
    Mem mem{s};
    mem.stream = stream;
    if (static_memory) mem.fixed = s.static_scratch;
    if (!user_cfg && !tiled_path_ok(a, b, c, m, n) && (double)m * n * k >= kPadThresholdMacs)
        return launch_padded(s, mem, a, b, as, bs, c, m, n, k, stream);
    return launch_locked(s, mem, a, b, as, bs, c, m, n, k, user_cfg, stream);
}

// The plan a launch with aligned pointers takes: a shape the tiled kernels do not take as it is is planned at its padded size.
void plan_of_shape(int m, int n, int k, int num_cu, rf_gemm_config *out) {
    auto pad16 = [](int x) { return x < 16 ? 16 : (x + 15) / 16 * 16; };
    const int mp = pad16(m), np = pad16(n);
    if ((mp != m || np != n) && (double)m * n * k < kPadThresholdMacs) *out = {-1, 1, 8, RF_SCHEDULE_TILES};
    else select_config(mp, np, k, num_cu, stage_flags(m, n, 0, 0, 0), out);
}

// ---- timing record for run() ----------------------------------------------------------------
struct TimerJob {
    hipEvent_t start, stop;
    double flop;
    float *time_ms, *gflops;
    State *owner;                        // the device state whose event pool the pair came from
};
void timer_callback(hipStream_t, hipError_t status, void *user) {
    TimerJob *job = static_cast<TimerJob *>(user);
    if (status == hipSuccess) {
        float ms = 0.f;
        if (hipEventElapsedTime(&ms, job->start, job->stop) == hipSuccess) {
            if (job->time_ms) *job->time_ms = ms;
            if (job->gflops) *job->gflops = (float)(job->flop / (ms * 1e-3) / 1e9);
        }
    }
    State &s = *job->owner;               // the callback thread has no current device of its own
    {
        // the pool has a lock of its own: the launch path may hold the library lock while it waits for the device,
        // and the device may be waiting for this callback
        std::lock_guard<std::mutex> lock(s.ev_mu);
        s.free_events.emplace_back(job->start, job->stop);   // recycled, unlike the reference's growing list
    }
    delete job;
}

}  // namespace

extern "C" {

int rf_fp8_gemm(const void *a, const void *b, const float *as, const float *bs, void *c, int m, int n, int k,
                hipStream_t stream) {
    return launch(a, b, as, bs, c, m, n, k, nullptr, stream);
}

int rf_fp8_gemm_static(const void *a, const void *b, const float *as, const float *bs, void *c, int m, int n, int k,
                       hipStream_t stream) {
    return launch(a, b, as, bs, c, m, n, k, nullptr, stream, /*static_memory=*/true);
}

size_t rf_gemm_static_scratch_bytes(void) { return kStaticScratchBytes; }

int rf_fp8_gemm_ex(const void *a, const void *b, const float *as, const float *bs, void *c, int m, int n, int k,
                   const rf_gemm_config *cfg, hipStream_t stream) {
    return launch(a, b, as, bs, c, m, n, k, cfg, stream);
}

int rf_fp8_gemm_time(const void *a, const void *b, const float *as, const float *bs, void *c, int m, int n, int k,
                     const rf_gemm_config *cfg, int warmup, int iters, float *us_per_launch, hipStream_t stream) {
    if (!us_per_launch || iters < 1 || warmup < 0) {
        g_last_error.clear();
        return fail(RF_ERR_BAD_CONFIG, "rf_fp8_gemm_time needs iters >= 1, warmup >= 0 and a result pointer");
    }
    for (int i = 0; i < warmup; i++) {
        int rc = launch(a, b, as, bs, c, m, n, k, cfg, stream);
        if (rc != RF_OK) return rc;
    }
    hipEvent_t e0, e1;
    RF_HIP(hipEventCreate(&e0));
    RF_HIP(hipEventCreate(&e1));
    int rc = RF_OK;
    hipError_t err = hipEventRecord(e0, stream);
    for (int i = 0; i < iters && rc == RF_OK && err == hipSuccess; i++) rc = launch(a, b, as, bs, c, m, n, k, cfg, stream);
    if (err == hipSuccess) err = hipEventRecord(e1, stream);
    if (err == hipSuccess) err = hipEventSynchronize(e1);
    float ms = 0.f;
    if (err == hipSuccess) err = hipEventElapsedTime(&ms, e0, e1);
    (void)hipEventDestroy(e0);
    (void)hipEventDestroy(e1);
    if (rc != RF_OK) return rc;
    if (err != hipSuccess) return fail(RF_ERR_HIP, std::string("rf_fp8_gemm_time: ") + hipGetErrorString(err));
    *us_per_launch = ms * 1e3f / iters;
    return RF_OK;
}

int rf_gemm_select_config(int m, int n, int k, rf_gemm_config *out) {
    g_last_error.clear();
    if (!out) return fail(RF_ERR_NULL_POINTER, "out is null");
    if (m < 1 || n < 1 || k < rf::BK || k % rf::BK != 0) return fail(RF_ERR_BAD_SHAPE, "unsupported shape");
    State &s = state();
    std::lock_guard<std::mutex> lock(shared().mu);
    int rc = ensure_device_info(s);
    if (rc != RF_OK) return rc;
    plan_of_shape(m, n, k, s.num_cu, out);
    return RF_OK;
}

int rf_gemm_plan_for(int m, int n, int k, int num_cu, rf_gemm_config *out) {
    g_last_error.clear();
    if (!out) return fail(RF_ERR_NULL_POINTER, "out is null");
    if (m < 1 || n < 1 || k < rf::BK || k % rf::BK != 0 || num_cu < 1) return fail(RF_ERR_BAD_SHAPE, "unsupported shape");
    std::lock_guard<std::mutex> lock(shared().mu);
    plan_of_shape(m, n, k, num_cu, out);
    return RF_OK;
}

int rf_gemm_load_plans(const char *path, int *count) {
    g_last_error.clear();
    if (!path) return fail(RF_ERR_NULL_POINTER, "path is null");
    std::lock_guard<std::mutex> lock(shared().mu);
    const size_t before = shared().user_plans.size();
    int rc = parse_plans(path, shared().user_plans);
    if (rc != RF_OK) return rc;
    shared().plan_generation++;
    if (count) *count = (int)(shared().user_plans.size() - before);
    return RF_OK;
}

void rf_gemm_clear_plans(void) {
    std::lock_guard<std::mutex> lock(shared().mu);
    shared().user_plans.clear();
    shared().plan_generation++;
}

int rf_gemm_num_variants(void) { return kNumVariants; }

int rf_gemm_variant_info(int variant, int *block_m, int *block_n, int *waves_m, int *waves_n, int *lds_bytes) {
    if (variant < 0 || variant >= kNumVariants) return RF_ERR_BAD_CONFIG;
    const Variant &v = kVariants[variant];
    if (block_m) *block_m = v.bm;
    if (block_n) *block_n = v.bn;
    if (waves_m) *waves_m = v.waves_m;
    if (waves_n) *waves_n = v.waves_n;
    if (lds_bytes) *lds_bytes = v.lds_bytes();
    return RF_OK;
}

int rf_gemm_variant_k_groups(int variant) {
    return variant >= 0 && variant < kNumVariants ? kVariants[variant].k_groups : 0;
}

int rf_gemm_variant_kind(int variant) {
    if (variant < 0 || variant >= kNumVariants) return -1;
    return kVariants[variant].is_fewrows() ? RF_VARIANT_KIND_FEW_ROWS : kVariants[variant].is_any_tile() ? RF_VARIANT_KIND_ANY_ALIGNMENT : RF_VARIANT_KIND_TILE;
}

int rf_gemm_variant_has_persistent(int variant) {
    return variant >= 0 && variant < kNumVariants && kVariants[variant].persistent != nullptr;
}

int rf_gemm_variant_has_stream_k(int variant) {
    return variant >= 0 && variant < kNumVariants && kVariants[variant].streamk != nullptr;
}

size_t rf_gemm_workspace_bytes(int m, int n, int k) {
    rf_gemm_config cfg;
    if (rf_gemm_select_config(m, n, k, &cfg) != RF_OK) return 0;
    State &s = state();
    if (cfg.variant < 0 && fewrows_ok(m, n)) fewrows_plan(m, n, k, s.num_cu, n % 16 != 0, &cfg);   // as launch_locked
    if (cfg.variant < 0) return 0;
    const Variant &v = kVariants[cfg.variant];
    if (cfg.stream_k == RF_SCHEDULE_STREAM_K) return (size_t)2 * s.num_cu * v.bm * v.bn * sizeof(float);
    const int qk = k / rf::BK, parts = ceil_div(qk, ceil_div(qk, cfg.split_k));
    if (parts <= 1) return 0;
    if (cfg.variant >= kFirstFewRows) return fewrows_slot_bytes(v, m, n, parts);   // (whole tiles: a little more than variants 28 to 30 need)
    // a ragged shape runs (and splits K) at its padded size; its staging copies live in a buffer of their own
    const size_t mp = m < 16 ? 16 : (m + 15) / 16 * 16, np = n < 16 ? 16 : (n + 15) / 16 * 16;
    return mp * np * sizeof(float) * parts;
}

int rf_gemm_init(size_t workspace_bytes) {
    g_last_error.clear();
    State &s = state();
    std::lock_guard<std::mutex> lock(shared().mu);
    int rc = ensure_device_info(s);
    if (rc != RF_OK) return rc;
    if (workspace_bytes == 0) return RF_OK;
    // a buffer set that belongs to no stream yet: the first stream that needs one takes it over
    StreamBuffers *sb = nullptr;
    rc = buffers_of(s, (hipStream_t)kUnboundStream, &sb);
    if (rc != RF_OK) return rc;
    Mem mem{s, sb};
    float *ws = nullptr;
    return mem.workspace(workspace_bytes, &ws);
}

void rf_gemm_destroy(void) {
    State &s = state();
    std::lock_guard<std::mutex> lock(shared().mu);
    if (!s.buffers.empty() || !s.retired.empty()) (void)hipDeviceSynchronize();   // launches may still use them
    for (StreamBuffers &b : s.buffers) {
        if (b.ws) (void)hipFree(b.ws);
        if (b.pad) (void)hipFree(b.pad);
    }
    // a fresh start also after launches that overlapped on a queue's counters (every other use leaves zeros behind)
    if (!s.buffers.empty()) {
        (void)hipMemset(s.counters, 0, s.buffers.size() * sizeof(CounterSet));
        (void)hipDeviceSynchronize();
    }
    s.buffers.clear();
    for (void *p : s.retired) (void)hipFree(p);
    s.retired.clear();
    std::lock_guard<std::mutex> ev_lock(s.ev_mu);
    for (auto &p : s.free_events) {
        (void)hipEventDestroy(p.first);
        (void)hipEventDestroy(p.second);
    }
    s.free_events.clear();
}

const char *rf_gemm_last_error(void) { return g_last_error.c_str(); }

}  // extern "C"

namespace {
// Up to this many elements the activations' quantiser works in 16-row pieces instead of 128-row blocks (both measured at
// quantize_rows16: the line lies between 7 and 10 million, within 8 % either way).
constexpr double kQuantRows16Elements = 1.0e7;
// rows x K source (row-major, K contiguous) -> fp8 [K][rows] + scales; see quantize_kernels.h
template <bool PER_ROW, bool IN_BF16>
int launch_quantize(const void *x, int rows, int k, void *out, float *scales, hipStream_t stream) {
    g_last_error.clear();
    if (rows < 1 || k < rf::BK || k % rf::BK != 0)
        return fail(RF_ERR_BAD_SHAPE, "unsupported shape rows=" + std::to_string(rows) + " K=" + std::to_string(k) +
                                          " (need rows>=1, K a positive multiple of 128)");
    if (!x || !out || !scales) return fail(RF_ERR_NULL_POINTER, "null device pointer");
    if ((uintptr_t)x % 16 != 0 || (uintptr_t)scales % 4 != 0)
        return fail(RF_ERR_BAD_CONFIG, "source must be 16-byte aligned, scales 4-byte aligned");
    State &s = state();
    {
        std::lock_guard<std::mutex> lock(shared().mu);
        int rc = ensure_device_info(s);
        if (rc != RF_OK) return rc;
    }
    if (PER_ROW && (double)rows * k <= kQuantRows16Elements) {
        const int blocks = k / rf::BK;
        if (blocks % rf::NUM_XCD != 0 && rows >= 128)
            enqueue((rf::quantize_rows16<IN_BF16, true>), dim3(ceil_div(ceil_div(rows, 128) * blocks, rf::NUM_XCD) * 8 * rf::NUM_XCD),
                    dim3(256), 0, stream, x, rows, k, (uint8_t *)out, scales);
        else
            enqueue((rf::quantize_rows16<IN_BF16, false>), dim3(blocks, ceil_div(rows, 16)), dim3(256), 0, stream, x, rows, k,
                    (uint8_t *)out, scales);
        RF_HIP(hipGetLastError());
        return RF_OK;
    }
    const bool vector_store = rows % 16 == 0 && (uintptr_t)out % 16 == 0;
    const int row_blocks = ceil_div(rows, 128);
    dim3 grid(k / rf::BK, row_blocks);
    enqueue((rf::quantize_block128<PER_ROW, IN_BF16>), grid, dim3(rf::QuantShape<IN_BF16>::NT), 0, stream, x, rows,
            k, (uint8_t *)out, scales, PER_ROW ? rows : row_blocks, vector_store);
    RF_HIP(hipGetLastError());
    return RF_OK;
}
}  // namespace

namespace {
typedef void (*grouped_kernel_t)(const uint8_t *, const uint8_t *, const float *, const float *, uint16_t *, int, int, int,
                                 int, const rf::GroupTable);
struct GroupedVariant {
    int bm, bn, threads, lds;
    grouped_kernel_t kernel;
    bool mixed;          // 256-row tiles plus one shorter tile for what is left over (one 128-row tile for at most 128
                         // rows; the queue form: 64, 128, 192 or 256 rows)
    bool queue = false;  // resident workgroups that take tiles from per-XCD queues (gemm_fp8_blockscale_grouped_queue)
    bool fewrows = false;  // fp8_gemm_fewrows.h: groups may start at any row of a
    grouped_kernel_t streamed = nullptr;   // few-rows strips: the kernel whose weights carry the non-temporal hint
    // row tiles of a group of `rows` rows
    int tiles_m(int rows) const {
        if (!mixed) return ceil_div(rows, bm);
        return rows / 256 + (rows % 256 > 0 ? 1 : 0);
    }
};

#define RF_GROUPED(BM, BN, WM, WN, NS) \
    GroupedVariant { BM, BN, WM *WN * 64, rf::TileGeom<BM, BN, WM, WN, NS>::LDS_BYTES, rf::gemm_fp8_blockscale_grouped<BM, BN, WM, WN, NS>, false }
#define RF_GROUPED_STRIPS(TM, NW, DEPTH, WAVES_PER_SIMD)                                            \
    GroupedVariant { 16 * TM, 128 * NW, 64 * NW, NW *rf::BK * 16 * (TM + 8),                        \
                     rf::gemm_fp8_blockscale_grouped_strips<TM, 8, NW, DEPTH, WAVES_PER_SIMD, false>, false, false, true, \
                     rf::gemm_fp8_blockscale_grouped_strips<TM, 8, NW, DEPTH, WAVES_PER_SIMD, true> }
constexpr int kMixedLds = rf::TileGeom<256, 256, 2, 4>::LDS_BYTES > rf::TileGeom<128, 256, 2, 4, 3>::LDS_BYTES
                              ? rf::TileGeom<256, 256, 2, 4>::LDS_BYTES : rf::TileGeom<128, 256, 2, 4, 3>::LDS_BYTES;
const GroupedVariant kGroupedVariants[] = {
    RF_GROUPED(256, 256, 2, 4, 2), RF_GROUPED(128, 256, 2, 4, 3), RF_GROUPED(128, 128, 4, 2, 3), RF_GROUPED(128, 64, 2, 1, 2),
    GroupedVariant{256, 256, 512, kMixedLds, rf::gemm_fp8_blockscale_grouped_mixed, true},
    GroupedVariant{256, 256, 512, rf::kQueueLds, nullptr, true, true},
    RF_GROUPED_STRIPS(1, 2, 2, 1),    // 6: 16 rows, two waves of 128 columns
    RF_GROUPED_STRIPS(1, 1, 1, 2),    // 7: 16 rows, one wave
    RF_GROUPED_STRIPS(2, 1, 1, 1),    // 8: 32 rows, one wave
    GroupedVariant{16, 64, 512, 8 * rf::BK * 16 * 5, rf::gemm_fp8_blockscale_grouped_ksplit<1, 4, 8, 1, 4>, false, false, true},   // 9: 16 rows, K split between eight waves
    RF_GROUPED_STRIPS(1, 4, 1, 2)};   // 10: 16 rows, four waves
constexpr int kGroupedMixed = 4, kGroupedQueue = 5, kGroupedFewRows = 6;
// Estimated time of a 256-column tile of the queue form by its height in units of 64 rows, relative to a 256-row tile
constexpr double kQueueTileCost[5] = {0.0, 0.68, 0.75, 0.97, 1.0};
constexpr int kNumGroupedVariants = sizeof(kGroupedVariants) / sizeof(kGroupedVariants[0]);

long grouped_tiles(const GroupedVariant &v, const int *row_offsets, int groups, int n) {
    long t = 0;
    for (int g = 0; g < groups; g++) t += (long)v.tiles_m(row_offsets[g + 1] - row_offsets[g]) * ceil_div(n, v.bn);
    return t;
}
}  // namespace

namespace {
// The few-rows form for these groups, or -1: groups of at most 16 rows (variants 6, 7, 9 and 10) or 32 (variant 8); more rows
// would stream the weights once per row block. Estimated time in us: the stream of the weights at the rate the form reaches
// once the chip is full, or the chain of one wave's K blocks. Measured on 52 layouts (8 to 64 groups, 16 to 900 rows,
// N x K = 2048 x 7168, 4096 x 7168, 7168 x 2048, 4096 x 2048) against the tiled forms with their staging copy: up to 50 %
// faster where this picks one, 14 % on average, never slower; beyond 1 GB of weights, or max_rounds rounds of resident workgroups,
// the tiled forms' steady state is as good or better (64 groups of 64 rows in all, 4096 x 7168: 306 us here, 284 tiled; of
// 300 rows, 7168 x 2048: 210 against 191).
int choose_grouped_fewrows(const int *row_offsets, int groups, int n, int k, int num_cu) {
    int most = 0, busy = 0;
    for (int g = 0; g < groups; g++) {
        const int rows = row_offsets[g + 1] - row_offsets[g];
        most = std::max(most, rows);
        busy += rows > 0;
    }
    const double bytes = (double)busy * n * k;
    if (most < 1 || most > 32 || n % 16 != 0 || bytes > 1.0e9 || !fewrows_ok((long)row_offsets[groups] + 16 * groups, n)) return -1;
    struct Form { int variant, wgs_per_cu; double max_rounds, start, per_k_block, bytes_per_us; };
    const Form forms[] = {{6, 2, 3.0, 4.0, 1.0, 5.1e6}, {7, 8, 1.0, 3.5, 0.93, 4.6e6}, {8, 4, 2.0, 3.0, 1.2, 5.0e6},
                          {9, 2, 1.0, 3.0, 0.0, 3.3e6}, {10, 2, 2.0, 4.0, 1.6, 5.4e6}};
    int best = -1;
    double best_t = 0;
    for (const Form &f : forms) {
        const GroupedVariant &v = kGroupedVariants[f.variant];
        const double rounds = (double)busy * ceil_div(n, v.bn) / (f.wgs_per_cu * num_cu);
        if (most > v.bm || rounds > f.max_rounds) continue;
        // strips of 512 columns: only where there is nearly one for every compute unit (8 % faster than 256 columns then; with
        // 128 of them for 256 units a third slower)
        if (f.variant == 10 && (long)busy * ceil_div(n, v.bn) * 8 < 7L * num_cu) continue;
        const double t = std::max(f.start + f.per_k_block * (k / rf::BK), 3.0 + bytes / f.bytes_per_us * 256.0 / num_cu);
        if (best < 0 || t < best_t) { best = f.variant; best_t = t; }
    }
    return best;
}

// The automatic choice of rf_fp8_gemm_grouped (variant = -1) for groups of these sizes on a device with num_cu compute units.
int choose_grouped_variant(const int *row_offsets, int groups, int n, int k, int num_cu) {
    const int few = choose_grouped_fewrows(row_offsets, groups, n, k, num_cu);
    if (few >= 0) return few;
    // the largest tile that still gives every CU a workgroup; failing that, the one with the most workgroups
    int variant = -1;
    long most = -1;
    int most_v = 0;
    for (int v = 0; v < kGroupedFewRows && variant < 0; v++) {
        const long t = grouped_tiles(kGroupedVariants[v], row_offsets, groups, n);
        if (t >= num_cu) variant = v;
        if (t > most) { most = t; most_v = v; }
    }
    if (variant < 0) variant = most_v;
    // Too few 128 x 256 tiles for every CU: a launch is the chain of one tile's K blocks, shortest for the 128 x 128 tiles (eight
    // waves, three stages), so smaller tiles pay only while they are alone on their CU. us on N x K = 2048 x 7168 with tiles of
    // 64, 128 and 256 columns: 1000 rows in 8 groups 92, 48, 57; 3000 rows (more 128 x 128 tiles than CUs) 176, 103, 81; 4096 x
    // 2048: 355 rows in 8 groups -, 19, 21. With four waves and two stages the 128 x 128 tiles took 62, 95 and 23. (Below
    // K = 2048 not measured.)
    if ((variant == 2 || variant == 3) && k >= 2048)
        return grouped_tiles(kGroupedVariants[2], row_offsets, groups, n) <= num_cu ? 2 : 1;
    if (variant == 1) variant = 0;      // 128-row tiles fill the chip: the 256-wide family, chosen below
    // Enough tiles for the 256-wide family (128-row tiles would give every CU one): 256-row tiles, 128-row tiles
    // (three stages) or the mixed form, by a
    // small model of what was measured (N = 4096, K = 7168, twelve group layouts). A tile costs its compute
    // (91 for 256 rows, 52 for 128, arbitrary units) plus a share of streaming its column tile of the group's
    // weights (36, divided among the row tiles that use it: they run side by side on one XCD); the launch takes
    // as many rounds of one tile per CU as the tile count needs, a last partial round counting 0.6 + 0.4 x its
    // fill. Round counts decide most cases: 32 uneven groups of 16..816 rows are 816 mixed tiles (3.19 rounds,
    // 369 us) or 1280 tiles of 128 rows (5.00 rounds, 342 us); 20 groups of 384 rows 287 against 246 us; 64 groups
    // of 16..176 rows 408 against 447 us. On the twelve layouts the choice is 0.9 % slower than the best of the
    // three on average, 8 % at worst (always taking the mixed form: 2.6 % and 17 %).
    if (variant == 0) {
        const int tiles_n256 = ceil_div(n, 256);
        double best_t = 0;
        for (int cand : {0, 1, kGroupedMixed}) {
            double cost = 0;
            long items = 0;
            for (int g = 0; g < groups; g++) {
                const int rows = row_offsets[g + 1] - row_offsets[g];
                if (rows == 0) continue;
                int big, small;
                if (cand == 0) { big = ceil_div(rows, 256); small = 0; }
                else if (cand == 1) { big = 0; small = ceil_div(rows, 128); }
                else { big = rows / 256 + (rows % 256 > 128 ? 1 : 0); small = rows % 256 > 0 && rows % 256 <= 128 ? 1 : 0; }
                cost += tiles_n256 * (91.0 * big + 52.0 * small + 36.0);      // 36 / t for each of the t row tiles
                items += (long)tiles_n256 * (big + small);
            }
            const double rounds_exact = (double)items / num_cu;
            const double full = std::floor(rounds_exact), frac = rounds_exact - full;
            const double t = (full + (frac > 0 ? 0.6 + 0.4 * frac : 0.0)) * cost / (double)items;
            if (best_t == 0 || t < best_t) { best_t = t; variant = cand; }
        }
        // The queue form (tiles of 64 to 256 rows, resident workgroups): where its shorter last tiles save at least
        // 7 % of the rows the chosen tiles compute and it has enough items to go round (a few more than CUs; 2.5 per
        // CU when K is below 4096 and an item is short against the cost of drawing it; K = 7168 and 1.1 to 1.4 items per
        // CU: 166 -> 155, 178 -> 164, 162 -> 150 us, with no more items than CUs 107 -> 111). Measured on 68 layouts (8 to 128 groups of
        // uniform, exponential or equal sizes; N x K = 4096 x 7168, 7168 x 2048, 2048 x 7168, 4096 x 2048) against
        // the best of the four 256-wide forms: this rule 0.8 % behind on average, 11 % at worst; never the queue form
        // 4.6 % and 16 %; the queue form on row savings alone 2.2 % and 41 % (16 groups of 16..384 rows at
        // N = 2048: 170 items for 256 CUs, 91 against 65 us with 128-row tiles).
        long rows_chosen = 0, rows_queue = 0, items_queue = 0;
        for (int g = 0; g < groups; g++) {
            const int rows = row_offsets[g + 1] - row_offsets[g];
            rows_queue += ceil_div(rows, 64) * 64;
            items_queue += (long)ceil_div(rows, 256) * tiles_n256;
            rows_chosen += variant == 0 ? ceil_div(rows, 256) * 256 : variant == 1 ? ceil_div(rows, 128) * 128
                           : rows / 256 * 256 + (rows % 256 == 0 ? 0 : rows % 256 <= 128 ? 128 : 256);
        }
        const long items_needed = k >= 4096 ? 17L * num_cu / 16 : 5L * num_cu / 2;
        if (rows_queue * 100 <= rows_chosen * 93 && items_queue >= items_needed) variant = kGroupedQueue;
    }
    return variant;
}
// prepadded: a and as already hold every group from a multiple of 16 rows on (the layout rf_quantize_a_grouped_* writes
// and rf_grouped_padded_offsets describes); otherwise they hold the groups back to back as row_offsets says.
int grouped_gemm(const void *a, const void *b, const float *as, const float *bs, void *c, const int *row_offsets,
                 int groups, int n, int k, int variant, hipStream_t stream, bool prepadded) {
    g_last_error.clear();
    if (!row_offsets) return fail(RF_ERR_NULL_POINTER, "row_offsets is null");
    if (groups < 1 || groups > rf::kMaxGroups)
        return fail(RF_ERR_BAD_SHAPE, "groups must be between 1 and " + std::to_string(rf::kMaxGroups));
    if (n < 1 || k < rf::BK || k % rf::BK != 0 || row_offsets[0] != 0)
        return fail(RF_ERR_BAD_SHAPE, "unsupported shape (need N>=1, K a positive multiple of 128, row_offsets[0] == 0)");
    for (int g = 0; g < groups; g++)
        if (row_offsets[g + 1] < row_offsets[g]) return fail(RF_ERR_BAD_SHAPE, "row_offsets must not decrease");
    const int m_total = row_offsets[groups];
    if (m_total == 0) return RF_OK;
    if (!a || !b || !as || !bs || !c) return fail(RF_ERR_NULL_POINTER, "null device pointer");
    if (variant >= kNumGroupedVariants || variant < -1) return fail(RF_ERR_BAD_CONFIG, "no such grouped variant");
    State &s = state();
    std::lock_guard<std::mutex> lock(shared().mu);
    int rc = ensure_device_info(s);
    if (rc != RF_OK) return rc;
    if (!s.grouped_attrs_set) {
        for (const GroupedVariant &v : kGroupedVariants)
            for (grouped_kernel_t f : {v.kernel, v.streamed})
                if (f) RF_HIP(hipFuncSetAttribute((const void *)f, hipFuncAttributeMaxDynamicSharedMemorySize, v.lds));
        RF_HIP(hipFuncSetAttribute((const void *)rf::gemm_fp8_blockscale_grouped_queue,
                                   hipFuncAttributeMaxDynamicSharedMemorySize, rf::kQueueLds));
        s.grouped_attrs_set = true;
    }
    const int qk = k / rf::BK, qn = ceil_div(n, 128);
    const bool direct = n % 16 == 0 && ((uintptr_t)b % 16) == 0 && ((uintptr_t)c % 16) == 0;
    bool stage = ((uintptr_t)a % 16) != 0;
    for (int g = 0; g <= groups; g++) stage = stage || row_offsets[g] % 16 != 0;
    if (prepadded) {
        if (!direct || ((uintptr_t)a % 16) != 0)
            return fail(RF_ERR_BAD_CONFIG, "the padded layout needs N % 16 == 0 and 16-byte aligned a, b and c");
        stage = false;
    }
    if (!direct || (stage && (double)m_total * n * k < kPadThresholdMacs)) {
        // ragged N, unaligned weights or output, or next to no work: the bounds-checked kernel, one launch per
        // non-empty group
        for (int g = 0; g < groups; g++) {
            const int r0 = row_offsets[g], rows = row_offsets[g + 1] - r0;
            if (rows == 0) continue;
            dim3 grid(ceil_div(n, 16), ceil_div(rows, 16));
            enqueue(rf::gemm_fp8_blockscale_checked, grid, dim3(64), 0, stream, (const uint8_t *)a + r0,
                    (const uint8_t *)b + (size_t)g * k * n, as + r0, bs + (size_t)g * qk * qn,
                    (uint16_t *)c + (size_t)r0 * n, rows, m_total, n, k);
            RF_HIP(hipGetLastError());
        }
        return RF_OK;
    }
    if (variant < 0) {
        variant = choose_grouped_variant(row_offsets, groups, n, k, s.num_cu);
        if (kGroupedVariants[variant].queue) {
            // no counters to be had (a stream under capture that would have to take over another stream's set): the form
            // without queues, whose results are the same to the bit
            Mem mem{s};
            mem.stream = stream;
            CounterSet *counters = nullptr;
            if (mem.counters(&counters) != RF_OK) {
                (void)hipGetLastError();
                g_last_error.clear();
                variant = kGroupedMixed;
            }
        }
    }
    const GroupedVariant &v = kGroupedVariants[variant];
    if (v.fewrows && !fewrows_ok((long)m_total + 16 * groups, n))
        return fail(RF_ERR_BAD_CONFIG, "the few-rows forms need fewer than 2^25 rows and columns");
    rf::GroupTable table;
    int m_rows = m_total;                      // rows of the A matrix the kernel reads
    if (stage && !v.fewrows) {
        // Group sizes that are not multiples of 16 (token counts per expert never are): A and a_scale are copied
        // into the staging buffer with every group starting at a multiple of 16, the kernel reads those and writes
        // each group's true rows straight into the caller's C. Costs one pass over A; the bounds-checked kernel
        // per group would be 10 to 30 times slower than the tiled one.
        // Starts at a multiple of 128, whole cache lines (a tile's 128-byte pieces of A are then one line each, not two), where
        // that makes the copy at most an eighth longer. us: 3623 rows in 8 groups, 7168 x 2048, 94.2 -> 88.4; 3077 in 16,
        // 4096 x 7168, 167.0 -> 159.5; 1076 in 8, the same, 85.3 -> 81.9; a copy a fifth longer lost up to 2 %.
        long by16 = 0, by128 = 0;
        for (int g = 0; g < groups; g++) {
            by16 += (row_offsets[g + 1] - row_offsets[g] + 15) / 16 * 16;
            by128 += (long)ceil_div(row_offsets[g + 1] - row_offsets[g], 128) * 128;
        }
        const int unit = by128 * 8 <= by16 * 9 && by128 < (1L << 30) ? 128 : 16;
        int at = 0;
        for (int g = 0; g < groups; g++) {
            table.row_start[g] = at;
            at += ceil_div(row_offsets[g + 1] - row_offsets[g], unit) * unit;
        }
        for (int g = groups; g <= rf::kMaxGroups; g++) table.row_start[g] = at;
        for (int g = 0; g <= rf::kMaxGroups; g++) table.out_row_start[g] = row_offsets[g < groups ? g : groups];
        m_rows = at;
        const size_t a_bytes = ((size_t)k * m_rows + 255) / 256 * 256;
        Mem mem{s};
        mem.stream = stream;
        uint8_t *pad = nullptr;
        rc = mem.pad(a_bytes + (size_t)qk * m_rows * sizeof(float), &pad);
        if (rc != RF_OK) return rc;
        launch_pad_a_and_scales(a, as, 0, m_total, m_rows, k, groups, pad, (float *)(pad + a_bytes), table, stream);
        RF_HIP(hipGetLastError());
        a = pad;
        as = (const float *)(pad + a_bytes);
    } else if (prepadded) {
        int at = 0;
        for (int g = 0; g < groups; g++) {
            table.row_start[g] = at;
            at += (row_offsets[g + 1] - row_offsets[g] + 15) / 16 * 16;
        }
        for (int g = groups; g <= rf::kMaxGroups; g++) table.row_start[g] = at;
        for (int g = 0; g <= rf::kMaxGroups; g++) table.out_row_start[g] = row_offsets[g < groups ? g : groups];
        m_rows = at;
    } else {
        for (int g = 0; g <= rf::kMaxGroups; g++)
            table.row_start[g] = table.out_row_start[g] = row_offsets[g < groups ? g : groups];
    }
    const int tiles_n = ceil_div(n, v.bn);
    int tiles = 0, busy = 0;
    for (int g = 0; g < groups; g++) {
        table.tile_start[g] = tiles;
        tiles += v.tiles_m(row_offsets[g + 1] - row_offsets[g]) * tiles_n;
        busy += row_offsets[g + 1] > row_offsets[g];
    }
    const bool stream_b = rf::grouped_weights_streamed((double)busy * n * k, v.queue, v.bn);
    for (int g = groups; g <= rf::kMaxGroups; g++) table.tile_start[g] = tiles;
    if (v.queue) {
        // The line of items and its eight pieces. Estimated time of a group = column tiles x (256-row tiles + what
        // its last, shorter tile costs relative to one). With at least two groups per XCD: whole groups per queue,
        // each group to the queue with the least work so far, the longest group first (so every queue's groups are in
        // falling order). Fewer groups: the groups as they come, cut where the estimated time reaches each eighth.
        auto rows_of = [&](int g) { return row_offsets[g + 1] - row_offsets[g]; };
        auto cost_of_tile = [&](int rows, int i) { return i < rows / 256 ? 1.0 : kQueueTileCost[(rows % 256 + 63) / 64]; };
        auto cost_of = [&](int g) {
            return tiles_n * (rows_of(g) / 256 + kQueueTileCost[(rows_of(g) % 256 + 63) / 64]);
        };
        rf::GroupQueues queues;
        std::vector<int> order(groups);
        for (int g = 0; g < groups; g++) order[g] = g;
        int piece_groups[rf::NUM_XCD + 1] = {0};          // positions of the line where the pieces start, if whole groups
        const bool whole_groups = groups >= 2 * rf::NUM_XCD;
        if (whole_groups) {
            std::stable_sort(order.begin(), order.end(), [&](int x, int y) { return cost_of(x) > cost_of(y); });
            std::vector<int> lists[rf::NUM_XCD];
            double load[rf::NUM_XCD] = {0};
            for (int g : order) {
                int least = 0;
                for (int x = 1; x < rf::NUM_XCD; x++)
                    if (load[x] < load[least]) least = x;
                lists[least].push_back(g);
                load[least] += cost_of(g);
            }
            int p = 0;
            for (int x = 0; x < rf::NUM_XCD; x++) {
                piece_groups[x] = p;
                for (int g : lists[x]) order[p++] = g;
            }
            piece_groups[rf::NUM_XCD] = p;
        }
        int items = 0;
        for (int p = 0; p < groups; p++) {
            queues.order[p] = (uint8_t)order[p];
            table.tile_start[p] = items;
            items += v.tiles_m(rows_of(order[p])) * tiles_n;
        }
        for (int p = groups; p <= rf::kMaxGroups; p++) table.tile_start[p] = items;
        for (int p = groups; p < rf::kMaxGroups; p++) queues.order[p] = 0;
        if (whole_groups) {
            for (int x = 0; x <= rf::NUM_XCD; x++) queues.piece_start[x] = table.tile_start[piece_groups[x]];
        } else {
            double total = 0, before = 0;
            for (int g = 0; g < groups; g++) total += cost_of(g);
            queues.piece_start[0] = 0;
            int piece = 1, item = 0;
            for (int g = 0; g < groups; g++) {
                const int tm = v.tiles_m(rows_of(g));
                for (int tn = 0; tn < tiles_n && tm > 0; tn++)
                    for (int i = 0; i < tm; i++, item++) {
                        while (piece < rf::NUM_XCD && before >= total * piece / rf::NUM_XCD) queues.piece_start[piece++] = item;
                        before += cost_of_tile(rows_of(g), i);
                    }
            }
            while (piece <= rf::NUM_XCD) queues.piece_start[piece++] = items;
        }
        queues.workgroups = s.num_cu >= rf::NUM_XCD ? s.num_cu / rf::NUM_XCD * rf::NUM_XCD : rf::NUM_XCD;
        if (tiles < queues.workgroups) queues.workgroups = ceil_div(tiles, rf::NUM_XCD) * rf::NUM_XCD;
        Mem mem{s};
        mem.stream = stream;
        CounterSet *counters = nullptr;
        rc = mem.counters(&counters);
        if (rc != RF_OK) return rc;
        enqueue(rf::gemm_fp8_blockscale_grouped_queue, dim3(queues.workgroups), dim3(v.threads), v.lds, stream,
                (const uint8_t *)a, (const uint8_t *)b, as, bs, (uint16_t *)c, m_rows, n, k, groups, table,
                queues, stream_b, counters->queue);
        RF_HIP(hipGetLastError());
        return RF_OK;
    }
    const grouped_kernel_t kernel = stream_b && v.streamed ? v.streamed : v.kernel;
    const int longest = ceil_div(tiles, rf::NUM_XCD);          // every XCD takes an eighth of the tiles, rounded
    enqueue(kernel, dim3(longest * rf::NUM_XCD), dim3(v.threads), v.lds, stream, (const uint8_t *)a,
            (const uint8_t *)b, as, bs, (uint16_t *)c, m_rows, n, k, groups, table);
    RF_HIP(hipGetLastError());
    return RF_OK;
}

template <bool IN_BF16>
int quantize_a_grouped(const void *x, const int *row_offsets, int groups, int k, void *a, float *as, hipStream_t stream) {
    g_last_error.clear();
    if (!row_offsets) return fail(RF_ERR_NULL_POINTER, "row_offsets is null");
    if (groups < 1 || groups > rf::kQuantMaxGroups || k < rf::BK || k % rf::BK != 0 || row_offsets[0] != 0)
        return fail(RF_ERR_BAD_SHAPE, "unsupported shape (need 1 <= groups <= 256, K a positive multiple of 128, row_offsets[0] == 0)");
    rf::QuantGroups tab;
    int at = 0;
    for (int g = 0; g < groups; g++) {
        if (row_offsets[g + 1] < row_offsets[g]) return fail(RF_ERR_BAD_SHAPE, "row_offsets must not decrease");
        tab.pad_start[g] = at;
        tab.src_start[g] = row_offsets[g];
        at += (row_offsets[g + 1] - row_offsets[g] + 15) / 16 * 16;
    }
    for (int g = groups; g <= rf::kQuantMaxGroups; g++) { tab.pad_start[g] = at; tab.src_start[g] = row_offsets[groups]; }
    tab.groups = groups;
    for (int blk = 0, g = 0; blk < rf::kQuantBlockTable; blk++) {        // last g with pad_start[g] <= 128 * blk
        while (g + 1 < groups && tab.pad_start[g + 1] <= 128 * blk) g++;
        tab.block_group[blk] = (unsigned short)g;
    }
    if (at == 0) return RF_OK;
    if (!x || !a || !as) return fail(RF_ERR_NULL_POINTER, "null device pointer");
    if ((uintptr_t)x % 16 != 0 || (uintptr_t)a % 16 != 0 || (uintptr_t)as % 4 != 0)
        return fail(RF_ERR_BAD_CONFIG, "source and a must be 16-byte aligned, scales 4-byte aligned");
    State &s = state();
    {
        std::lock_guard<std::mutex> lock(shared().mu);
        int rc = ensure_device_info(s);
        if (rc != RF_OK) return rc;
    }
    if ((double)at * k <= kQuantRows16Elements)
        enqueue((rf::quantize_rows16_grouped<IN_BF16>), dim3(k / rf::BK, at / 16), dim3(256), 0, stream, x, at, k,
                (uint8_t *)a, as, tab);
    else
        enqueue((rf::quantize_block128_grouped<IN_BF16>), dim3(k / rf::BK, ceil_div(at, 128)),
                dim3(rf::QuantShape<IN_BF16>::NT), 0, stream, x, at, k, (uint8_t *)a, as, tab);
    RF_HIP(hipGetLastError());
    return RF_OK;
}
}  // namespace

extern "C" {

int rf_fp8_gemm_grouped(const void *a, const void *b, const float *as, const float *bs, void *c, const int *row_offsets,
                        int groups, int n, int k, int variant, hipStream_t stream) {
    return grouped_gemm(a, b, as, bs, c, row_offsets, groups, n, k, variant, stream, false);
}

int rf_fp8_gemm_grouped_padded(const void *a, const void *b, const float *as, const float *bs, void *c,
                               const int *row_offsets, int groups, int n, int k, int variant, hipStream_t stream) {
    return grouped_gemm(a, b, as, bs, c, row_offsets, groups, n, k, variant, stream, true);
}

int rf_grouped_variant_for(const int *row_offsets, int groups, int n, int k, int num_cu, int *variant) {
    g_last_error.clear();
    if (!row_offsets || !variant) return fail(RF_ERR_NULL_POINTER, "row_offsets or variant is null");
    if (groups < 1 || groups > rf::kMaxGroups || n < 1 || k < rf::BK || k % rf::BK != 0 || num_cu < 1 || row_offsets[0] != 0)
        return fail(RF_ERR_BAD_SHAPE, "unsupported shape (need 1 <= groups <= 256, N >= 1, K a positive multiple of 128, "
                                      "a compute unit count, row_offsets[0] == 0)");
    for (int g = 0; g < groups; g++)
        if (row_offsets[g + 1] < row_offsets[g]) return fail(RF_ERR_BAD_SHAPE, "row_offsets must not decrease");
    *variant = choose_grouped_variant(row_offsets, groups, n, k, num_cu);
    return RF_OK;
}

int rf_grouped_padded_offsets(const int *row_offsets, int groups, int *padded_offsets) {
    g_last_error.clear();
    if (!row_offsets || !padded_offsets) return fail(RF_ERR_NULL_POINTER, "null pointer");
    if (groups < 1 || groups > rf::kMaxGroups || row_offsets[0] != 0) return fail(RF_ERR_BAD_SHAPE, "unsupported groups");
    int at = 0;
    for (int g = 0; g < groups; g++) {
        if (row_offsets[g + 1] < row_offsets[g]) return fail(RF_ERR_BAD_SHAPE, "row_offsets must not decrease");
        padded_offsets[g] = at;
        at += (row_offsets[g + 1] - row_offsets[g] + 15) / 16 * 16;
    }
    padded_offsets[groups] = at;
    return RF_OK;
}

int rf_quantize_a_grouped_f32(const float *x, const int *row_offsets, int groups, int k, void *a, float *as,
                              hipStream_t stream) {
    return quantize_a_grouped<false>(x, row_offsets, groups, k, a, as, stream);
}
int rf_quantize_a_grouped_bf16(const void *x, const int *row_offsets, int groups, int k, void *a, float *as,
                               hipStream_t stream) {
    return quantize_a_grouped<true>(x, row_offsets, groups, k, a, as, stream);
}

int rf_cast_f32_to_e4m3fn(const float *x, size_t count, void *out, hipStream_t stream) {
    g_last_error.clear();
    if (count == 0) return RF_OK;
    if (!x || !out) return fail(RF_ERR_NULL_POINTER, "null device pointer");
    if ((uintptr_t)x % 16 != 0 || (uintptr_t)out % 4 != 0)
        return fail(RF_ERR_BAD_CONFIG, "source must be 16-byte aligned, destination 4-byte aligned");
    enqueue(rf::cast_f32_to_e4m3fn, dim3((unsigned)((count + 1023) / 1024)), dim3(256), 0, stream, x,
            (uint8_t *)out, count);
    RF_HIP(hipGetLastError());
    return RF_OK;
}

int rf_quantize_a_f32(const float *x, int m, int k, void *a, float *as, hipStream_t stream) {
    return launch_quantize<true, false>(x, m, k, a, as, stream);
}
int rf_quantize_a_bf16(const void *x, int m, int k, void *a, float *as, hipStream_t stream) {
    return launch_quantize<true, true>(x, m, k, a, as, stream);
}
int rf_quantize_b_f32(const float *w, int n, int k, void *b, float *bs, hipStream_t stream) {
    return launch_quantize<false, false>(w, n, k, b, bs, stream);
}
int rf_quantize_b_bf16(const void *w, int n, int k, void *b, float *bs, hipStream_t stream) {
    return launch_quantize<false, true>(w, n, k, b, bs, stream);
}

void run(void *a, void *b, void *as, void *bs, void *c, int m, int n, int k, PerfMetrics *metrics,
         hipStream_t job_stream0) {
    TimerJob *job = nullptr;
    if (metrics) {
        job = new TimerJob();
        State &s = state();
        job->owner = &s;
        {
            std::lock_guard<std::mutex> lock(s.ev_mu);
            if (!s.free_events.empty()) {
                job->start = s.free_events.back().first;
                job->stop = s.free_events.back().second;
                s.free_events.pop_back();
            } else {
                job->start = job->stop = nullptr;
            }
        }
        if (!job->start && (hipEventCreate(&job->start) != hipSuccess || hipEventCreate(&job->stop) != hipSuccess)) {
            fprintf(stderr, "run: hipEventCreate failed\n");
            abort();
        }
        job->flop = 2.0 * m * n * k;
        job->time_ms = &metrics->entries[0].time;
        job->gflops = &metrics->entries[0].gflops;
        if (hipEventRecord(job->start, job_stream0) != hipSuccess) {
            fprintf(stderr, "run: hipEventRecord failed\n");
            abort();
        }
    }
    int rc = launch(a, b, (const float *)as, (const float *)bs, c, m, n, k, nullptr, job_stream0);
    if (rc != RF_OK) {
        if (rc == RF_ERR_BAD_SHAPE) printf("Error: Unsupported shape M=%d, K=%d, N=%d\n", m, k, n);
        fprintf(stderr, "Kernel execution failed.\n%s\n", g_last_error.c_str());
        fflush(stdout);
        abort();
    }
    if (job) {
        if (hipEventRecord(job->stop, job_stream0) != hipSuccess ||
            hipStreamAddCallback(job_stream0, timer_callback, job, 0) != hipSuccess) {
            fprintf(stderr, "run: could not enqueue the timing callback\n");
            abort();
        }
    }
}

}  // extern "C"

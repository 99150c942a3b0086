// extern "C" layer of the library: argument checks, kernel choice, workspace,
// launches.  Declarations and the reference interfaces they replace are in
// include/qgemm.h.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <memory>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <mutex>
#include <string>
#include <vector>

#include "aux_kernels.cuh"
#include "gemm_any.cuh"
#include "quant_kernels.cuh"
#include "selftest.cuh"
#include "variants.h"

using namespace qgemm;

#define QGEMM_EXPORT __attribute__((visibility("default")))

namespace {

// Scratch of the entry point that allocates nothing (qgemm_scaled_gemm_static): split-K partial planes,
// transposed block scales and transposed operands of one call.  One copy per device, held until the process
// ends; host code never uses the array's name as an address, only what hipGetSymbolAddress returned for the
// device that is current (static_scratch_locked).
constexpr size_t kStaticScratchBytes = QGEMM_STATIC_SCRATCH_BYTES;
static __device__ __align__(256) unsigned char scratch[kStaticScratchBytes];
constexpr int kMaxDevices = 64;
constexpr uint32_t kMaxGridY = 65535;

struct WsBlock {
    void *p = nullptr;
    size_t bytes = 0;
};
constexpr int kOwnBlocks = 3;
constexpr size_t kOwnBytes = (size_t)128 << 20;         // fits all but the largest calls, whose time hides an event
constexpr size_t kLeastBlock = (size_t)64 << 20;        // of the shared block, what a first call allocates

struct Context {
    std::mutex mu;
    bool ready = false;
    int device = -1;
    int num_cus = 256;
    // Workspace (split-K partial planes, transposed and packed operands and scales, quantiser partials): one shared block, which every
    // eager call makes as large as it needs, and kOwnBlocks blocks of kOwnBytes (or what was reserved), one each for the first streams that ask.  In its own
    // block a stream's calls follow one another as the stream has them.  The shared block is for calls that need more, for the streams beyond
    // those (and hipStreamPerThread, one handle for many streams), where there is no memory for another block, and for captured
    // calls; its eager users are ordered through ws_event: every call that
    // used it records the event on its stream when it has enqueued its launches, and a call on another stream waits for it first.
    // (Recording costs a call 4.3 - 5.4 us of host time, twice a launch, and the GPU a packet that the next launch waits for.  With
    // one block for all streams every call that used the workspace paid that, eager calls, us: quantise 50 x 5296 fp16 to int8 per
    // matrix 11.1 -> 8.0, forward and backward 505 x 531 x 1059 43.1 -> 37.0, fp8_mm 2080 x 4096 x 4096 50.6 -> 47.5.)
    // A shared block that is outgrown is replaced and kept in `retired` until qgemm_shutdown: launches
    // already enqueued and graphs already captured keep pointing at live memory.
    WsBlock ws;
    WsBlock ws_own[kOwnBlocks];
    hipStream_t ws_stream[kOwnBlocks] = {};    // whose they are
    int ws_owners = 0;
    bool ws_own_failed = false;                // there was no memory for one of them: no more are tried
    std::vector<void *> retired;
    hipEvent_t ws_event = nullptr;
    hipStream_t ws_last_stream = nullptr;
    bool ws_event_recorded = false;
    bool ws_shared_by_call = false;            // the running entry asked for the shared block
    long quant_wait = -2;       // microseconds its workgroups wait for one another; -1: per-matrix scales in two passes; -2: quant_wait_of
    struct QuantStream {
        hipStream_t stream;
        uint64_t last;                         // number of its last call
        bool whole_chip;                       // its kernels may run on every CU
        uint32_t launches;                     // of quant_whole_matrix_kernel from this place, which number them
    } quant_streams[2] = {};                   // see may_exchange_maxima
    uint64_t quant_calls = 0;
    bool static_call = false;                  // the running entry takes its workspace from the static scratch
    void *static_ptr[kMaxDevices] = {};        // device address of `scratch`, per device
    std::string force_config;   // name of a row of the variant tables, empty = heuristic (qgemm_force_config)
    long force_split = 0;       // 0 = heuristic
    long force_group_m = 0;     // 0 = default
#if QGEMM_DEBUG_BUILD
    long dbg_ptr = 0;           // measurement builds: device buffer for the kernels' time stamps (GemmArgs::dbg_cycles)
#endif
    long as_groups = 1;         // 0: no copies of four K blocks of a_scale: one block per copy on the rows with two K groups (see run_nt), a
                                // transposed copy of a_scale for the row with copying waves (see settle_scale_layout)
    long small_tiles = 1;       // 0: 17 .. 256 rows never go to several row tiles of the skinny-M kernel in place of a K split (and up to 400
                                // rows follow the rules, as the estimate likes such tiles)
    long few_rows = 1;          // ragged operands, up to 128 rows: 0: never gemm_few_kernel, 2: wherever it can, 1: by its estimate (few_estimate)
    long row_estimate = 1;      // 0: up to 400 rows follow the rules (choose_by_rules) instead of the estimate of every row (choose_variant)
    long k_rot = -1;            // -1: rotated K start for at most 256 rows (see plan_nt), 0: never, n: steps per column tile
    long stagger = -1;          // -1: staggered start where it pays (4-byte C, three or more rounds), else microseconds per group
    long stagger_groups = 8;    // groups the workgroups of the first round start in
    long c_plain = -1;          // -1: the library decides; 0 / 1: non-temporal / ordinary stores for C
    long b_stream = -1;         // -1: the library decides; 0 / 1: B copies of the skinny-M kernel without / with the streaming hint
    long row_split = 1;         // 0: never run the rows (or columns) of a last, mostly empty round of 256 x 256 tiles as a second launch;
                                // 2 / 3: the rows / the columns always where the geometry allows it, whatever the estimate says
                                // (for measurements)
    long any_shape = 1;         // rows that are not whole 16-byte chunks on 16 bytes: 0: the any-shape kernel, 1: what is estimated fastest of
                                // it, the other kernels on the rows as they stand, and on packed rows; 2 / 3: packed / as they stand wherever
                                // possible (for measurements and tests)
    long kmajor = 1;            // 0: K-major operands (NN, reference fp8 layout) always go through the transposes; 2: never
                                // where a K-major kernel fits the shape (for measurements and tests)
    std::string last_config;
    const char *last_any_kernel = "";    // what launch_any_t launched last
};

Context g_ctx;

#define HIP_TRY(expr)                                  \
    do {                                               \
        hipError_t e_ = (expr);                        \
        if (e_ != hipSuccess) return QGEMM_ERR_LAUNCH; \
    } while (0)

int static_scratch_locked(void **out);

int ensure_init_locked() {
    if (g_ctx.ready) return QGEMM_OK;
    int n = 0;
    if (hipGetDeviceCount(&n) != hipSuccess || n <= 0) return QGEMM_ERR_NO_DEVICE;
    int dev = 0;
    HIP_TRY(hipGetDevice(&dev));
    hipDeviceProp_t prop;
    HIP_TRY(hipGetDeviceProperties(&prop, dev));
    // The address of the static scratch on this device is looked up here, once, so that qgemm_scaled_gemm_static
    // finds it without a runtime call of its own; if the lookup fails only that entry is affected (it tries again
    // and reports the failure), every other entry works without the scratch.
    void *scratch_dev = nullptr;
    (void)static_scratch_locked(&scratch_dev);
    g_ctx.device = dev;
    g_ctx.num_cus = prop.multiProcessorCount > 0 ? prop.multiProcessorCount : 256;
    // tuning knobs, also reachable through qgemm_set_option
    if (const char *e = std::getenv("QGEMM_FORCE_CONFIG")) g_ctx.force_config = e;
    if (const char *e = std::getenv("QGEMM_GROUP_M")) g_ctx.force_group_m = std::atol(e);
    g_ctx.ready = true;
    return QGEMM_OK;
}

// Device address of the static scratch on the current device (looked up once per device).
int static_scratch_locked(void **out) {
    int dev = 0;
    HIP_TRY(hipGetDevice(&dev));
    if (dev < 0 || dev >= kMaxDevices) return QGEMM_ERR_UNSUPPORTED;
    if (!g_ctx.static_ptr[dev]) {
        void *p = nullptr;
        if (hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)) != hipSuccess || !p) return QGEMM_ERR_LAUNCH;
        g_ctx.static_ptr[dev] = p;
    }
    *out = g_ctx.static_ptr[dev];
    return QGEMM_OK;
}

bool stream_is_capturing(hipStream_t stream) {
    hipStreamCaptureStatus cap = hipStreamCaptureStatusNone;
    if (hipStreamIsCapturing(stream, &cap) != hipSuccess) {
        (void)hipGetLastError();
        return false;
    }
    return cap != hipStreamCaptureStatusNone;
}

// Makes a block at least `bytes` large, twice its size if it has to grow; the old memory is retired (see Context).
int grow_block(WsBlock &block, size_t bytes, size_t least) {
    if (bytes <= block.bytes) return QGEMM_OK;
    const size_t want = std::max({bytes, 2 * block.bytes, least});
    // (another thread may be capturing a stream of its own: this allocation is none of its business)
    hipStreamCaptureMode mode = hipStreamCaptureModeRelaxed;
    const bool exchanged = hipThreadExchangeStreamCaptureMode(&mode) == hipSuccess;
    void *p = nullptr;
    const hipError_t e = hipMalloc(&p, want);
    if (exchanged) (void)hipThreadExchangeStreamCaptureMode(&mode);
    if (e != hipSuccess) {
        (void)hipGetLastError();
        return QGEMM_ERR_ALLOC;
    }
    if (block.p) g_ctx.retired.push_back(block.p);
    block.p = p;
    block.bytes = want;
    return QGEMM_OK;
}

// An own block of `bytes`, unless it is as large already; false where there is no memory for it
bool make_own_block(WsBlock &block, size_t bytes) {
    if (bytes <= block.bytes) return true;
    WsBlock larger;
    if (!g_ctx.ws_own_failed) g_ctx.ws_own_failed = grow_block(larger, bytes, 0) != QGEMM_OK;
    if (g_ctx.ws_own_failed) return false;
    if (block.p) g_ctx.retired.push_back(block.p);
    block = larger;
    return true;
}
// The stream's own block for a call that needs `bytes` (kOwnBytes at most), null where it has none
void *own_block(hipStream_t stream, size_t bytes) {
    if (stream == hipStreamPerThread) return nullptr;
    int i = 0;
    while (i < g_ctx.ws_owners && g_ctx.ws_stream[i] != stream) ++i;
    if (i == kOwnBlocks || (bytes > g_ctx.ws_own[i].bytes && !make_own_block(g_ctx.ws_own[i], kOwnBytes))) return nullptr;
    if (i == g_ctx.ws_owners) g_ctx.ws_stream[g_ctx.ws_owners++] = stream;
    return g_ctx.ws_own[i].p;
}

// Workspace of `bytes` for a call enqueued on `stream`.
//   * qgemm_scaled_gemm_static: the static scratch; larger requests are an error, nothing is allocated.
//   * otherwise the stream's own block or the shared one (see Context), which grows when too small.  While the stream is being captured into
//     a graph nothing is allocated and no event is waited for or recorded: such a call takes the shared block, and one that would need
//     more fails with QGEMM_ERR_ALLOC (the caller reserves the room before the capture, qgemm_reserve_workspace, or runs the
//     call once eagerly), and ordering replays against other users of the workspace is the caller's business.
int ensure_workspace_locked(size_t bytes, hipStream_t stream, void **out) {
    if (g_ctx.static_call) {
        if (bytes > kStaticScratchBytes) return QGEMM_ERR_SCRATCH_TOO_SMALL;
        return static_scratch_locked(out);
    }
    if (stream_is_capturing(stream)) {
        *out = g_ctx.ws.p;
        return bytes > g_ctx.ws.bytes ? QGEMM_ERR_ALLOC : QGEMM_OK;
    }
    const int st = grow_block(g_ctx.ws, bytes, kLeastBlock);
    *out = bytes <= kOwnBytes ? own_block(stream, bytes) : nullptr;
    if (*out) return QGEMM_OK;
    if (st != QGEMM_OK) return st;
    if (!g_ctx.ws_shared_by_call) {
        if (g_ctx.ws_event_recorded && (g_ctx.ws_last_stream != stream || stream == hipStreamPerThread))
            HIP_TRY(hipStreamWaitEvent(stream, g_ctx.ws_event, 0));
        g_ctx.ws_shared_by_call = true;
    }
    *out = g_ctx.ws.p;
    return QGEMM_OK;
}

// Around the body of every entry that may use the workspace: when it used the shared block, the end of its launches is recorded
// on its stream for the next user on another stream to wait for.
struct WorkspaceUse {
    hipStream_t stream;
    explicit WorkspaceUse(hipStream_t s) : stream(s) { g_ctx.ws_shared_by_call = false; }
    ~WorkspaceUse() {
        if (!g_ctx.ws_shared_by_call) return;
        g_ctx.ws_shared_by_call = false;
        if (!g_ctx.ws_event && hipEventCreateWithFlags(&g_ctx.ws_event, hipEventDisableTiming) != hipSuccess) {
            (void)hipGetLastError();
            g_ctx.ws_event = nullptr;
            return;
        }
        if (hipEventRecord(g_ctx.ws_event, stream) == hipSuccess) {
            g_ctx.ws_event_recorded = true;
            g_ctx.ws_last_stream = stream;
        } else {
            (void)hipGetLastError();
        }
    }
};

// kmaj: GemmCfg::KMAJ of the wanted family (0: both operands K-contiguous)
const Variant *table_for(int arith, bool block, int kmaj, int *count) {
    if (kmaj == 3) return (block && arith == AR_F8) ? variants_f8_block_tn(count) : nullptr;
    if (kmaj == 2) return block ? nullptr : (arith == AR_BF16 ? variants_bf16_nn(count) : (arith == AR_F16 ? variants_f16_nn(count) : nullptr));
    if (kmaj != 0) return nullptr;
    if (block && arith == AR_F8W) return variants_f8w_block(count);
    if (block) return arith == AR_F8 ? variants_f8_block(count) : (arith == AR_I8 ? variants_i8_block(count) : nullptr);
    switch (arith) {
        case AR_I8: return variants_i8(count);
        case AR_F8: return variants_f8(count);
        case AR_F8W: return variants_f8w(count);
        case AR_BF16: return variants_bf16(count);
        case AR_F16: return variants_f16(count);
    }
    return nullptr;
}

// Row `name` of a table, -1 when the family has no such row.
int row_by_name(const Variant *tab, int count, const std::string &name) {
    for (int i = 0; tab && i < count; ++i)
        if (name == tab[i].name) return i;
    return -1;
}
bool forced() { return !g_ctx.force_config.empty(); }

int arith_of(int in_dtype) {
    switch (in_dtype) {
        case QGEMM_DT_I8: return AR_I8;
        case QGEMM_DT_F8E4M3: return AR_F8;
        case QGEMM_DT_BF16: return AR_BF16;
        case QGEMM_DT_F16: return AR_F16;
    }
    return -1;
}

bool out_dtype_ok(int in_dtype, int out_dtype) {
    if (out_dtype == QGEMM_DT_F32 || out_dtype == QGEMM_DT_BF16 || out_dtype == QGEMM_DT_F16) return true;
    return out_dtype == QGEMM_DT_I32 && in_dtype == QGEMM_DT_I8;
}

// What copying 128 bytes of a row of A or B into LDS takes a CU, us, where it is known to bound a step: rows that do not start on 16 bytes
// (0: the planner's times per step have it).
struct RowCopies {
    double a = 0, b = 0;
    bool tile64 = true;          // 64 x 64 with two K groups may be chosen (see copies_of)
};
struct NtProblem {
    int arith;
    bool block;
    const void *A, *B;
    void *C;
    size_t lda_bytes, ldb_bytes, ldc;   // ldc in elements; lda / ldb: stride between rows of m / n, or, for a
                                        // K-major operand (kmaj), between rows of k
    size_t M, N, Kbytes;
    size_t k_rest;                      // bytes of K behind Kbytes, which then ends with the last whole 16-byte chunk (GemmArgs::k_rest)
    int kmaj;                           // bit 0: A is stored K x M, bit 1: B is stored K x N
    const float *as, *bs;
    uint32_t as_ms, as_ks, bs_ns, bs_ks;
    int out_dtype, per_matrix, split_k;
    bool no_planes;                     // never a K split (a second launch for rows or columns all the same)
    RowCopies copies;
};

bool aligned16(const void *p) { return ((uintptr_t)p & 15u) == 0; }

size_t ksteps_of(const NtProblem &q) { return (q.Kbytes + 127) / 128; }      // the last one may be partial

// Shapes the MFMA kernel takes (mfma_shape_ok: with whole rows, pointer alignment checked separately; everything else: launch_unaligned,
// launch_packed, launch_any).  K is a whole number of 16-byte chunks (the unit of a copy); a last K step of fewer than 128 bytes is
// filled up with zeros on the way into LDS (GemmArgs::k_tail), which the reference's dispatch covers with its
// 64- and 32-wide K tiles (hip_mix_gemm_kernel.cpp:442-463).
bool mfma_sizes_ok(const NtProblem &q) {
    const size_t es = (q.arith == AR_BF16 || q.arith == AR_F16) ? 2 : 1, krows = q.Kbytes / es;
    // 32-bit buffer offsets: 256 tile rows of a K-contiguous operand (plus the 3072 bytes by which the solo kernels
    // shift their descriptors), every k row of a K-major one.  With a partial last K step the lanes past the end of
    // a row mark their offsets with bit 31: every valid offset then has to stay below 2^31.
    const size_t lim = (size_t)1 << (q.Kbytes % 128 ? 31 : 32);
    const bool a_ok = (q.kmaj & 1) ? (krows * q.lda_bytes < ((size_t)1 << 32) && q.lda_bytes >= q.M * es)
                                   : q.lda_bytes * 256 + 4096 < lim;
    const bool b_ok = (q.kmaj & 2) ? (krows * q.ldb_bytes < ((size_t)1 << 32) && q.ldb_bytes >= q.N * es)
                                   : q.ldb_bytes * 256 + 4096 < lim;
    // block scales: the kernel addresses a_scale with 32-bit byte offsets ((kb * as_ks + m) * 4)
    const bool s_ok = !q.block || ((q.Kbytes + 127) / 128) * std::max<size_t>(q.M, q.as_ks) * 4 < ((size_t)1 << 32);
    return q.Kbytes % 16 == 0 && q.Kbytes > 0 && a_ok && b_ok && s_ok && q.M < ((size_t)1 << 31) && q.N < ((size_t)1 << 31) && q.ldc < ((size_t)1 << 32);
}
bool mfma_shape_ok(const NtProblem &q) { return q.lda_bytes % 16 == 0 && q.ldb_bytes % 16 == 0 && mfma_sizes_ok(q); }

// Which tile, and how many K slices.
//
// M > 64: a cost estimate over the tiles worth having there (256 x 256 solo, 128 x 128 in two forms, 64 x 128, 128 x 32) and
// 1 / 2 / 4 / 8 K slices.  Workgroups run in rounds of CUs x (workgroups that fit a CU); a round costs
// (K steps x time per step + a fixed prologue / epilogue), a last partial round that leaves a 128 x 128
// workgroup alone on its CU runs its steps faster, and a K split pays a second launch plus the traffic of the
// partial planes.  The times per 128-byte K step were read off a sweep of every variant over square and oblong
// shapes from 1024 to 8192 (fp8 and bf16 agree per step; block scales have figures of their own): 1.25 us for the
// 256 x 256 tile (one per CU), 0.85 us for 128 x 128 with two per CU and 0.66 us alone, 0.43 us for the 128 x 128
// row with two K groups (one per CU: it only wins where there are no more tiles than CUs; 2048 x 2048 x 2048 / 8192
// 12.1 / 32.5 us), 0.52 us for 64 x 128 and 0.27 us for its row with two K groups (512 x 4096 x 4096 13.5 us, two
// rounds of 64 steps 44 us), 0.39 us for 128 x 32; for 256 x 128 with its copying waves 0.71 us with every CU at work,
// which is what the 256 x 256 tile needs per flop, and 0.58 us with 160 - 224 tiles (0.93 / 0.76 with block scales),
// plus 6 us around a round (2048 x 4096 x 4096 29.3 us, 1024 x 8192 x 8192 50.8, 1536 x 4096 x 4096 25.2,
// 768 x 7168 x 2048 14.8; it wins where its tiles make one round of CUs and the 256 x 256 tiles would leave half of
// them idle: 6 - 17 % over the two-stage 128 x 128 row there, with block scales up to 24 %).
// 192 x 256 (8-wave solo schedule) for row counts whose 256-row tiles leave a round partly empty: 1.03 us a step in a
// full round, 0.97 in a partly filled one (1.27 / 1.18 with block scales), 6 us around a round (3072 x 4096 x 4096 fp8
// 43.7 us against 47.5 on 192 tiles of 256 x 256, 2560 rows 37.7 against 42.8, 1536 x 7168 x 2048 23.3 against 26.8,
// bf16 1152 x 8192 x 4096 64.6 against 78.3).  Full rounds refitted on 36 large shapes per type with every large row
// forced (they had been priced at 1.10 / 1.30, 7 - 10 % above what was measured): shapes whose 192-row tiles make
// whole rounds now run on them in one launch instead of a 256 x 256 launch and a rest (6144^3: 768 tiles, three
// rounds; fp8 165.9 -> 163.7 us, block scales 206.9 -> 198.1, bf16 327.4 -> 318.5; over the 71 of 1440 grid shapes
// whose plan changed the new plan is 3.0 % faster on average, at worst 1.6 % slower).
// A K split adds 4 us and the partial planes at 3 TB/s.
// The reference's storage has 64 x 128 with two K groups as well: few rows left most of a 128-row tile empty and most CUs idle (fp8_mm, us,
// 128 x 128 / so: 32 x 1280 x 832 7.4 / 6.3, 96 x 1536 x 3328 11.3 / 10.0, 288 x 4736 x 3840 18.0 / 15.8, 544 x 1792 x 3072 15.8 / 13.2).
// The K-major families have 64 x 64 with two K groups too, two workgroups a CU: mid-sized products make few tiles, and a CU's work on one is
// latency (start, first copies, a step of 0.18 us, the way out).  Graph replays, us, the best other row / so: B stored K x N bf16 505 x 1056 x
// 531 8.7 / 6.6, 512 x 512 x 2048 11.7 / 9.2, 384 x 1280 x 1184 8.2 / 7.0, 64 x 2816 x 560 6.1 / 5.1; fp8_mm 160 x 3168 x 448 5.7 / 4.6, 1024 x
// 544 x 2080 9.7 / 7.7, 512 x 1984 x 1792 9.0 / 7.4, 1024 x 1024 x 1024 6.8 / 5.5, bf16 7.7 / 6.6.  136 shapes of 32 .. 1280 rows: 7 - 24 % ahead
// wherever there are no more tiles than CUs.  With more, two share a CU: up to five K steps level with the best other row and ahead of
// what the estimates would take instead (fp8_mm 352 x 2848 x 352 5.8 / 5.0); beyond, with block scales, level to 60 % behind (224 shapes; 1280 x 1280 x
// 1024 7.2 / 8.1, 608 x 3232 x 3008 16.8 / 21.0), where the estimate is up to 29 % low; 16-bit types are behind by as much, and the estimate knows it.
// In the K-contiguous families, whose other rows need no transposing reads, it is level or behind, but for what choose_by_rules gives it.
//
// M <= 64 (bandwidth-bound, B is streamed once): the largest tile that still gives three quarters of the CUs a
// workgroup, else the shortest tile that covers the rows; narrow tiles instead of a K split.  (65 .. 128 rows go
// through the estimate as well: it keeps the 128 x 32 tile for the short K of config 5 and prefers a 128 x 128 tile
// with a K split where K is long, 128 x 8192 x 8192 bf16 38 against 48 us.)
struct TileModel {
    int bm, bn, per_cu;
    double step_shared, step_alone, fixed;     // microseconds
    bool kgroups;                              // the row of this tile with two K groups per workgroup (GemmCfg::KG)
    // the same with 128-block scales (fp8): the fold costs the 8-wave 256 x 256 kernel a tenth, the simple pipeline
    // more (its block-scaled rows have two stages, so more workgroups share a CU), the K-group rows most
    int blk_per_cu;
    double blk_shared, blk_alone;
};
// (block scales, graph replays: 256 x 256 2048 x 4608 x 7168 77 us, 1536 x 7168 x 2048 27.6; 128 x 128 1024 x 7168 x 2048 25.9,
// 1024 x 4608 x 7168 75.0; 64 x 128 1024 x 4608 x 7168 69.9, 512 x 4608 x 7168 47.8; K groups 128 x 128 2048 x 2048 x 2048 /
// 8192 14 / 43, 64 x 128 512 x 4096 x 4096 18, and with the a_scale values of four K blocks per copy (GemmArgs::as_groups)
// 38 - 41 and 15.3; 128 x 32 256 x 7168 x 2048 12.9)
const TileModel kTileModels[] = {{256, 256, 1, 1.25, 1.25, 4.0, false, 1, 1.40, 1.40}, {128, 128, 2, 0.85, 0.66, 2.0, false, 2, 1.32, 1.04},
                                 {128, 128, 1, 0.43, 0.43, 4.5, true, 1, 0.50, 0.50},  {64, 128, 1, 0.52, 0.52, 1.5, false, 3, 1.21, 0.83},
                                 {64, 128, 1, 0.27, 0.27, 4.5, true, 1, 0.34, 0.34},   {128, 32, 1, 0.39, 0.39, 1.0, false, 2, 0.74, 0.60},
                                 {256, 128, 1, 0.71, 0.58, 6.0, false, 1, 0.93, 0.76}, {192, 256, 1, 1.03, 0.97, 6.0, false, 1, 1.27, 1.18},
                                 {64, 64, 2, 0.47, 0.23, 2.9, true, 2, 0.56, 0.24}};
// Widened fp8 (AR_F8W: packed operands): twice the matrix instructions of a 16-bit step and the conversions in front of them, on
// the rows that family has.  Fitted on 56 ragged shapes of 1 .. 4096 rows x 1024 .. 7168 columns x 777 .. 7161, every row forced
// (within 5 % of the measured time on average).  Priced as fp8 before, us in a kernel trace: 512 x 4608 x 7161 58.5 (128 x 128) ->
// 44.4 (192 x 256, four slices), 1024 x 4608 x 7161 88.6 -> 69.8, block scales 512 x 5000 x 3004 41.7 (64 x 128 with K groups) ->
// 30.3 (128 x 32).
const TileModel kWideTileModels[] = {{128, 128, 2, 1.55, 0.96, 3.5, false, 2, 1.95, 1.19}, {64, 128, 1, 0.70, 0.72, 3.0, false, 3, 1.49, 0.87},
                                     {64, 128, 1, 0.41, 0.44, 4.5, true, 1, 0.68, 0.72},   {128, 32, 1, 0.43, 0.47, 2.0, false, 3, 0.99, 0.71},
                                     {192, 256, 1, 1.99, 1.70, 5.5, false, 1, 2.36, 2.01}};
// `wgs` workgroups of `steps` K steps, `slots` of them on the chip at a time
double rounds_cost(size_t wgs, size_t slots, size_t cus, size_t steps, double shared, double alone, double fixed) {
    const size_t full = wgs / slots, rem = wgs % slots;
    double t = (double)full * (steps * shared + fixed);
    if (rem) t += steps * (rem <= cus ? alone : shared) + fixed;
    return t;
}
// rows with two K groups: two sets of computing waves on a tile that otherwise has one (one workgroup per CU)
bool is_kgroup_row(const Variant &v) { return v.kgroups == 2; }

// An fp32 output that shows how its sums are made keeps the rows, and with them the parts of a sum, that it had before the 64 x 64 tile.
// (fp8 does not show them: 70 shapes whose row, K split or both the tile replaced are 1.8e-5 of the result from 64 bits either way, the
// two within 1.3e-4 of each other.)
bool output_shows_sums(int arith, bool block, int out_dtype);
RowCopies copies_of(const NtProblem &q) {
    RowCopies c = q.copies;
    c.tile64 = !output_shows_sums(q.arith, q.block, q.out_dtype);
    return c;
}

int choose_by_cost(const Variant *tab, int count, size_t M, size_t N, size_t ksteps, bool block, int cus, bool may_split,
                   uint32_t *nsplit_out, double *cost_out = nullptr, RowCopies copies = {}) {
    int best = -1;
    double best_t = 0;
    const bool wide = tab[0].arith == AR_F8W;
    const TileModel *models = wide ? kWideTileModels : kTileModels;
    for (size_t mi = 0; mi < (wide ? std::size(kWideTileModels) : std::size(kTileModels)); ++mi) {
        const TileModel &tm = models[mi];
        int vi = -1;
        for (int i = 0; i < count; ++i)
            if (tab[i].auto_ok && tab[i].bm == tm.bm && tab[i].bn == tm.bn && is_kgroup_row(tab[i]) == tm.kgroups) vi = i;
        if (vi < 0) continue;
        const size_t tiles = ((M + tm.bm - 1) / tm.bm) * ((N + tm.bn - 1) / tm.bn);
        if (tm.bm == 64 && tm.bn == 64 && (!copies.tile64 || (block && tiles > (size_t)cus && ksteps > 5))) continue;
        for (uint32_t ns = 1; ns <= 8; ns *= 2) {
            if (ns > 1 && (!may_split || ksteps / ns < 4)) break;
            const size_t wgs = tiles * ns, slots = (size_t)cus * (block ? tm.blk_per_cu : tm.per_cu), steps = (ksteps + ns - 1) / ns;
            const double copy = tm.bm * copies.a + tm.bn * copies.b;
            double t = rounds_cost(wgs, slots, cus, steps, std::max(block ? tm.blk_shared : tm.step_shared, copy * (block ? tm.blk_per_cu : tm.per_cu)),
                                   std::max(block ? tm.blk_alone : tm.step_alone, copy), tm.fixed);
            if (ns > 1) t += 4.0 + (double)M * N * 4.0 * (ns + 1) / 3.0e6;
            if (best < 0 || t < best_t) {
                best = vi;
                best_t = t;
                *nsplit_out = ns;
            }
        }
    }
    if (cost_out) *cost_out = best_t;
    return best;
}

int choose_tile(const Variant *tab, int count, size_t M, size_t N, size_t ksteps, bool block, int kmaj, int cus,
                bool may_split, uint32_t *nsplit_out, RowCopies copies);
size_t rows_for_full_rounds(const Variant *tab, int count, size_t M, size_t N, size_t ksteps, bool block, int cus,
                            double t_single, double *t_split = nullptr, size_t *padding = nullptr, RowCopies copies = {});
size_t cols_for_full_rounds(const Variant *tab, int count, size_t M, size_t N, size_t ksteps, bool block, int cus,
                            double t_single, double *t_split = nullptr, size_t *padding = nullptr, bool whatever_the_estimate = false, RowCopies copies = {});

// The skinny-M kernel (gemm_skinny.cuh: the K split inside the workgroup, eight waves each on every eighth K step)
// takes over from the narrow simple-pipeline tiles where it is faster: one row tile (M <= 128), a strip of 32
// columns per workgroup as the tile choice below would have it, and enough K steps for the eight waves (two each;
// one each is enough up to 16 rows).  Graph replays over rotated B, fp8, microseconds per launch, narrow tile
// against skinny kernel: 16 x 7168 x 2048 7.6 / 5.4, 64 x 7168 x 2048 9.0 / 6.7, 128 x 7168 x 2048 11.0 / 8.2,
// 16 x 7168 x 8192 24.6 / 15.2, 32 x 4096 x 4096 12.7 / 8.3, 128 x 4096 x 4096 18.3 / 12.5, 16 x 1024 x 1024
// 5.6 / 3.1; with K = 1024 and more than 16 rows or K = 512 the narrow tiles stay ahead (64 x 8192 x 1024 5.0 / 5.2,
// 128 x 7168 x 512 4.6 / 6.0).  The same rule serves block scales (B resident: 16 x 7168 x 2048 10.8 / 6.6,
// 128 x 7168 x 2048 15.7 / 9.5).
// A K split across workgroups on top pays only where the strips leave at least half of the CUs without work and K is
// long: a workgroup moves its strip of B and its rows of A at about 45 GB/s, a split divides that time and adds a
// reduction launch of about 4.5 us.  B out of HBM, microseconds per launch, one workgroup per strip against the split
// this estimate picks: 16 x 4096 x 14336 fp8 20.6 / 17.2 (two slices), bf16 37.1 / 26.9; 64 x 4096 x 14336 27.3 / 22.7,
// bf16 53.7 / 37.2; 64 x 2048 x 8192 15.2 / 11.3 (four slices), bf16 26.8 / 14.7; no split for 16 x 4096 x 4096 (7.6
// against 9.5 with two slices) and none where the strips fill the CUs (16 x 8192 x 8192 15.2 against 18.8).
// kmaj: the table is a K-major family, which has no narrow tiles: the estimate then serves every M
int choose_by_rules(const Variant *tab, int count, size_t M, size_t N, size_t ksteps, bool block, int kmaj, int cus,
                   bool may_split, uint32_t *nsplit_out, RowCopies copies) {
    const int vi = choose_tile(tab, count, M, N, ksteps, block, kmaj, cus, may_split, nsplit_out, copies);
    // The same kernel on 64 x 64 tiles: shapes with several row tiles whose 64 x 64 tiles fit one
    // round of CUs and give most of them work, 16 K steps or more.  Against whatever the estimate picks (narrow
    // tiles, K-group tiles with a K split) it is 13 - 33 % faster over 512 .. 2048 rows x 256 .. 3000 columns x 2 .. 8 KiB
    // of K (fp16 1024^3 7.3 -> 6.3 us, fp8 1000 x 1000 x 4096 13.1 -> 8.8), slower only with 8 K steps (one per wave)
    // or with 64 tiles and 64 K steps; beyond 64 K steps the tiles with a K split across workgroups catch up
    // (bf16 256 x 2048 x 7168, 112 steps: 18.9 against 22.9 us).  With block scales the gain is larger, the small tiles
    // of the simple pipeline being slower there: 512 x 2048 x 4096 18.3 -> 11.7 us, 256 x 4096 x 4096 17.8 -> 11.8.
    // From 65 rows on: with two row tiles a workgroup pulls half of A (an L2 hit, but through its CU's load path) next
    // to twice the strip of B, 256 KiB instead of 320 KiB at 128 x 7168 x 2048, the smallest sum a tile of that area
    // has (config 5 at M = 128, B out of HBM: 8.9 -> 8.3 us; M = 64 stays on 32-column strips, 6.8 us).
    // 17 .. 256 rows against few columns, 32 .. 48 K steps: tiles of 16 x 32, 32 x 32, 64 x 32 or 64 x 64 on the skinny-M kernel,
    // several over the rows, whichever fills at most one round of CUs with the least to move: a workgroup moves its rows
    // of A at about 100 GB/s (L2 hits) and its strip of B at about 45 GB/s (out of memory), all of them together about
    // 12 TB/s (the row tiles of a strip share it in the L2s); constants fitted on 90 shapes x 4 tiles x (one B, B in
    // rotation through 600 MB).  That beats a taller tile with a K split across workgroups (a second launch of 4.5 us)
    // and the 64 x 64 form where smaller tiles still fit a round.  Graph replays, us, one B / B in rotation through
    // 600 MB, what the rules below took against this: 128 x 1024 x 4096 fp8 10.0 / 10.7 (128 x 32, four slices) ->
    // 5.4 / 6.6 (32 x 32), 96 x 2048 x 4096 8.8 / 11.3 (64 x 64) -> 6.5 / 7.9, 128 x 2048 x 4096 8.8 / 11.8 -> 7.6 / 9.1
    // (64 x 32), 130 x 1536 x 6144 12.8 / 13.7 -> 10.0 / 11.0; bf16 the same at the same bytes of K, block scales
    // 128 x 2048 x 4096 10.5 / 13.0 -> 8.7 / 9.7.  From 56 K steps on the small tiles still win with B resident
    // (160 x 2048 x 7168 13.5 -> 12.2) but lose with B streamed (14.9 -> 17.7: fewer, longer streams), so the K split
    // stays there; block scales only up to 32 K steps (their fold makes the longer loops of the small tiles slower).
    // 24 .. 256 rows x 1024 .. 7168 columns x 4 and 6 KiB of K, fp8, 90 shapes: 13 % less time with B resident, 9.5 % with B
    // streamed, two shapes more than 3 % slower (7 % at worst); 64 x 1024 x 4096 fp8 7.7 / 8.5 (64 x 32, four slices) ->
    // 4.7 / 5.6 (16 x 32).  A smaller tile has to be estimated 3 % ahead of a larger one.
    if (vi >= 0 && !kmaj && g_ctx.small_tiles && M > 16 && M <= 256 && ksteps >= 32 && ksteps <= (block ? 32u : 48u)) {
        int best = -1;
        double best_t = 0;
        static const int kSmall[4][2] = {{64, 64}, {64, 32}, {32, 32}, {16, 32}};       // (a smaller tile has to be 3 % ahead)
        for (const auto &bt : kSmall)
            for (int i = 0; i < count; ++i) {
                const Variant &v = tab[i];
                if (v.kgroups != 8 || v.bm != bt[0] || v.bn != bt[1]) continue;
                const size_t tiles = ((M + v.bm - 1) / v.bm) * ((N + v.bn - 1) / v.bn);
                if (tiles > (size_t)cus) continue;
                const double kb = ksteps * 128.0;
                const double t = std::max(v.bm * kb / 100.0e3 + v.bn * kb / 45.0e3, tiles * (v.bm + v.bn) * kb / 12.0e6);
                if (best < 0 || t < 0.97 * best_t) {
                    best = i;
                    best_t = t;
                }
            }
        if (best >= 0) {
            *nsplit_out = 1;
            return best;
        }
    }
    if (vi >= 0 && !kmaj && M > 64 && ksteps >= 16 && ksteps <= 64) {
        const size_t t64 = ((M + 63) / 64) * ((N + 63) / 64);
        // (with more than 48 K steps and weights streamed out of memory, half a round of such tiles is behind a wider tile
        // with a K split, which has twice the streams: 256 x 2048 x 8192 fp8 18.3 against 16.1 us, 13.5 against 13.8 with
        // B resident; from 160 tiles on the 64 x 64 form is ahead either way)
        if (t64 <= (size_t)cus && ((t64 >= 128 && (ksteps <= 48 || t64 >= 160)) || (t64 >= 64 && ksteps <= 32)))
            for (int i = 0; i < count; ++i)
                if (tab[i].kgroups == 8 && tab[i].bm == 64 && tab[i].bn == 64) {
                    *nsplit_out = 1;
                    return i;
                }
    }
    // 64 x 64 with two K groups where such tiles fit a round and 9 .. 15 K steps (block scales: 8 .. 15) are too few for the eight waves above;
    // fewer do not pay for its start.  More than 400 rows (below, the estimate of choose_variant decides) that start on whole chunks.  Graph
    // replays, us, the rows of the estimate (128 x 32, 64 x 128 with K groups) / so: int8 600 x 512 x 1152 5.6 / 5.3, fp8 600 x 1536 x 1792 7.3 /
    // 6.4, bf16 896 x 688 x 768 7.1 / 6.4, block scales fp8 416 x 1728 x 1792 8.7 / 7.0, int8 1200 x 832 x 1152 7.4 / 6.0; 4 steps 4.1 / 4.5,
    // 6 steps 4.7 / 4.8; 24 steps against the eight waves 8.3 / 8.5, 32 steps 8.6 / 10.3.
    if (vi >= 0 && !kmaj && M > 400 && ksteps >= (block ? 8 : 9) && ksteps <= 15 && copies.tile64 && copies.a == 0 && copies.b == 0 &&
        ((M + 63) / 64) * ((N + 63) / 64) <= (size_t)cus)
        for (int i = 0; i < count; ++i)
            if (tab[i].kgroups == 2 && tab[i].bm == 64 && tab[i].bn == 64) {
                *nsplit_out = 1;
                return i;
            }
    if (vi < 0 || kmaj || M > 128) return vi;
    const size_t strips = (N + 31) / 32;
    // Up to 32 rows against so few columns that 32-column strips leave half of the CUs idle, 32 .. 112 K steps: strips of
    // 16 columns, one workgroup each and no K split across workgroups (which costs a second launch).  Graph replays, us,
    // one B / B in rotation through 600 MB, fp8 (bf16 the same at the same bytes of K): 16 x 4096 x 14336 14.7 / 15.8
    // (32-column strips, two slices) -> 12.6 / 13.0 (vendor library 12.7 / 14.7), 16 x 4096 x 8192 11.5 / 12.1 -> 9.4 / 9.0,
    // 16 x 2048 x 8192 7.2 / 9.6 -> 5.6 / 7.7, 32 x 4096 x 14336 16.2 / 18.1 -> 15.8 / 16.6; from 128 K steps on the split is
    // ahead (16 x 2048 x 16384 10.2 / 11.0 against 12.2 / 13.2), and with 64 rows the two are level or the split ahead.
    // With fewer than 192 such strips (N < 3072) only up to 16 rows and 64 K steps: beyond that the streams are too few
    // and too long, and the split is 4 - 50 % ahead with B streamed (32 x 1024 x 14336 9.5 against 14.7 us).  Not with block
    // scales (3 - 30 % slower throughout).
    const size_t strips16 = (N + 15) / 16;
    if (g_ctx.small_tiles && !block && M <= 32 && ksteps >= 32 && ksteps <= 112 && strips * 2 <= (size_t)cus && strips16 <= (size_t)cus &&
        (strips16 >= 192 || (M <= 16 && ksteps <= 64)))
        for (int i = 0; i < count; ++i)
            if (tab[i].kgroups == 8 && tab[i].bn == 16 && (size_t)tab[i].bm >= M) {     // (rows of the table in ascending height)
                *nsplit_out = 1;
                return i;
            }
    // 17 .. 64 rows against so many columns that the 32-column strips need a second round of CUs while 64-column
    // strips fit in one: the 64 x 64 form (half the strips, each row of A fetched half as often).  B out of HBM:
    // 64 x 14336 x 4096 bf16 34.3 -> 26.7 us, fp8 20.4 -> 17.0; 48 rows 33.4 -> 27.4 and 19.4 -> 16.5; 32 rows bf16
    // 26.4 -> 23.5, 32 x 14336 x 8192 49.7 -> 41.2, 24 x 11008 x 4096 24.4 -> 22.5, 32 x 12288 x 2048 fp8 10.4 -> 9.1
    // (up to 16 rows the two are level).
    if (M > 16 && M <= 64 && ksteps >= 16 && strips > (size_t)cus && (N + 63) / 64 <= (size_t)cus)
        for (int i = 0; i < count; ++i)
            if (tab[i].kgroups == 8 && tab[i].bm == 64 && tab[i].bn == 64) {
                *nsplit_out = 1;
                return i;
            }
    // 65 .. 128 rows come out of the estimate above, whose times per step are those of operands that sit in the caches;
    // with B streamed out of memory the skinny-M kernel is ahead wherever its strips fit one round of CUs and K is
    // not long enough for a K split to pay (128 x 7168 x 2048 bf16 17.8 -> 13.6 us, 128 x 8192 x 8192 fp8 26.9 -> 24.8)
    const bool mid_rows = M > 64 && strips <= (size_t)cus && ksteps >= 16 && ksteps <= 64;
    // (up to 64 rows the choice above takes a wide tile with a K split where 32-column tiles of its height would need
    // more than two rounds; up to two rounds of strips the skinny-M kernel is ahead of that too: 32 x 14336 x 4096 fp8
    // 24.6 -> 17.2 us, bf16 36.4 -> 29.7; with 896 strips the wide tiles stay, 32 x 28672 x 8192 46.8 against 55.1)
    const bool few_strips = M <= 64 && strips <= 2 * (size_t)cus && ksteps >= 16;
    if (!mid_rows && !few_strips && (tab[vi].bn != 32 || tab[vi].kgroups != 1)) return vi;
    if (ksteps < 8 || (ksteps < 16 && M > 16)) return vi;
    for (int i = 0; i < count; ++i)
        if (tab[i].kgroups == 8 && tab[i].bn == 32 && (size_t)tab[i].bm >= M) {        // (rows of the table in ascending height)
            *nsplit_out = 1;
            if (may_split && strips * 2 <= (size_t)cus) {
                const double t_one = (double)(32 + tab[i].bm) * ksteps * 128.0 / 45.0e3;     // us, one workgroup per strip
                double best = t_one;
                for (uint32_t ns = 2; ns <= 8 && strips * ns <= (size_t)cus && ksteps / ns >= 8; ++ns) {
                    const double t = t_one / ns + 4.5;
                    if (t < best) {
                        best = t;
                        *nsplit_out = ns;
                    }
                }
            }
            return i;
        }
    return vi;
}

// Up to 400 rows: an estimate of every row worth having there, fitted on 980 shapes (1 .. 400 rows x 512 .. 14336 columns x 512 ..
// 8192 elements of K; fp8, int8 and bf16, and fp8 with block scales), every row forced, as the geometric mean of weights streamed
// out of memory and weights resident.  The rules above were made on a few dozen shapes around 32 K steps, and with kernels that
// started later; measured against the fastest row they are 15 % behind on average, at worst twice its time: 48 x 1200 x 1024 int8
// 6.34 (two K slices) -> 4.05 us (16 x 16 tiles), 24 x 4432 x 1152 with block scales 7.52 -> 5.00, 110 x 1024 x 1280
// 7.90 -> 3.97, 124 x 3072 x 1792 8.97 -> 5.87.  What the estimate takes (few_rows_doubtful left out) is 2.4 % behind.
// A row costs `fixed`, and every round of `slots` workgroups per CU `round` plus its K steps at `alone` (few workgroups) .. `full`
// (all CUs at work) us each, or, where that is longer, `late` and B at `stream` us/MB.  (The eight waves of the skinny-M kernel
// take the steps in turn: halfway between the steps and the next multiple of eight.)
struct FewRowsModel {
    int slots;
    double fixed, round, alone, full, late, stream;
};
struct FewRowsTile {
    int bm, bn, kgroups;
    FewRowsModel plain, block;
};
const FewRowsTile kFewRows[] = {
    {16, 16, 8, {1, 1.51, 0.92, 0.0322, 0.0701, 2.91, 0.080}, {1, 1.60, 1.08, 0.0379, 0.0726, 1.23, 0.142}},
    {32, 16, 8, {1, 1.57, 1.20, 0.0405, 0.0760, 0.47, 0.279}, {1, 1.47, 1.39, 0.0571, 0.0861, 2.70, 0.201}},
    {16, 32, 8, {1, 1.37, 0.87, 0.0580, 0.1362, 3.22, 0.082}, {1, 1.11, 1.25, 0.0704, 0.1325, 3.30, 0.084}},
    {32, 32, 8, {1, 1.64, 1.27, 0.0619, 0.1399, 1.40, 0.231}, {1, 1.65, 1.38, 0.0742, 0.1468, 2.68, 0.118}},
    {64, 32, 8, {1, 1.54, 1.92, 0.0918, 0.1658, 0.00, 0.369}, {1, 1.98, 1.62, 0.1140, 0.1946, 1.52, 0.287}},
    {128, 32, 8, {1, 1.16, 3.28, 0.1514, 0.2366, 3.00, 0.250}, {1, 1.89, 2.83, 0.2255, 0.2790, 3.00, 0.250}},
    {64, 64, 8, {1, 1.04, 3.41, 0.1437, 0.1852, 2.72, 0.274}, {1, 1.89, 2.73, 0.1700, 0.2182, 3.17, 0.353}},
    {16, 32, 1, {5, 2.44, 0.00, 0.1888, 0.5637, 2.90, 0.186}, {8, 0.33, 1.73, 0.3657, 0.9489, 0.94, 0.503}},
    {64, 32, 1, {1, 1.51, 1.17, 0.2213, 0.2290, 3.64, 0.216}, {5, 1.74, 0.29, 0.3816, 1.1589, 2.88, 0.382}},
    {128, 32, 1, {1, 1.62, 1.46, 0.3006, 0.3251, 3.00, 0.250}, {4, 2.09, 0.00, 0.4505, 1.4063, 3.00, 0.250}},
    {64, 128, 1, {1, 1.47, 1.64, 0.5108, 0.5546, 3.00, 0.250}, {3, 2.03, 0.45, 0.6274, 1.4203, 3.00, 0.250}},
    {64, 128, 2, {1, 1.42, 2.72, 0.2736, 0.3462, 4.01, 0.312}, {1, 2.64, 1.61, 0.3269, 0.5024, 3.00, 0.250}},
    {128, 128, 2, {1, 1.97, 2.90, 0.3409, 0.5439, 3.00, 0.250}, {1, 2.50, 2.25, 0.4247, 0.6367, 3.00, 0.250}}};

// slices of K a launch has where the choice of a row has no opinion (see plan_nt)
uint32_t slices_for_few_tiles(size_t tiles, uint32_t ksteps, int cus) {
    if (tiles * 2 > (size_t)cus || ksteps < 8) return 1;
    // enough slices to cover the CUs about twice, at least 4 K steps each
    const uint32_t want = (uint32_t)((2 * (size_t)cus + tiles - 1) / tiles);
    return std::min<uint32_t>(want, ksteps / 4);
}

// K steps of a slice as a row counts them
inline double few_rows_steps(int kgroups, uint32_t steps) { return kgroups == 8 ? (steps + (steps + 7) / 8 * 8) * 0.5 : (double)steps; }
// us on `tiles` tiles
double few_rows_estimate(const FewRowsTile &t, size_t M, size_t N, size_t tiles, uint32_t ksteps, bool block, int cus, uint32_t nsplit) {
    const FewRowsModel &m = block ? t.block : t.plain;
    uint32_t steps = ksteps, slices = 1;
    if (nsplit > 1) {
        steps = (ksteps + nsplit - 1) / nsplit;
        slices = (ksteps + steps - 1) / steps;
    }
    const size_t wgs = tiles * slices, slots = (size_t)cus * m.slots;
    double load = 1, rounds = 1;
    if (wgs < slots) load = (double)wgs / slots;
    else rounds = (double)((wgs + slots - 1) / slots);
    double us = std::max(m.fixed + rounds * (m.round + few_rows_steps(t.kgroups, steps) * (m.alone + (m.full - m.alone) * load)),
                         m.late + (double)N * ksteps * 128e-6 * m.stream);
    if (slices > 1) us += 2.6 + (double)M * N * 4e-6 * (slices + 1) / 4.5;
    return us;
}
// ... and what it cannot be below on any number of tiles, K in one slice
inline double few_rows_least(const FewRowsTile &t, size_t N, uint32_t ksteps, bool block) {
    const FewRowsModel &m = block ? t.block : t.plain;
    return std::max(m.fixed + (m.round + few_rows_steps(t.kgroups, ksteps) * m.alone), m.late + (double)N * ksteps * 128e-6 * m.stream);
}

// Changes of row that the estimate gets wrong, by the tile of the rules and the one it puts ahead: both timed on 5700 shapes (1 .. 400 rows
// x 256 .. 100 000 columns x 512 .. 8192; fp8, int8, bf16 and the two with block scales), geometric mean of weights streamed and resident,
// and on 2500 of 17 .. 128 rows x 3000 .. 16384 x 4096 .. 8192 with block scales.
// At each, the gain that the estimate promises and what was measured.  Of the other 5250 changes ten are more than 5 % behind
// the rules, at worst 18 %; together they gain 26 %.
bool few_rows_doubtful(const FewRowsTile &rules, size_t rules_tiles, const FewRowsTile &t, size_t tiles, size_t M, size_t N, uint32_t ksteps,
                       bool block, int cus) {
    const size_t round = (size_t)cus;
    const bool two_rounds = N > 32 * round;                  // of strips of 32 columns
    auto is = [](const FewRowsTile &x, int bm, int bn, int kgroups) { return x.bm == bm && x.bn == bn && x.kgroups == kgroups; };
    // 1.33, 0.89: strips of 64 columns, up to 64 rows, where 32-column strips need a second round (64 x 128 tiles with block scales 0.78)
    // 1.11, 0.74: ... or with block scales 65 .. 128 rows from two such tiles of 64 rows to one of 128 x 32 (84 x 7632 x 6992 20.2 -> 30.7 us)
    if (is(rules, 64, 64, 8) && (M <= 64 || is(t, 128, 32, 8))) return true;
    // 1.10, 0.96: ... and 33 .. 64 rows from two K slices of 64 x 32 to two tiles of 32 rows over all of a K of 56 steps or more (39 x 4016 x
    // 8112 13.2 -> 14.3 us; 48 .. 55 steps 1.08 ahead)
    if (is(rules, 64, 32, 8) && is(t, 32, 32, 8) && rules_tiles < round && ksteps >= 56) return true;
    // 1.14, 0.77: 65 .. 128 rows x 11000 .. 16384 columns from 64 x 128 to one row of 128 x 128 tiles, two K groups each
    if (is(t, 128, 128, 2)) return true;
    // 1.18, 0.82: ... or to a second round of 64 x 64 tiles
    if (!block && is(rules, 64, 128, 2) && is(t, 64, 64, 8) && tiles > round) return true;
    // 1.15, 0.88: the same tile without its K groups; except strips of 16 x 32 in three rounds or more (1.24, 1.28), and in two up to 12 steps
    // (1.24, 1.05; from 13 steps on 1.19, 0.92)
    if (t.bm == rules.bm && t.bn == rules.bn && t.kgroups == 1)
        return !(is(rules, 16, 32, 8) && (ksteps <= 12 || rules_tiles > 2 * round));
    // 1.16, 0.81: strips of 16 x 32, many on a CU, to one row of the skinny-M kernel a CU, in a second round
    if (is(rules, 16, 32, 1) && t.kgroups == 8 && two_rounds) return true;
    // 1.11, 0.93: tiles of 64 rows on eight waves of which some have no step
    if (t.kgroups == 8 && t.bm == 64 && ksteps < 8 && t.bn == (block ? 64 : 32)) return true;
    // 1.06, 1.00, at worst 0.89: strips of 16 columns in a third round
    if (!block && is(t, 16, 16, 8) && tiles > 2 * round) return true;
    // 1.21, 0.89: block scales, strips of 64 x 32 to anything else in a second round; from 12 steps on, to 64 x 128 in a third round 1.44, 1.15
    // and to the skinny-M kernel in a second 1.09, 1.05
    return block && is(rules, 64, 32, 1) && two_rounds &&
           !(ksteps >= 12 && (rules_tiles > 2 * round ? t.bm == 64 && t.bn == 128 : t.kgroups == 8));
}

// How many partial sums an element of C is made of: K groups of the row times K slices.
struct PartialSums {
    uint32_t groups, slices;
};
// Are sums in parts `b` no further from 64 bits than in parts `a`, as far as the output shows it?  Only fp32 does, and not where the
// sums are exact (int8 with one scale) or the matrix instruction's own rounding covers them (fp8: 1.5e-5 of the result in any order).
// 16-bit operands: the more parts the shorter the chains.  Relative error, 1e-8, bf16 at 8 / 16 / 31 K steps: one chain 12.3 / 18.2 /
// 26.5, two groups 8.9 / 12.8 / 18.2, two groups in four slices - / 7.7 / 9.8, eight groups 7.0 / 8.2 / 10.1, in two slices 6.5 / 7.6 / 8.6.
// int8 blocks: no such order (eight groups add few blocks each and round once more where they meet; one chain 5.9 / 7.8 / 10.4, two
// groups 5.5 / 6.6 / 8.1, eight 6.6 / 6.9 / 7.4), so only the same parts.
bool output_shows_sums(int arith, bool block, int out_dtype) {
    return out_dtype == QGEMM_DT_F32 && arith != AR_F8 && (arith != AR_I8 || block);
}
bool sums_as_exact(int arith, bool block, int out_dtype, PartialSums a, PartialSums b) {
    if (!output_shows_sums(arith, block, out_dtype)) return true;
    if (a.groups == b.groups && a.slices == b.slices) return true;
    return !block && b.groups * b.slices > a.groups * a.slices;
}

// The row of the rules, or where the estimate puts another one 3 % ahead of it that one, with no more K slices than the rules asked
// for (so that no call needs a workspace that did not need one).  Below 32 K steps, and with block scales up to 128 rows; from 32
// K steps on the rules above are 7 - 8 % behind, and their choice, which was measured with streamed weights, stays.  With 8 K steps
// and one scale the waves of the skinny-M kernel have a single step each and the estimate is less sure of them: 13 %.
// (whole: not the rows or columns beside a first launch, whose estimate the split of the two was made with)
// Where an fp32 output would show it, only rows whose sums are as exact as those of the rules' row (sums_as_exact): bf16 8 x 8788 x 544
// is 7.4e-8 of the result off on eight groups, which the rules ask for, 13.0e-8 in the one chain that the estimate likes.
int choose_variant(const Variant *tab, int count, size_t M, size_t N, size_t ksteps, bool block, int kmaj, int cus,
                   bool may_split, bool whole, int out_dtype, uint32_t *nsplit_out, RowCopies copies) {
    const int vi = choose_by_rules(tab, count, M, N, ksteps, block, kmaj, cus, may_split, nsplit_out, copies);
    if (vi < 0 || kmaj || !whole || M > 400 || tab[vi].arith == AR_F8W || !g_ctx.row_estimate || !g_ctx.small_tiles || !(ksteps < 32 || (block && M <= 128))) return vi;
    // (tile sides are powers of two)
    auto tiles_of = [&](int bm, int bn) { return ((M + bm - 1) >> __builtin_ctz(bm)) * ((N + bn - 1) >> __builtin_ctz(bn)); };
    const uint32_t steps = (uint32_t)ksteps;
    uint32_t asked = std::max<uint32_t>(1, *nsplit_out);
    if (*nsplit_out == 0 && may_split) asked = std::max<uint32_t>(1, slices_for_few_tiles(tiles_of(tab[vi].bm, tab[vi].bn), steps, cus));
    const FewRowsTile *rules = nullptr;
    for (const FewRowsTile &t : kFewRows)
        if (t.bm == tab[vi].bm && t.bn == tab[vi].bn && t.kgroups == tab[vi].kgroups) rules = &t;
    if (!rules) return vi;
    const size_t rules_tiles = tiles_of(rules->bm, rules->bn);
    // Margins: with streamed weights tiles of a second round, rows without a K split inside the workgroup where they stand several on a CU,
    // and those rows behind long loops with block scales cost more than the estimate says, which is a mean of streamed and
    // resident weights.  What each keeps back, 110 shapes that it decides: 0.87 9.8 % of gain and one shape more than 5 % slower, 0.93 and 1.15
    // together 7.4 % and seven, 1.12 9.5 % and eight.
    const bool one_round = rules_tiles * asked <= (size_t)cus;
    const FewRowsTile *best = nullptr;
    uint32_t best_ns = *nsplit_out;
    double best_t = few_rows_estimate(*rules, M, N, rules_tiles, steps, block, cus, asked) * (ksteps == 8 && !block ? 0.87 : ksteps >= 32 ? 0.93 : 0.97);
    // (this is on the way of every eager call: rows that cannot win on any number of tiles are left out first, which in one slice is
    // most of them, and only the winner is looked up in the table.  Host time of qgemm_plan, us, rules alone / every row of the table priced /
    // so: fp8 1 x 2048 x 1024 0.13 / 0.30 / 0.17, bf16 64 x 4096 x 1024 0.14 / 0.46 / 0.24, block scales 100 x 4096 x 2992 0.39 / 0.69 / 0.42,
    // 300 x 8192 x 3968 0.62 / 0.90 / 0.62)
    for (const FewRowsTile &t : kFewRows) {
        if ((t.bm > 32 && (size_t)t.bm > 2 * M) || M > 12 * (size_t)t.bm) continue;
        if (asked == 1 && few_rows_least(t, N, steps, block) >= best_t) continue;
        const size_t tiles = tiles_of(t.bm, t.bn);
        if (tiles > 1400 || few_rows_doubtful(*rules, rules_tiles, t, tiles, M, N, steps, block, cus)) continue;
        for (uint32_t ns = 1; ns <= 8 && ns <= asked; ns *= 2) {
            if (ns > 1 && (ksteps / ns < 6 || tiles * ns > 300)) break;
            if (!sums_as_exact(tab[vi].arith, block, out_dtype, {(uint32_t)rules->kgroups, asked}, {(uint32_t)t.kgroups, ns})) continue;
            double us = few_rows_estimate(t, M, N, tiles, steps, block, cus, ns);
            if (tiles * ns > (size_t)cus && (one_round || t.kgroups == 1)) us *= 1.12;
            if (ksteps >= 32 && t.kgroups != 8) us *= 1.15;
            if (us < best_t) {
                best = &t;
                best_ns = ns;
                best_t = us;
            }
        }
    }
    if (!best) return vi;
    for (int i = 0; i < count; ++i)
        if (tab[i].bm == best->bm && tab[i].bn == best->bn && tab[i].kgroups == best->kgroups) {
            *nsplit_out = best_ns;
            return i;
        }
    return vi;
}

int choose_tile(const Variant *tab, int count, size_t M, size_t N, size_t ksteps, bool block, int kmaj, int cus,
                bool may_split, uint32_t *nsplit_out, RowCopies copies) {
    *nsplit_out = 0;                                       // 0: no opinion, plan_nt decides
    if (M > 64 || kmaj) {
        int vi = choose_by_cost(tab, count, M, N, ksteps, block, cus, may_split, nsplit_out, nullptr, copies);
        if (vi >= 0) {
            // 256 x 256, int8 and 16-bit types: the 8-wave form needs fewer cycles per tile, the 4-wave form a third
            // fewer LDS reads.  With at least one full round of CUs the part runs at its power limit and the 4-wave
            // form wins by 2 - 3 % (higher clock; level in the partly filled rounds of such shapes); with fewer
            // tiles than CUs the clock is not what limits and the 8-wave form wins by 1 - 5 %.  (fp8 per-matrix:
            // the 4-wave form either way; block scales: 8 waves.)
            const Variant &v = tab[vi];
            const size_t tiles = ((M + 255) / 256) * ((N + 255) / 256);
            if (v.bm == 256 && v.bn == 256 && v.threads == 512 && !block && kmaj == 0 && *nsplit_out <= 1 && tiles >= (size_t)cus)
                for (int i = 0; i < count; ++i)
                    if (tab[i].bm == 256 && tab[i].bn == 256 && tab[i].threads == 256 && tab[i].lds_bytes == v.lds_bytes &&
                        !std::strcmp(tab[i].name, "256x256_w2x2_solo"))
                        vi = i;
            return vi;
        }
        *nsplit_out = 0;
    }
    const size_t m16 = std::max<size_t>(16, (M + 15) / 16 * 16);
    const size_t target = std::min<size_t>(m16, 128);   // shorter tiles would stream B more than once
    int best = -1;
    size_t best_area = 0;
    for (int i = 0; i < count; ++i) {
        if (!tab[i].auto_ok || is_kgroup_row(tab[i]) || (size_t)tab[i].bm > m16 || (size_t)tab[i].bm < target) continue;
        const size_t tiles = ((M + tab[i].bm - 1) / tab[i].bm) * ((N + tab[i].bn - 1) / tab[i].bn);
        const size_t area = (size_t)tab[i].bm * tab[i].bn;
        if (tiles * 4 >= (size_t)cus * 3 && area > best_area) {     // at least three quarters of the CUs get a tile
            best = i;
            best_area = area;
        }
    }
    if (best >= 0) return best;
    // Nothing fills the CUs: 16 x 32 tiles, several over the rows, while they make at most two rounds (B is read once
    // per 16 rows then, out of the L2: 48 x 4096 x 4096 fp8 10.5 us against 14.7 with a 64 x 128 tile and a K split);
    // else the shortest tile that covers the rows, the narrowest of that height.
    for (int i = 0; i < count; ++i)
        if (tab[i].auto_ok && tab[i].bm == 16 && tab[i].bn == 32 && ((M + 15) / 16) * ((N + 31) / 32) <= 2 * (size_t)cus) return i;
    for (int i = 0; i < count; ++i) {
        if (!tab[i].auto_ok || is_kgroup_row(tab[i]) || (size_t)tab[i].bm < target) continue;
        if (best < 0 || tab[i].bm < tab[best].bm || (tab[i].bm == tab[best].bm && tab[i].bn < tab[best].bn)) best = i;
    }
    return best;
}

// Should the problem run with these operands read K-major, as they are stored (strides between k rows given)?
// Yes when the shape fits and the estimate for the K-major family beats the K-contiguous kernel plus the transpose
// launches in front of it (4 us per operand and the matrix read and written at 5.5 TB/s; block scales 2048^3 in the
// reference's layout: 23.3 us as stored, 29.3 us behind two transposes; 1024 x 4096 x 4096: 39.9 against 37.2).
// The simple-pipeline rows pay 15 % on top of the estimate for their transposing reads.  The 256 x 128 row with
// copying waves needs per K step what its K-contiguous form needs, and is taken up to 2.5 % above the other route's
// estimate (which counts a row split where the K-contiguous plan would make one, and runs low for one round of
// 256 x 256 tiles behind transposes).  Measured, as stored against through the transposes, us: fp8_mm 4096^3
// 65.3 / 73.9, 2048 x 4096 x 4096 35.0 / 46.9, 3072 x 8192 x 4096 102.8 / 110.4, bf16 with B stored K x N 4096^3
// 101.4 / 109.6, 2048 x 8192 x 8192 194.6 / 223.3, 2048 x 4096 x 4096 52.2 / 68.2; the largest shapes keep the
// transposes and the 256 x 256 tile: config 4 in the reference's storage 207.8 / 194.6, 8192^3 506.6 / 465.2 (fp8_mm)
// and 786.0 / 742.4 (bf16), 6144^3 240.3 / 229.6 and 356.7 / 348.6.  Over 19 shapes the ratio of the two estimates is
// within 4 % of the measured ratio on 15 and the choice is the faster route on all but bf16 3072 x 4096 x 4096 (4 %).
bool kmajor_problem_ok(NtProblem q, int kmaj, size_t lda_bytes, size_t ldb_bytes) {
    if (!g_ctx.kmajor) return false;
    q.kmaj = kmaj;
    q.lda_bytes = lda_bytes;
    q.ldb_bytes = ldb_bytes;
    if (!mfma_shape_ok(q)) return false;
    int count = 0, count_km = 0;
    const Variant *tab = table_for(q.arith, q.block, 0, &count), *tab_km = table_for(q.arith, q.block, kmaj, &count_km);
    if (!tab || !tab_km) return false;
    if (forced()) return row_by_name(tab_km, count_km, g_ctx.force_config) >= 0;   // a forced row: as stored where the K-major family has it
    if (g_ctx.kmajor == 2) return true;                                        // measurements: as stored wherever possible
    const size_t ksteps = ksteps_of(q);
    const bool may_split = q.split_k == 0;
    uint32_t ns = 0;
    double t_km = 0, t_nt = 8.0;                    // a skinny K-contiguous launch: about 8 us
    const int vk = choose_by_cost(tab_km, count_km, q.M, q.N, ksteps, q.block, g_ctx.num_cus, may_split, &ns, &t_km, copies_of(q));
    if (vk < 0) return false;
    if (q.M > 128 && choose_by_cost(tab, count, q.M, q.N, ksteps, q.block, g_ctx.num_cus, may_split, &ns, &t_nt) < 0)
        return false;
    if (q.M > 128 && may_split) {                    // (the K-contiguous route may split the rows into two launches)
        double t_single = 0, t_split = 0;
        uint32_t ns1 = 0;
        if (choose_by_cost(tab, count, q.M, q.N, ksteps, q.block, g_ctx.num_cus, false, &ns1, &t_single) >= 0) {
            if (rows_for_full_rounds(tab, count, q.M, q.N, ksteps, q.block, g_ctx.num_cus, t_single, &t_split) && t_split < t_nt)
                t_nt = t_split;
            if (cols_for_full_rounds(tab, count, q.M, q.N, ksteps, q.block, g_ctx.num_cus, t_single, &t_split) && t_split < t_nt)
                t_nt = t_split;
        }
    }
    const double kbytes = (double)q.Kbytes;         // K * element size
    t_nt += 1.0;                                     // a transpose launch per operand: 4 us and the matrix read and written
    if (kmaj & 1) t_nt += 4.0 + 2.0 * (double)q.M * kbytes / 5.5e6;
    if (kmaj & 2) t_nt += 4.0 + 2.0 * (double)q.N * kbytes / 5.5e6;
    return tab_km[vk].copy_waves ? t_km <= 1.025 * t_nt : 1.15 * t_km <= t_nt;
}

struct Plan {
    const Variant *v = nullptr;
    GemmArgs a;
    size_t tiles = 0;
    size_t split_bytes = 0;   // workspace the K split needs (0 when not split)
    // Row split: this plan covers rows [0, m_main) of the problem and `rest` the rows below, as a second launch
    // with a tile of its own (m_main = 0: no split, the plan covers everything).
    size_t m_main = 0;
    // Column split, the same along N: columns [0, n_main) here, the columns to the right in `rest` (never both splits)
    size_t n_main = 0;
    std::unique_ptr<Plan> rest;
};

// elements the tiles of a launch compute beyond the M x N asked for
size_t padded_area(size_t bm, size_t bn, size_t M, size_t N) {
    return ((M + bm - 1) / bm * bm) * ((N + bn - 1) / bn * bn) - M * N;
}

// Rows of the problem that 256 x 256 tiles should take when such tiles do not fill the last round of CUs.
// 576 tiles on 256 CUs are 2.25 rounds and cost three: the rows of the two full rounds go to one launch, and the
// rows below to whatever the tile choice likes best for them (smaller tiles, which fill the CUs; the skinny-M
// kernel for up to 128 rows).  Also where a single launch would rather take smaller tiles for everything
// (5000 x 4096 x 7168: 1.25 rounds of 256 x 256 tiles; fp8 148 us as one launch of 128 x 128 tiles, 113 us as 4096 rows
// of 256 x 256 tiles and 904 rows of 128 x 128 ones; 7000 x 7168 x 2048: 106 -> 93 us with the last 88 rows on the
// skinny-M kernel).  Returns 0 for "do not split": when the estimate of the two launches (plus 6 us for the
// second) is not at least 2.5 % below the estimate t_single of the one (config 4 with block scales: estimate
// 160.5 against 164.8 us, 2.6 %; measured 170.9 - 172.5 against 175.1 - 176.9 us in three interleaved runs).
size_t rows_for_full_rounds(const Variant *tab, int count, size_t M, size_t N, size_t ksteps, bool block, int cus,
                            double t_single, double *t_split, size_t *padding, RowCopies copies) {
    if (!g_ctx.row_split) return 0;
    const size_t tn = (N + 255) / 256, tiles = ((M + 255) / 256) * tn, full = tiles / cus;
    if (full == 0 || tiles % cus == 0) return 0;
    const size_t m_main = (full * cus / tn) * 256;
    if (m_main == 0 || m_main >= M) return 0;
    uint32_t ns = 0;
    double t_main = 0, t_rest = 0;
    const int vm = choose_by_cost(tab, count, m_main, N, ksteps, block, cus, false, &ns, &t_main, copies);
    if (vm < 0 || tab[vm].bm != 256 || tab[vm].bn != 256) return 0;
    size_t pad = padded_area(256, 256, m_main, N);
    if (M - m_main > 128) {
        const int vr = choose_by_cost(tab, count, M - m_main, N, ksteps, block, cus, false, &ns, &t_rest, copies);
        if (vr < 0) return 0;
        pad += padded_area(tab[vr].bm, tab[vr].bn, M - m_main, N);
    } else {
        t_rest = 5.0 + (double)N * ksteps * 128.0 / 4.0e6;      // B streamed once, about 4 TB/s
    }
    if (t_split) *t_split = t_main + t_rest + 6.0;
    if (padding) *padding = pad;
    if (g_ctx.row_split == 2) return m_main;
    return t_main + t_rest + 6.0 < 0.975 * t_single ? m_main : 0;
}

// The same along N, for shapes whose row tiles do not divide the full rounds but whose column tiles do:
// 4096 x 14336 x 4096 is 16 x 56 tiles, 3.5 rounds; 13 of its 16 row tiles are 2.84 rounds and still cost three, while
// 48 of its 56 column tiles are exactly three, and the 4096 x 2048 to their right fill a round of smaller tiles.
// Returns the columns of the first launch (a multiple of 256, so the right part starts on a 128-block of b_scale).
size_t cols_for_full_rounds(const Variant *tab, int count, size_t M, size_t N, size_t ksteps, bool block, int cus,
                            double t_single, double *t_split, size_t *padding, bool whatever_the_estimate, RowCopies copies) {
    if (!g_ctx.row_split) return 0;
    const size_t tm = (M + 255) / 256, tiles = tm * ((N + 255) / 256), full = tiles / cus;
    if (full == 0 || tiles % cus == 0) return 0;
    const size_t n_main = (full * cus / tm) * 256;
    if (n_main == 0 || n_main >= N) return 0;
    uint32_t ns = 0;
    double t_main = 0, t_rest = 0;
    const int vm = choose_by_cost(tab, count, M, n_main, ksteps, block, cus, false, &ns, &t_main, copies);
    if (vm < 0 || tab[vm].bm != 256 || tab[vm].bn != 256) return 0;
    const int vr = choose_by_cost(tab, count, M, N - n_main, ksteps, block, cus, false, &ns, &t_rest, copies);
    if (vr < 0) return 0;
    if (t_split) *t_split = t_main + t_rest + 6.0;
    if (padding) *padding = padded_area(256, 256, M, n_main) + padded_area(tab[vr].bm, tab[vr].bn, M, N - n_main);
    if (g_ctx.row_split == 3 || whatever_the_estimate) return n_main;
    return t_main + t_rest + 6.0 < 0.975 * t_single ? n_main : 0;
}

int plan_nt(const NtProblem &q, Plan &pl, bool may_split_rows = true) {
    int count = 0;
    const Variant *tab = table_for(q.arith, q.block, q.kmaj, &count);
    if (!tab) return QGEMM_ERR_UNSUPPORTED;
    uint32_t model_split = 0;
    int vi = choose_variant(tab, count, q.M, q.N, ksteps_of(q), q.block, q.kmaj, g_ctx.num_cus, q.split_k == 0 && !q.no_planes, may_split_rows, q.out_dtype,
                            &model_split, copies_of(q));
    if (may_split_rows && vi >= 0 && !forced() && (g_ctx.force_split <= 0 || q.no_planes) && q.split_k == 0 && model_split <= 1 &&
        q.M > 128 && q.kmaj == 0) {
        uint32_t ns = 0;
        double t_single = 0;
        const int ci = choose_by_cost(tab, count, q.M, q.N, ksteps_of(q), q.block, g_ctx.num_cus, false, &ns, &t_single, copies_of(q));
        if (ci >= 0 && tab[ci].bm == tab[vi].bm && tab[ci].bn == tab[vi].bn && tab[ci].kgroups == tab[vi].kgroups) {
            double t_rows = 0, t_cols = 0;
            size_t pad_rows = 0, pad_cols = 0;
            size_t m_main = rows_for_full_rounds(tab, count, q.M, q.N, ksteps_of(q), q.block, g_ctx.num_cus, t_single, &t_rows, &pad_rows, copies_of(q));
            size_t n_main = g_ctx.row_split == 2 ? 0
                                : cols_for_full_rounds(tab, count, q.M, q.N, ksteps_of(q), q.block, g_ctx.num_cus, t_single, &t_cols, &pad_cols, m_main != 0, copies_of(q));
            // The columns by themselves where they are estimated at least 2.5 % ahead of the single launch, as the rows are.
            // Where the rows pass that test, the columns take their place if they are estimated 5 % faster, or no more
            // than 5 % slower with tiles that compute less beyond the matrix: the estimate prices tiles, not the rows in
            // them that count, and a full round of 256 tiles more than one of 252.  Config 4 is 14 row bands of 256 x 256
            // tiles and 2560 rows below on 192 x 256 ones, the last band of which is two thirds padding, or 10 column bands
            // and 2048 columns to the right that 32 x 8 such tiles cover exactly: 172.8 against 170.8 us, and 143.0
            // against 139.8 with per-matrix scales.  (Measured, the two are never further apart than 2.3 %.)
            if (g_ctx.row_split == 3) m_main = 0;
            if (m_main && n_main) {
                const bool cols = t_cols < 0.95 * t_rows || (t_cols <= 1.05 * t_rows && pad_cols < pad_rows);
                (cols ? m_main : n_main) = 0;
            }
            if (m_main || n_main) {
                NtProblem q_main = q, q_rest = q;
                if (m_main) {
                    q_main.M = m_main;
                    q_rest.M = q.M - m_main;
                } else {
                    q_main.N = n_main;
                    q_rest.N = q.N - n_main;
                }
                int st = plan_nt(q_main, pl, false);
                if (st != QGEMM_OK) return st;
                pl.rest.reset(new Plan());
                st = plan_nt(q_rest, *pl.rest, false);
                if (st != QGEMM_OK) return st;
                pl.m_main = m_main;
                pl.n_main = n_main;
                pl.split_bytes = std::max(pl.split_bytes, pl.rest->split_bytes);     // one after the other on the stream
                return QGEMM_OK;
            }
        }
    }
    if (forced()) {
        vi = row_by_name(tab, count, g_ctx.force_config);       // (a name this family does not have: unsupported)
        model_split = 0;
    }
    if (vi < 0) return QGEMM_ERR_UNSUPPORTED;
    const Variant &v = tab[vi];
    pl.v = &v;
    GemmArgs &a = pl.a;
    std::memset(&a, 0, sizeof(a));
    a.as = q.as;
    a.bs = q.bs;
    a.M = (uint32_t)q.M;
    a.N = (uint32_t)q.N;
    a.ksteps = (uint32_t)ksteps_of(q);
    a.k_tail = (uint32_t)(q.Kbytes % 128);
    a.k_rest = (uint32_t)q.k_rest;
    if (q.k_rest && !v.launch_rest) return QGEMM_ERR_UNSUPPORTED;
    a.lda = (uint32_t)q.lda_bytes;
    a.ldb = (uint32_t)q.ldb_bytes;
    const uint32_t tiles_m = (uint32_t)((q.M + v.bm - 1) / v.bm), tiles_n = (uint32_t)((q.N + v.bn - 1) / v.bn);
    a.map = make_tile_map(tiles_m, tiles_n, g_ctx.force_group_m > 0 ? (uint32_t)std::min<long>(g_ctx.force_group_m, kHeadGroupMax) : 8);
    a.inv_tiles_m = inverse_of(tiles_m);
    // Few rows (every workgroup streams a strip of B of its own out of memory, all of them at the same k): the workgroups
    // of column tile i (which share that strip of B and stay in step) start their K loops k_rot * i steps in and wrap
    // round, so that at any time the column tiles read at different offsets
    // inside their rows; with rows a power of two apart they otherwise all ask the same few memory channels
    // (16 x 28672 x 8192 fp8 with B out of HBM: 53 us from step 0, 45 - 46 us with 1, 2, 3 or 16 steps per workgroup,
    // 53 again with 32, i.e. 4 KiB; 8 steps are worse than none for the skinny-M kernel, whose waves share 16 steps).
    a.k_rot = g_ctx.k_rot >= 0 ? (uint32_t)g_ctx.k_rot : (q.M <= 256 ? 3u : 0u);
    a.as_ms = q.as_ms;
    a.as_ks = q.as_ks;
    a.bs_ns = q.bs_ns;
    a.bs_ks = q.bs_ks;
    a.nb_max = (uint32_t)((q.N + 127) / 128 - 1);
    // Copies of B with the streaming hint: where the launch reads B once (one row tile) and B is unlikely to be found in
    // the 256 MB memory-side cache by the next call (32 MiB or more: beyond what the L2s hold together).  With B out of
    // memory the hint is worth 2 - 12 %
    // (16 x 28672 x 8192 fp8 44.6 -> 40.2 us, 1 x 8192 x 8192 14.8 -> 13.0, 16 / 64 x 7168 x 2048 5.67 / 6.96 -> 5.40 / 6.75);
    // a caller who loops over one small B that sits in that cache loses 14 - 30 % with it (the same shapes with one B:
    // 3.56 / 5.04 -> 4.61 / 5.73), and with two row tiles sharing a strip of B it costs up to 8 %.  Option b_stream = 1
    // puts it on for every launch with one row tile: for callers whose weights do not stay in the cache between calls.
    a.b_stream = g_ctx.b_stream >= 0 ? (int)(g_ctx.b_stream && tiles_m == 1)
                                     : (tiles_m == 1 && q.N * q.Kbytes >= ((size_t)32 << 20));
    pl.tiles = (size_t)tiles_m * tiles_n;
    if (pl.tiles * 64 >= ((size_t)1 << 31)) return QGEMM_ERR_TOO_LARGE;

    uint32_t nsplit = 1;
    if (q.no_planes) nsplit = 1;
    else if (q.split_k > 1) nsplit = (uint32_t)q.split_k;
    else if (q.split_k == 0) {
        if (g_ctx.force_split > 0) nsplit = (uint32_t)g_ctx.force_split;
        else if (model_split > 0) nsplit = model_split;
        else nsplit = slices_for_few_tiles(pl.tiles, a.ksteps, g_ctx.num_cus);
    }
    nsplit = std::max<uint32_t>(1, std::min<uint32_t>(nsplit, a.ksteps));
    a.ksteps_per_split = (a.ksteps + nsplit - 1) / nsplit;
    nsplit = (a.ksteps + a.ksteps_per_split - 1) / a.ksteps_per_split;   // no empty slices
    a.nsplit = nsplit;
    a.inv_nsplit = inverse_of(nsplit);
    a.inv_nk = inverse_of(a.ksteps_per_split);
    a.inv_nk_last = inverse_of(a.ksteps - (nsplit - 1) * a.ksteps_per_split);
    // (a start further in than the launch head holds: the same start in a whole slice, and still a multiple of four where it and the
    // slices are, which run_nt asks about)
    if (a.k_rot > kHeadRotMax) a.k_rot = std::min(a.k_rot % a.ksteps_per_split, kHeadRotMax & ~3u);
    pl.split_bytes = nsplit > 1 ? q.M * q.N * 4 * (size_t)nsplit : 0;
    return QGEMM_OK;
}

const char *kmaj_suffix(int kmaj) { return kmaj == 3 ? "_tn" : (kmaj == 2 ? "_nn" : ""); }

// split_ws: workspace of pl.split_bytes (ignored when the plan does not split)
int run_nt(const NtProblem &q, Plan &pl, void *split_ws, hipStream_t stream) {
    if (pl.rest) {
        // rows [0, m_main) with this plan, the rows below with the other: operands, scales and C move down m_main rows
        NtProblem q_main = q, q_rest = q;
        if (pl.m_main) {
            q_main.M = pl.m_main;
            q_rest.M = q.M - pl.m_main;
            q_rest.A = (const char *)q.A + pl.m_main * q.lda_bytes;            // (K-contiguous operands only: plan_nt)
            q_rest.C = (char *)q.C + pl.m_main * q.ldc * dtype_bytes(q.out_dtype);
            if (q.block && q.as) q_rest.as = q.as + pl.m_main * q.as_ms;
        } else {
            // columns [0, n_main) with this plan, the columns to the right with the other: B, its scale blocks and C move
            q_main.N = pl.n_main;
            q_rest.N = q.N - pl.n_main;
            q_rest.B = (const char *)q.B + pl.n_main * q.ldb_bytes;
            q_rest.C = (char *)q.C + pl.n_main * dtype_bytes(q.out_dtype);
            if (q.block && q.bs) q_rest.bs = q.bs + (pl.n_main / 128) * q.bs_ns;
        }
        std::unique_ptr<Plan> rest = std::move(pl.rest);
        int st = run_nt(q_main, pl, split_ws, stream);
        const std::string first = g_ctx.last_config;
        if (st == QGEMM_OK) st = run_nt(q_rest, *rest, split_ws, stream);
        g_ctx.last_config = first + (pl.m_main ? "+" : "|") + g_ctx.last_config;        // rows + rows below, columns | columns to the right
        pl.rest = std::move(rest);
        return st;
    }
    const Variant &v = *pl.v;
    GemmArgs &a = pl.a;
    a.A = (const char *)q.A;
    a.B = (const char *)q.B;
    a.as = q.as;
    a.bs = q.bs;
    a.as_ms = q.as_ms;
    a.as_ks = q.as_ks;
    a.bs_ns = q.bs_ns;
    a.bs_ks = q.bs_ks;
    a.as_groups = 0;
    if (q.block && v.kgroups == 2 && g_ctx.as_groups) {
        // K-contiguous a_scale on the rows with two K groups: four K blocks of a row per copy (GemmArgs::as_groups), at any
        // 4-byte address (what a row's last group brings beyond the row nobody uses, past the end of the array it is
        // zeros: probed by qgemm_selftest_layouts).  A rotated start has to move, and to wrap round, by whole groups: it
        // moves by four steps a column tile where the slices are multiples of four, and is left out where they are
        // not (rows of B an odd number of K blocks apart do not ask the same memory channels anyway).  One K block per copy
        // against four, us, B streamed / resident: 500 x 4608 x 7200 53.2 / 41.7 -> 48.0 / 35.7, 512 x 4096 x 4224
        // 24.2 / 18.0 -> 20.3 / 15.9; up to 256 rows, with the rotation given up for it: 256 x 4608 x 7200 46.2 / 32.8 ->
        // 40.4 / 27.6, 160 x 7168 x 7200 42.5 / 30.0 -> 39.8 / 25.8, 256 x 7168 x 2176 14.3 / 10.4 -> 12.8 / 10.0.
        const bool slices4 = a.ksteps % 4 == 0 && (a.nsplit == 1 || a.ksteps_per_split % 4 == 0);
        const bool k_contiguous = q.as_ks == 1 && ((uintptr_t)q.as & 3u) == 0;
        if (k_contiguous && g_ctx.k_rot < 0 && a.k_rot) a.k_rot = slices4 ? 4 : 0;
        a.as_groups = k_contiguous && (a.k_rot == 0 || (slices4 && a.k_rot % 4 == 0));
    }
#if QGEMM_DEBUG_BUILD
    a.dbg_cycles = (unsigned long long *)g_ctx.dbg_ptr;
#endif
    const bool i32_acc = q.arith == AR_I8 && !q.block;        // (int8 with block scales sums in fp32)
    if (a.nsplit == 1) {
        a.C = (char *)q.C;
        a.ldc = (uint32_t)q.ldc;
        a.out_dtype = q.out_dtype;
        a.per_matrix_scale = q.per_matrix;
        const int ob = dtype_bytes(q.out_dtype);
        // 4-byte C over at least three rounds of 256 x 256 tiles: spread the write bursts (see gemm_nt_kernel)
        // (with fewer than 32 K steps the offsets are too large a part of a tile's time: 7000 x 7168 x 2048 int8 to
        // f32 128 us without, 139 us with)
        const bool spread = v.bm == 256 && v.bn == 256 && ob == 4 && pl.tiles >= 3 * (size_t)g_ctx.num_cus && a.ksteps >= 32;
        a.stagger = g_ctx.stagger >= 0 ? (uint32_t)g_ctx.stagger : (spread ? 1u : 0u);
        // 4-byte C from 256 x 256 tiles: ordinary stores up to two rounds of tiles, non-temporal ones (and the staggered
        // start) from three on.  int8 to f32, ordinary against non-temporal, interleaved: 4096^3 59.1 against 61.1 us,
        // 4096 x 8192 x 4096 (two rounds) 114.2 against 124.0, 6144 x 8192 x 4096 (three) 165.6 against 169.9 with the
        // stagger, 8192^3 (four) 399.4 against 386.9; 2-byte C and every other tile are 1 - 6 % slower with ordinary
        // stores (the row with copying waves, 192 x 256, the K-group rows, 64 x 128).
        a.c_plain = g_ctx.c_plain >= 0 ? (int)g_ctx.c_plain
                                       : (v.bm == 256 && v.bn == 256 && ob == 4 && pl.tiles < 3 * (size_t)g_ctx.num_cus);
        a.stagger_wgs = (uint32_t)g_ctx.num_cus;
        a.stagger_groups = (uint32_t)std::max<long>(1, std::min<long>(32, g_ctx.stagger_groups));
        hipError_t e = (a.k_rest ? v.launch_rest : v.launch)(a, (uint32_t)pl.tiles, stream);
        g_ctx.last_config = std::string(v.name) + kmaj_suffix(q.kmaj);
        return e == hipSuccess ? QGEMM_OK : QGEMM_ERR_LAUNCH;
    }

    // split-K: raw accumulators to the workspace, then one ordered reduction
    const size_t plane = q.M * q.N;
    a.C = (char *)split_ws;
    a.ldc = (uint32_t)q.N;
    a.split_stride = plane;
    a.out_dtype = i32_acc ? QGEMM_DT_I32 : QGEMM_DT_F32;
    a.per_matrix_scale = 0;
    hipError_t e = (a.k_rest ? v.launch_rest : v.launch)(a, (uint32_t)(pl.tiles * a.nsplit), stream);
    if (e != hipSuccess) return QGEMM_ERR_LAUNCH;

    const uint32_t per_row = (uint32_t)((q.N + 3) / 4);
    const dim3 grid((unsigned)((q.M * per_row + 255) / 256));
    e = launch_kernel(i32_acc ? splitk_reduce4_kernel<true> : splitk_reduce4_kernel<false>, grid, dim3(256), 0, stream, split_ws, q.C, q.as,
                       q.bs, (uint32_t)q.M, (uint32_t)q.N, a.nsplit, (uint32_t)q.ldc, inverse_of(per_row), (uint32_t)q.out_dtype,
                       (uint32_t)(q.per_matrix != 0));
    g_ctx.last_config = std::string(v.name) + kmaj_suffix(q.kmaj) + "_splitk" + std::to_string(a.nsplit);
    return e == hipSuccess ? QGEMM_OK : QGEMM_ERR_LAUNCH;
}

// plan, get the split workspace (plus `extra` bytes behind it for transposed operands), run
int launch_transpose(int elem_bytes, const void *in, void *out, size_t M, size_t N, hipStream_t stream);

// The MFMA kernels read a_scale with the rows contiguous (a_scale[m + kb*M], the reference's own
// arrangement, hip_mix_gemm_kernel.cpp:149): 64 rows of one K block are one 256-byte request.  Scales
// given with K contiguous (a_scale[m*KB + kb]) are brought to that form first: M*KB floats, a few
// microseconds.  `room` is where in the workspace the copy goes.
// Which arrangement of a_scale the kernels of a block-scaled plan read.  Most want it rows-contiguous
// (a_scale[m + kb * ld], what QGEMM_LAYOUT_REFERENCE passes); the block-scaled 8-wave solo kernel has a twin
// (GemmCfg::ASK, table name "<name>_ks") that reads it with the K blocks contiguous, as QGEMM_LAYOUT_K_CONTIGUOUS
// passes it, two K blocks per 8-byte load (any number of K blocks per row and per K slice: see below).
// Puts the right one of each pair into the plan.  Returns true when the plan then reads q's scales as they are,
// false when they first have to be copied rows-contiguous (scales_rows_contiguous).
bool settle_scale_layout(const NtProblem &q, Plan &pl) {
    if (!q.block) return true;
    int count = 0;
    const Variant *tab = table_for(q.arith, q.block, q.kmaj, &count);
    auto partner = [&](const Variant *v, bool ks) -> const Variant * {      // the row of the pair with / without ASK
        if (v->a_scale_k_contiguous == ks) return v;
        return (tab && v->twin >= 0 && v->twin < count) ? &tab[v->twin] : nullptr;
    };
    if (q.as_ms == 1) {                                  // rows-contiguous: every kernel but the twins reads that
        for (Plan *p = &pl; p; p = p->rest.get())
            if (const Variant *v = partner(p->v, false)) p->v = v;
        return true;
    }
    // some other arrangement (K-contiguous, as QGEMM_LAYOUT_K_CONTIGUOUS passes it): fine where every launch of the
    // plan either takes any strides (simple pipeline, skinny-M kernel) or has a twin for it
    // (a twin fetches the scales of Variant::ks_blocks K blocks of a row per load, two or four.  The one that fetches four
    // used to ask for rows and slices that are whole groups and took a transposed copy of a_scale otherwise: 2048 x 4096 x
    // 7200, 57 blocks, 66.4 -> 62.7 us, 1536 x 4096 x 4736 39.7 -> 32.3)
    bool as_is = true;
    for (const Plan *p = &pl; as_is && p; p = p->rest.get()) {
        if (p->v->a_scale_any_stride) continue;
        const Variant *twin = partner(p->v, true);
        if (!twin || q.as_ks != 1) {
            as_is = false;
            break;
        }
        // (any row length and any slice: loads of 8 bytes and LDS copies of 16 need 4-byte alignment only, what the load of
        // a row's last blocks brings beyond the row nobody uses, and at the end of the array the range check, which is
        // per dword, returns zeros for it: probed by qgemm_selftest_layouts.)
        as_is = (uintptr_t)q.as % 4 == 0 && (twin->ks_blocks != 4 || g_ctx.as_groups);
    }
    for (Plan *p = &pl; p; p = p->rest.get()) {
        if (p->v->a_scale_any_stride) continue;
        if (const Variant *v = partner(p->v, as_is)) p->v = v;
    }
    return as_is;
}

int scales_rows_contiguous(NtProblem &q, void *room, hipStream_t stream) {
    if (!q.block || q.as_ms == 1) return QGEMM_OK;
    const size_t KB = (q.Kbytes + 127) / 128;
    int st = launch_transpose(4, q.as, room, q.M, KB, stream);
    if (st != QGEMM_OK) return st;
    q.as = (const float *)room;
    q.as_ms = 1;
    q.as_ks = (uint32_t)q.M;
    return QGEMM_OK;
}
size_t scales_room(const NtProblem &q) {
    if (!q.block || q.as_ms == 1) return 0;
    return (q.M * ((q.Kbytes + 127) / 128) * 4 + 255) / 256 * 256;
}

int launch_nt(NtProblem q, hipStream_t stream) {
    Plan pl;
    int st = plan_nt(q, pl);
    if (st != QGEMM_OK) return st;
    void *ws = nullptr;
    const size_t split_room = (pl.split_bytes + 255) / 256 * 256;
    const size_t as_room = settle_scale_layout(q, pl) ? 0 : scales_room(q);
    if (split_room + as_room) {
        st = ensure_workspace_locked(split_room + as_room, stream, &ws);
        if (st != QGEMM_OK) return st;
    }
    if (as_room) {
        st = scales_rows_contiguous(q, (char *)ws + split_room, stream);      // (run_nt takes the scales from q)
        if (st != QGEMM_OK) return st;
    }
    return run_nt(q, pl, ws, stream);
}

// Tile side of the any-shape kernel (block: with block scales; km: an operand is transposed on the way): 128 x 128 tiles where
// they make at least one round of the CUs, half of one where operands are transposed: 64 x 64 / 128 x 128, us, K = 1001 and
// 3001: int8 512 x 4097 (132 tiles) 15.7 / 16.9 33.3 / 35.8, 1024 x 4097 (264) 22.7 / 22.5 52.2 / 44.1, 1500 x 4097 30.3 / 23.9
// 70.7 / 45.6; bf16 with B stored K x N 512 x 4097 33.2 / 30.6 87.8 / 78.1 (with fp32 output the smaller tiles, which add up more
// exactly: any_folded).
bool any_folded(int in_dtype, int out_dtype) { return dtype_bytes(in_dtype) == 2 && out_dtype == QGEMM_DT_F32; }
int any_tile(int in_dtype, int out_dtype, bool block, bool km, size_t M, size_t N) {
    if (block && (km || in_dtype == QGEMM_DT_I8)) return 64;        // (the partial products of int8 blocks would not fit the registers)
    const uint64_t wide = ((uint64_t)M + 127) / 128 * (((uint64_t)N + 127) / 128);
    return wide * (km && !any_folded(in_dtype, out_dtype) ? 2 : 1) >= (uint64_t)g_ctx.num_cus ? 128 : 64;
}

// Time of the any-shape kernel on operands that are not transposed on the way, us: 64 x 64 tiles, three on a CU, and 128 x 128, two
// on a CU.  (fitted as pack_pays says; fp8 on several 64 x 64 tiles a CU had been 15 % low in whole programs: block scales 1206 x 2045 x 2481 ran
// 43.9 us there, 37.0 packed)
double any_estimate(int in_dtype, int out_dtype, bool block, size_t M, size_t N, size_t K) {
    struct AnyModel {
        double shared64, alone64, fixed64, shared128, alone128, fixed128;
    };
    static const AnyModel kAny16{0.68, 0.45, 3.6, 1.29, 0.90, 10.4}, kAnyF8{0.72, 0.43, 3.2, 1.11, 0.72, 8.6},
        kAnyF8Block{0.82, 0.48, 2.7, 1.37, 0.99, 6.6}, kAnyI8{0.81, 0.47, 3.4, 1.37, 0.94, 8.9}, kAnyI8Block{1.18, 0.67, 1.6, 0, 0, 0};
    const AnyModel &m = in_dtype == QGEMM_DT_F8E4M3 ? (block ? kAnyF8Block : kAnyF8) : (in_dtype == QGEMM_DT_I8 ? (block ? kAnyI8Block : kAnyI8) : kAny16);
    const size_t cus = g_ctx.num_cus, tile = any_tile(in_dtype, out_dtype, block, false, M, N), steps = (K - 1) / (in_dtype == QGEMM_DT_I8 ? 128 : 64) + 1;
    const size_t tiles = ((M + tile - 1) / tile) * ((N + tile - 1) / tile);
    return tile == 64 ? rounds_cost(tiles, 3 * cus, cus, steps, m.shared64, m.alone64, m.fixed64)
                      : rounds_cost(tiles, 2 * cus, cus, steps, m.shared128, m.alone128, m.fixed128);
}

// ... and of the kernel for few rows (gemm_few_kernel), on 16 x 32 tiles up to 16 rows, else 32 x 32: every round of
// per_cu workgroups a CU costs `round` and its steps of 128 bytes at `alone` .. `full` (all CUs at work).  Fitted on 500 ragged shapes of 1 .. 128 rows x 512 ..
// 14336 columns x K = 301 .. 8191, graph replays: the faster of the two kernels by these estimates is 1 % behind the faster one
// measured, the any-shape kernel alone 78 %.  On average this kernel takes 1 / 2.18 of its time up to 16 rows, 1 / 1.96 up to 32,
// 1 / 1.55 up to 64 and 1 / 1.45 up to 128 (where it is behind on many columns: 64 x 8272 x 1109 bf16 13.8 against 17.1 us).
// 16-bit operands with fp32 output stay with the sums that any_folded says, and block scales with fp32 output below 3000 elements:
// a wave's few blocks are rounded once more where the partial sums meet (relative error, tiles / few rows, int8 16 x 300 x 1031
// 5.3e-8 / 6.4e-8, x 2051 6.8e-8 / 6.9e-8, but x 4001 8.4e-8 / 7.3e-8, fp8 x 7999 14.8e-8 / 8.3e-8; a 16-bit output hides it).
double few_estimate(int in_dtype, int out_dtype, bool block, size_t M, size_t N, size_t K) {
    // (its 512 threads for 32 columns stay below the 2^32 of a launch; the tiles have 256 for 64 or 128)
    if (M > 128 || (N + 31) / 32 >= ((size_t)1 << 23) || K >= ((size_t)1 << 30) || any_folded(in_dtype, out_dtype) || (block && out_dtype == QGEMM_DT_F32 && K < 3000)) return 1e30;
    if (g_ctx.few_rows != 1) return g_ctx.few_rows ? 0 : 1e30;
    struct FewModel {
        double fixed, round, alone, full;
        size_t per_cu;
    };
    static const FewModel k16[2] = {{1.39, 1.38, 0.098, 0.391, 2}, {2.28, 0.98, 0.154, 0.203, 1}}, kF8[2] = {{1.27, 1.27, 0.151, 0.446, 2}, {1.55, 1.41, 0.211, 0.268, 1}},
        kF8Block[2] = {{2.29, 0.32, 0.164, 0.252, 1}, {2.46, 0.53, 0.217, 0.285, 1}}, kI8[2] = {{1.19, 1.14, 0.136, 0.495, 2}, {2.11, 0.86, 0.183, 0.235, 1}},
        kI8Block[2] = {{1.22, 1.22, 0.133, 0.537, 2}, {2.12, 0.80, 0.199, 0.279, 1}};
    const FewModel &m = (in_dtype == QGEMM_DT_F8E4M3 ? (block ? kF8Block : kF8) : (in_dtype == QGEMM_DT_I8 ? (block ? kI8Block : kI8) : k16))[M > 16];
    const size_t slots = g_ctx.num_cus * m.per_cu, steps = (K * dtype_bytes(in_dtype) + 127) / 128, wgs = ((N + 31) / 32) * (M > 16 ? (M + 31) / 32 : 1);
    const double load = std::min(1.0, (double)wgs / slots), n = (steps + (steps + 7) / 8 * 8) * 0.5;
    return m.fixed + (double)((wgs + slots - 1) / slots) * (m.round + n * (m.alone + (m.full - m.alone) * load));
}

// Is a product on the any-shape path faster packed?  Estimates of both, in microseconds, fitted on ragged shapes (1 .. 4096
// rows x 1024 .. 7168 columns x K = 777 .. 7161; fp8 and int8 with one scale and with block scales, bf16), eager calls; two thresholds on
// the sizes, K and M N, were 21 % behind on average.  (The constant part of packing was 12 as long as every call that used the workspace
// recorded an event.  Unpacked / packed: int8 1002 x 2558 x 2881 with block scales 39.5 / 26.0, 353 x 11549 x 2008 30.5 / 26.1, bf16 485 x
// 1024 x 2075 18.6 / 16.0, 344 x 1664 x 515 8.0 / 9.5, fp8 501 x 2190 x 1638 18.6 / 16.1.)
// Operands that are transposed on the way (km) make the any-shape kernel twice as slow: thresholds do there (bf16 with B stored
// K x N 1024 x 2049 x 261 15.5 / 15.7, x 401 18.4 / 16.7).
// Rows at any address.  Share of them that start at no multiple of four (any distance between them), and RowCopies of such an operand: the
// copies of one CU, out of the L2 and with nothing else to do, reach 110 GB/s on whole lines, 75 off them and 36 where addresses are no
// multiple of four; fitted on products, 60 and 30.
double odd_rows(const void *p, size_t ld) {
    int odd = 0;
    for (size_t r = 0; r < 4; ++r) odd += ((uintptr_t)p + r * ld) % 4 != 0;
    return odd / 4.0;
}
double row_copy(const void *p, size_t ld) {
    if (((uintptr_t)p | ld) % 16 == 0) return 0;
    const double odd = odd_rows(p, ld);
    return 128.0 * ((1 - odd) / 60.0e3 + odd / 30.0e3);
}
// Time of a product on the MFMA rows, us: the tiles' estimate or, up to `few` rows, the skinny-M kernel's (see choose_variant), < 0 for none
double rows_estimate(const NtProblem &q, size_t few) {
    int count = 0;
    const Variant *tab = table_for(q.arith, q.block, q.kmaj, &count);
    uint32_t nsplit = 0;
    double t = 0;
    const size_t steps = ksteps_of(q), cus = g_ctx.num_cus;
    if (!tab) return -1;
    // (slices that the caller asks for are priced as those that the estimate would take)
    const int vi = choose_by_cost(tab, count, q.M, q.N, steps, q.block, (int)cus, q.split_k != 1 && !q.no_planes, &nsplit, &t, copies_of(q));
    if (vi < 0) return -1;
    if (q.kmaj) return tab[vi].copy_waves ? t : 1.15 * t;
    if (q.M <= few) {
        const size_t bm = q.M <= 16 ? 16 : (q.M <= 32 ? 32 : 64), strips = ((q.M + 63) / 64) * ((q.N + 31) / 32);
        const double piece = 128.0 / 50.0e3;
        t = std::min(t, std::max(4.0, (bm * std::max(piece, q.copies.a) + 32 * std::max(piece, q.copies.b)) * steps) * std::max(1.0, (double)strips / cus));
    }
    // (widening rows of 65 rows and more: the 64 x 64 form of the skinny-M kernel, as choose_by_rules takes it; without it fp8 with block
    // scales 184 x 4800 x 2037 ran on the any-shape kernel, 25.4 against 15.4 us)
    if (q.arith == AR_F8W && q.M > 64 && steps >= 16 && steps <= 48) {
        const size_t t64 = ((q.M + 63) / 64) * ((q.N + 63) / 64);
        if (t64 >= 128 && t64 <= cus) t = std::min(t, 0.52 * steps);
    }
    return t;
}
// What rows_estimate is never below: the start and the steps of the row that is fastest by itself, in eight slices where that is allowed.
// It spares products of few rows, whose calls the host bounds, two or three estimates of all rows (int8 block scales 5 x 1024 x 1213, one
// scale 1 x 2048 x 1037: 2.9 and 2.8 -> 2.2 us of host time a call).
double least_rows_estimate(const NtProblem &q) {
    const size_t steps = ksteps_of(q), eighth = (steps + 7) / 8;
    const bool wide = q.arith == AR_F8W, split = q.split_k != 1 && !q.no_planes;
    const TileModel *models = wide ? kWideTileModels : kTileModels;
    double t = wide || q.M <= 256 ? std::max(4.0, 0.12 * steps) : 1e30;             // (the skinny-M kernel)
    for (size_t i = 0; i < (wide ? std::size(kWideTileModels) : std::size(kTileModels)); ++i) {
        const TileModel &m = models[i];
        const double step = q.block ? std::min(m.blk_shared, m.blk_alone) : std::min(m.step_shared, m.step_alone);
        t = std::min(t, m.fixed + steps * step);
        if (split) t = std::min(t, m.fixed + eighth * step + 4.0);
    }
    return t;
}
// Packed: another launch that reads and writes both operands, then rows of whole K steps (q: the product; kbytes: its K).  Where an fp32
// output shows how sums are made, packed rows sum less exactly than the any-shape kernel (bf16 1445 x 640 x 1095 8.5e-8 / 7.8e-8 of the
// result) and keep the 12 us that a call with workspace once had as its constant part, so that no product comes to them for being faster now.
// (enough: an estimate that is known not to be below this is as good as none)
double packed_estimate(NtProblem q, size_t kbytes, double enough) {
    q.Kbytes = kbytes;
    q.kmaj = 0;
    q.copies = {};
    q.no_planes = false;
    const bool shows = output_shows_sums(q.arith, q.block, q.out_dtype);
    const double packing = (shows ? 12.0 : 6.3) + 0.2e-6 * (double)(q.M + q.N) * kbytes, rate = shows ? 1.0 : 1.05;
    if (packing + rate * least_rows_estimate(q) >= enough) return 1e30;
    const double t = rows_estimate(q, shows || q.arith != AR_F8W ? 256 : 64);
    return t < 0 ? 1e30 : packing + rate * t;
}
enum class Packing { NO, YES, UNLESS_FEW_ROWS };        // UNLESS_FEW_ROWS: gemm_few_kernel is faster still
Packing pack_pays(const NtProblem &q, int in_dtype, size_t K, bool km) {
    const size_t kbytes = K * dtype_bytes(in_dtype);
    if (km) return kbytes > 512 || (double)q.M * q.N >= 4e6 ? Packing::YES : Packing::NO;
    const double as_any = any_estimate(in_dtype, q.out_dtype, q.block, q.M, q.N, K), t_packed = packed_estimate(q, kbytes, as_any);
    if (t_packed >= as_any) return Packing::NO;
    return t_packed >= few_estimate(in_dtype, q.out_dtype, q.block, q.M, q.N, K) ? Packing::UNLESS_FEW_ROWS : Packing::YES;
}

// Operands that no MFMA kernel reads as they stand: pack_kernel writes what has to change into the workspace as rows of
// whole 128-byte K steps (one launch for both operands), and the K-contiguous kernels take it from there.  a_src / b_src:
// the operands as the caller has them, ld in bytes between rows, or, k_major, between rows of k.  q: everything else, with
// the caller's K.  *taken = false, and nothing launched, where the any-shape kernel is the one to run (launch_any), which
// needs no memory but the operands:
//   * calls that are captured and calls on the static scratch (which launch_unaligned may take first): replays of a captured graph, and the calls of several threads
//     on the scratch, are ordered by nobody, and packed operands in a block that they share would overwrite each other.
//     (The choice does not depend on how much room there happens to be: a call captured twice gives the same bits.)
//   * the device has no memory left for the workspace, or the shape exceeds what the MFMA kernels index;
//   * a product so small that the any-shape kernel is done first (pack_pays), or gemm_few_kernel, unless an fp32 output would show
//     that the packed rows sum more exactly than its eight parts (fp8 51 x 616 x 7907, seven slices: 6.3e-8 of the result off, in eight
//     parts 6.8e-8).
// fp8 operands run on the family that widens them to bf16 in front of the matrix core (AR_F8W), which adds in fp32 as these
// shapes have always been summed: the fp8 instructions keep some 18 bits of the largest product of a step.  Relative error
// against 64 bits, 301 x 100 x 4001 to fp32, one scale / block scales: in sequence 9.0e-8 / 1.1e-7, any-shape kernel 8.9e-8 /
// 1.1e-7, packed 6.9e-8 / 7.5e-8, packed on the fp8 instructions 1.4e-5.  It costs, us, fp8 instructions / widened: 500 x 4608 x
// 7161 41.8 / 61.1, block scales 44.9 / 65.3; 4096 x 4608 x 7161 125.5 / 239.9 and 148.7 / 267.7 (fp32 output, one thread per
// element before: 500 x 4608 x 7161 21 500 / 61).
struct SourceOperand {
    const void *p;
    size_t ld;
    bool k_major;
};
int launch_packed(NtProblem q, int in_dtype, const SourceOperand &a_src, const SourceOperand &b_src, size_t K, hipStream_t stream,
                  bool *taken) {
    *taken = false;
    const size_t eb = dtype_bytes(in_dtype);
    if (!g_ctx.any_shape) return QGEMM_OK;
    if (q.arith == AR_F8) q.arith = AR_F8W;
    const Packing pays = g_ctx.any_shape == 1 ? pack_pays(q, in_dtype, K, a_src.k_major || b_src.k_major) : Packing::YES;
    if (pays == Packing::NO || (pays == Packing::UNLESS_FEW_ROWS && !output_shows_sums(q.arith, q.block, q.out_dtype))) return QGEMM_OK;
    if (g_ctx.static_call || stream_is_capturing(stream)) return QGEMM_OK;
    if (q.M >= ((size_t)1 << 31) || q.N >= ((size_t)1 << 31) || K >= ((size_t)1 << 30)) return QGEMM_OK;
    // (a K that ends inside a 16-byte piece has to end in zeros in both operands)
    const bool whole = (K * eb) % 16 == 0;
    const SourceOperand *src[2] = {&a_src, &b_src};
    const size_t rows[2] = {q.M, q.N}, pitch = (K * eb + 127) / 128 * 128;
    bool pack[2];
    size_t room[2];
    for (int i = 0; i < 2; ++i) {
        pack[i] = !whole || src[i]->k_major || src[i]->ld % 16 != 0 || !aligned16(src[i]->p);
        room[i] = pack[i] ? rows[i] * pitch : 0;
        (i ? q.ldb_bytes : q.lda_bytes) = pack[i] ? pitch : src[i]->ld;
    }
    q.Kbytes = pack[0] && pack[1] ? pitch : K * eb;
    q.kmaj = 0;
    if (!mfma_shape_ok(q)) return QGEMM_OK;
    Plan pl;
    if (plan_nt(q, pl) != QGEMM_OK) return QGEMM_OK;
    if (pays == Packing::UNLESS_FEW_ROWS &&
        sums_as_exact(q.arith, q.block, q.out_dtype, {(uint32_t)pl.v->kgroups, pl.a.nsplit}, {8, 1})) return QGEMM_OK;
    const size_t split_room = (pl.split_bytes + 255) / 256 * 256;
    const size_t as_room = settle_scale_layout(q, pl) ? 0 : scales_room(q);
    PackArgs pa;
    std::memset(&pa, 0, sizeof(pa));
    uint64_t blocks = 0;
    for (int i = 0; i < 2; ++i) {
        if (!pack[i]) continue;
        PackOperand &o = pa.op[i];
        o.src = (const char *)src[i]->p;
        o.ld = src[i]->ld;
        o.rows = (uint32_t)rows[i];
        o.k = (uint32_t)K;
        o.pitch = (uint32_t)pitch;
        o.k_major = src[i]->k_major;
        uint64_t n;
        if (o.k_major) {        // tiles of 64 k x 256 rows (16-bit), 128 x 128 (bytes)
            o.tiles_k = (uint32_t)(eb == 2 ? pitch / 2 / 64 : pitch / 128);
            n = (uint64_t)o.tiles_k * (eb == 2 ? (rows[i] + 255) / 256 : (rows[i] + 127) / 128);
        } else {
            n = ((uint64_t)rows[i] * (pitch / 16) + 1023) / 1024;
            if (n >= ((uint64_t)1 << 22)) return QGEMM_OK;          // (32-bit piece numbers in pack_rows)
        }
        o.inv = inverse_of(o.k_major ? o.tiles_k : o.pitch / 16);
        o.blocks = (uint32_t)n;
        blocks += n;
    }
    if (blocks >= ((uint64_t)1 << 31)) return QGEMM_OK;
    void *ws = nullptr;
    int st = ensure_workspace_locked(split_room + as_room + room[0] + room[1], stream, &ws);
    if (st == QGEMM_ERR_ALLOC) return QGEMM_OK;
    *taken = true;
    if (st != QGEMM_OK) return st;
    char *at = (char *)ws + split_room + as_room, *bt = at + room[0];
    pa.op[0].dst = at;
    pa.op[1].dst = bt;
    q.A = pack[0] ? at : a_src.p;
    q.B = pack[1] ? bt : b_src.p;
    HIP_TRY(launch_kernel(eb == 2 ? pack_kernel<2> : pack_kernel<1>, dim3((unsigned)blocks), dim3(256), 0, stream, pa));
    if (as_room) {
        st = scales_rows_contiguous(q, (char *)ws + split_room, stream);
        if (st != QGEMM_OK) return st;
    }
    st = run_nt(q, pl, ws, stream);
    g_ctx.last_config = "pack+" + g_ctx.last_config;
    return st;
}

// Operands whose rows start or end anywhere, on the MFMA kernels as they stand: A, and B where it is N x K, may have any address, row
// distance and K of 16 bytes or more (see gemm_rest); B stored K x N only lets K end inside a chunk.  Which of the three ways a product
// goes is a matter of estimates, fitted on drawn ragged products: the tiles' own estimate runs low here, the copies being bound by a rate
// that LDS reads share, more so off multiples of four; on 70 programs that quantise and multiply, multiply or train a layer, operands changing
// from pass to pass, the way chosen is 2.3 % behind the fastest of the three.  Whole programs, us, as they stand / packed / any-shape kernel:
// fp16 510 x 3024 x 3026 with B stored K x N 23.5 / 29.4 / 41.0, 203 x 4320 x 1381 14.2 / 20.4 / 22.3, int8 7523 x 1024 x 1548 21.0 / 25.8 /
// 27.8, fp8 with block scales 164 x 1152 x 2407 15.2 / 17.4 / 25.4, training 2759 x 768 x 2304 55.7 / 59.1 / 76.3; but fp16 779 x 3968 x 3615 59.0 /
// 39.0 / 80.6, int8 1531 x 4100 x 3004 38.7 / 36.9 / 52.4, fp8 block 3942 x 4992 x 2901 135 / 122 / 187.
bool unaligned_pays(NtProblem &q, int in_dtype, size_t K, bool may_pack) {
    const double few = q.kmaj ? 1e30 : few_estimate(in_dtype, q.out_dtype, q.block, q.M, q.N, K);
    if (few < 1e30 && q.split_k == 0 && g_ctx.force_split <= 0) q.no_planes = true;       // (that kernel needs no second launch)
    constexpr double least = 4.3;                // (what a call takes the host)
    const double as_any = q.kmaj ? 1e30 : std::min(few, any_estimate(in_dtype, q.out_dtype, q.block, q.M, q.N, K));
    if (as_any <= least) return false;
    if (!q.kmaj && least_rows_estimate(q) * 1.25 * (few < 1e30 ? 1.35 : 1.0) >= as_any) return false;
    double t = rows_estimate(q, q.arith == AR_F8W ? 64 : 256);
    if (t < 0) return false;
    t *= 1.25 + (q.arith == AR_F8W ? 0 : 0.2) * (odd_rows(q.A, q.lda_bytes) + (q.kmaj ? 0 : odd_rows(q.B, q.ldb_bytes))) / 2;
    if (few < 1e30) t *= 1.35;
    if (std::max(least, t) >= as_any) return false;
    // (against packing the estimate of the widening rows runs low by 1.4, not 1.25: fp8 with block scales 2287 x 6912 x 859 as they stand /
    // packed 52.9 / 45.1 us, 2727 x 3136 x 2283 58.5 / 54.7, one scale 3384 x 6208 x 691 54.2 / 49.0)
    if (q.arith == AR_F8W) t *= 1.12;
    return !may_pack || t < packed_estimate(q, K * dtype_bytes(in_dtype), t * (1 + 1e-9));
}
// *taken as for launch_packed.
//   * Captured calls and calls on the static scratch run without a K split, also where the caller asks for one, and so without workspace.
//   * fp32 output that shows how sums are made (output_shows_sums): 16-bit operands, where the packed rows would run, in as many parts; not
//     with block scales, whose last block is folded in two parts here.
int launch_unaligned(NtProblem q, int in_dtype, const SourceOperand &a_src, const SourceOperand &b_src, size_t K, hipStream_t stream,
                     bool *taken) {
    *taken = false;
    const size_t eb = dtype_bytes(in_dtype);
    if (g_ctx.any_shape != 1 && g_ctx.any_shape != 3) return QGEMM_OK;
    if (q.arith == AR_F8) q.arith = AR_F8W;
    if (a_src.k_major || (b_src.k_major && (eb != 2 || b_src.ld % 16 != 0 || !aligned16(b_src.p)))) return QGEMM_OK;
    if (q.M >= ((size_t)1 << 31) || q.N >= ((size_t)1 << 31) || K >= ((size_t)1 << 30) || K * eb < 16) return QGEMM_OK;
    const bool may_pack = !g_ctx.static_call && !stream_is_capturing(stream), choose = g_ctx.any_shape == 1;
    const NtProblem whole = q;
    q.k_rest = K * eb % 16;
    q.Kbytes = K * eb - q.k_rest;
    q.A = a_src.p;
    q.B = b_src.p;
    q.lda_bytes = a_src.ld;
    q.ldb_bytes = b_src.ld;
    q.kmaj = b_src.k_major ? 2 : 0;
    q.copies = {row_copy(q.A, q.lda_bytes), q.kmaj ? 0 : row_copy(q.B, q.ldb_bytes)};
    if (!may_pack) {
        q.no_planes = true;
        q.split_k = std::min(q.split_k, 1);         // (1: nor a second launch)
    }
    // (K one element or more past whole steps, and as many slices asked for as there are steps with that one: packed rows have it)
    if (choose && q.split_k > 1 && ksteps_of(q) < std::min<size_t>(q.split_k, (K * eb + 127) / 128)) return QGEMM_OK;
    if (!mfma_sizes_ok(q) || (choose && !unaligned_pays(q, in_dtype, K, may_pack))) return QGEMM_OK;
    Plan pl;
    if (plan_nt(q, pl) != QGEMM_OK || !settle_scale_layout(q, pl)) return QGEMM_OK;
    if (choose && output_shows_sums(q.arith, q.block, q.out_dtype)) {
        NtProblem packed = whole;
        packed.arith = q.arith;
        packed.Kbytes = packed.lda_bytes = packed.ldb_bytes = (K * eb + 127) / 128 * 128;
        Plan other;
        if (!may_pack || q.block || q.arith == AR_F8W || pl.rest || pack_pays(packed, in_dtype, K, b_src.k_major) != Packing::YES || plan_nt(packed, other) != QGEMM_OK || other.rest ||
            !sums_as_exact(q.arith, q.block, q.out_dtype, {(uint32_t)other.v->kgroups, other.a.nsplit}, {(uint32_t)pl.v->kgroups, pl.a.nsplit}))
            return QGEMM_OK;
    }
    void *ws = nullptr;
    if (pl.split_bytes) {
        const int st = ensure_workspace_locked(pl.split_bytes, stream, &ws);
        if (st == QGEMM_ERR_ALLOC) return QGEMM_OK;
        if (st != QGEMM_OK) return st;
    }
    *taken = true;
    const int st = run_nt(q, pl, ws, stream);
    g_ctx.last_config = "unaligned+" + g_ctx.last_config;
    return st;
}

template <int DT, bool BLOCK>
int launch_any_t(AnyArgs &a, hipStream_t stream) {
    const uint64_t elements = (uint64_t)a.a.rows * a.b.rows;
    if (a.a.end - a.a.p < 16 || a.b.end - a.b.p < 16 || (a.K < 16 && elements * a.K <= 1000000)) {
        if (elements >= (uint64_t)1 << 39) return QGEMM_ERR_TOO_LARGE;     // grid limit
        g_ctx.last_any_kernel = "short";
        HIP_TRY(launch_kernel(gemm_short_kernel<DT, BLOCK>, dim3((unsigned)((elements + 255) / 256)), dim3(256), 0, stream, a));
        return QGEMM_OK;
    }
    constexpr int W = BLOCK && DT == QGEMM_DT_I8 ? 64 : 128;
    const bool km = a.a.k_major || a.b.k_major;
    if (!km && few_estimate(DT, a.out_dtype, BLOCK, a.a.rows, a.b.rows, a.K) < any_estimate(DT, a.out_dtype, BLOCK, a.a.rows, a.b.rows, a.K)) {
        constexpr int ARITH = DT == QGEMM_DT_I8 ? AR_I8 : DT == QGEMM_DT_F8E4M3 ? AR_F8W : DT == QGEMM_DT_BF16 ? AR_BF16 : AR_F16;
        const bool one = a.a.rows <= 16;
        g_ctx.last_any_kernel = one ? "few_rows_16x32" : "few_rows_32x32";
        const hipError_t e = launch_kernel(one ? gemm_few_kernel<ARITH, BLOCK, 1> : gemm_few_kernel<ARITH, BLOCK, 2>,
                                           dim3((a.b.rows + 31) / 32, one ? 1 : (a.a.rows + 31) / 32), dim3(512), 0, stream, a);
        return e == hipSuccess ? QGEMM_OK : QGEMM_ERR_LAUNCH;
    }
    const int T = any_tile(DT, a.out_dtype, BLOCK, km, a.a.rows, a.b.rows);
    const uint64_t tiles_m = ((uint64_t)a.a.rows + T - 1) / T, tiles_n = ((uint64_t)a.b.rows + T - 1) / T, tiles = tiles_m * tiles_n;
    if (tiles >= ((uint64_t)1 << 31)) return QGEMM_ERR_TOO_LARGE;    // grid limit
    a.map = make_tile_map((uint32_t)tiles_m, (uint32_t)tiles_n, 8);
    g_ctx.last_any_kernel = T == 64 ? "tiles_64x64" : "tiles_128x128";
    constexpr int SUM = BLOCK ? ANY_SCALED : ANY_CHAIN;
    auto kernel = T == 64 ? (km ? gemm_any_kernel<DT, SUM, 64, true> : gemm_any_kernel<DT, SUM, 64, false>)
                          : (km ? gemm_any_kernel<DT, SUM, BLOCK ? 64 : W, true> : gemm_any_kernel<DT, SUM, W, false>);
    if constexpr (DT == QGEMM_DT_BF16 || DT == QGEMM_DT_F16)
        if (T == 64 && any_folded(DT, a.out_dtype)) kernel = km ? gemm_any_kernel<DT, ANY_FOLDED, 64, true> : gemm_any_kernel<DT, ANY_FOLDED, 64, false>;
    HIP_TRY(launch_kernel(kernel, dim3((unsigned)tiles), dim3(256), 0, stream, a));
    return QGEMM_OK;
}

// The any-shape kernel on the operands as they stand (arguments as for launch_packed; M, N, K below 2^32)
int launch_any(const NtProblem &q, int in_dtype, const SourceOperand &a_src, const SourceOperand &b_src, size_t K, hipStream_t stream) {
    g_ctx.last_config = "strided_any_shape";
    const size_t eb = dtype_bytes(in_dtype);
    AnyArgs a;
    std::memset(&a, 0, sizeof(a));
    auto operand = [&](const SourceOperand &s, size_t rows) {
        const char *p = (const char *)s.p;
        return AnyOperand{p, p + (s.k_major ? (K - 1) * s.ld + rows * eb : (rows - 1) * s.ld + K * eb), s.ld, (uint32_t)rows, s.k_major};
    };
    a.a = operand(a_src, q.M);
    a.b = operand(b_src, q.N);
    a.C = q.C;
    a.as = q.as;
    a.bs = q.bs;
    a.K = (uint32_t)K;
    a.ldc = q.ldc;
    a.as_ms = q.as_ms;
    a.as_ks = q.as_ks;
    a.bs_ns = q.bs_ns;
    a.bs_ks = q.bs_ks;
    a.out_dtype = q.out_dtype;
    a.per_matrix_scale = q.per_matrix;
    switch (in_dtype) {
        case QGEMM_DT_I8: return q.block ? launch_any_t<QGEMM_DT_I8, true>(a, stream) : launch_any_t<QGEMM_DT_I8, false>(a, stream);
        case QGEMM_DT_F8E4M3: return q.block ? launch_any_t<QGEMM_DT_F8E4M3, true>(a, stream) : launch_any_t<QGEMM_DT_F8E4M3, false>(a, stream);
        case QGEMM_DT_BF16: return launch_any_t<QGEMM_DT_BF16, false>(a, stream);
        case QGEMM_DT_F16: return launch_any_t<QGEMM_DT_F16, false>(a, stream);
    }
    return QGEMM_ERR_UNSUPPORTED;
}

int launch_transpose(int elem_bytes, const void *in, void *out, size_t M, size_t N, hipStream_t stream) {
    if (M == 0 || N == 0) return QGEMM_OK;
    if (M >= ((size_t)1 << 31) || N >= ((size_t)1 << 31)) return QGEMM_ERR_TOO_LARGE;
    dim3 grid((unsigned)((N + 63) / 64), (unsigned)((M + 63) / 64));
    if (grid.y > 65535u * 1024u) return QGEMM_ERR_TOO_LARGE;
    // Sizes or addresses that rule out aligned 16-byte pieces take the same tiles with pieces at any address, stored in
    // parts on the edges.
    if (elem_bytes == 1) {
        const bool aligned = M % 16 == 0 && N % 4 == 0 && (uintptr_t)in % 4 == 0 && (uintptr_t)out % 16 == 0;
        const dim3 g((unsigned)((N + 127) / 128), (unsigned)((M + 127) / 128));
        const auto kernel = aligned ? transpose_bytes_kernel<true> : transpose_bytes_kernel<false>;
        HIP_TRY(launch_kernel(kernel, g, dim3(256), 0, stream, (const uint8_t *)in, (uint8_t *)out, (uint32_t)M, (uint32_t)N));
    } else if (elem_bytes == 2) {
        const bool aligned = M % 8 == 0 && N % 8 == 0 && (uintptr_t)in % 16 == 0 && (uintptr_t)out % 16 == 0;
        const dim3 g((unsigned)((N + 255) / 256), (unsigned)((M + 63) / 64));
        const auto kernel = aligned ? transpose_u16_kernel<true> : transpose_u16_kernel<false>;
        HIP_TRY(launch_kernel(kernel, g, dim3(256), 0, stream, (const uint16_t *)in, (uint16_t *)out, (uint32_t)M, (uint32_t)N));
    } else if (elem_bytes == 4) {
        HIP_TRY(launch_kernel(transpose_u32_kernel, grid, dim3(256), 0, stream, (const uint32_t *)in, (uint32_t *)out, (uint32_t)M, (uint32_t)N));
    } else {
        return QGEMM_ERR_UNSUPPORTED;
    }
    return QGEMM_OK;
}

// Slices of rows of the 1 x 128 quantiser (QuantArgs::rows_per_slice; blockIdx.y) and workgroups of one slice.  A launch takes fewer
// than 2^32 threads along x, 256 for `per_group` blocks (a 64 GiB matrix of fp32 is past that, or 8 GiB of rows of 16), and block
// numbers are 32-bit.
struct RowBlockGrid {
    uint32_t rows_per_slice, slices, groups;
};
RowBlockGrid row_block_grid(uint32_t rows, uint32_t per_row, uint32_t per_group) {
    const uint64_t most = std::min<uint64_t>((uint64_t)1 << 31, (uint64_t)per_group * ((1 << 24) - 1));        // blocks of a slice
    RowBlockGrid g;
    g.rows_per_slice = (uint32_t)std::max<uint64_t>(1, std::min<uint64_t>(rows, most / per_row));
    g.slices = (uint32_t)(((uint64_t)rows + g.rows_per_slice - 1) / g.rows_per_slice);
    g.groups = (uint32_t)(((uint64_t)g.rows_per_slice * per_row + per_group - 1) / per_group);
    return g;
}

// May a per-matrix quantisation on this stream be one launch whose workgroups wait for one another (quant_whole_matrix_kernel), and which
// of the places for such streams is its?  Two such
// launches have room on the chip side by side (two workgroups of 1024 threads and at most 64 registers a CU): kernels that wait for nobody
// then only delay them.  Three could each hold a part of it and wait for the rest until the wait ends.  So two streams may, those whose last
// such call lies fewer than 64 back; calls on others, on hipStreamPerThread and on streams that are kept to some of the CUs make two passes.
Context::QuantStream *may_exchange_maxima(hipStream_t stream) {
    if (stream == hipStreamPerThread) return nullptr;
    const uint64_t now = ++g_ctx.quant_calls;
    Context::QuantStream *oldest = &g_ctx.quant_streams[0];
    for (Context::QuantStream &q : g_ctx.quant_streams) {
        if (q.last && q.stream == stream) {
            q.last = now;
            return q.whole_chip ? &q : nullptr;
        }
        if (q.last < oldest->last) oldest = &q;
    }
    if (oldest->last && now - oldest->last < 64) return nullptr;
    uint32_t mask[64] = {}, bits = 0;
    const bool known = hipExtStreamGetCUMask(stream, 64, mask) == hipSuccess;
    if (!known) (void)hipGetLastError();
    for (uint32_t w : mask) bits += __builtin_popcount(w);
    *oldest = {stream, now, !known || bits >= (uint32_t)g_ctx.num_cus, oldest->launches};
    return oldest->whole_chip ? oldest : nullptr;
}
// How long its workgroups wait, us: what the exchange may take beside other work, and as long as reading `bytes` again takes a workgroup
// (some 100 GB/s), so that a wait in vain costs about twice what not waiting would have
uint32_t quant_wait_of(uint64_t bytes) {
    return g_ctx.quant_wait >= 0 ? (uint32_t)g_ctx.quant_wait : 20 + (uint32_t)(bytes / 100000);
}

template <int IN_DT, int OUT_DT>
int quantize_t(int mode, QuantArgs &a, hipStream_t stream) {
    typedef Piece<IN_DT> P;
    auto number = [&](uint32_t per_row) {       // see QuantArgs::per_row
        a.per_row = std::max<uint32_t>(1, per_row);
        a.inv = inverse_of(a.per_row);
        a.rows_per_slice = (uint32_t)std::max<uint64_t>(1, std::min<uint64_t>(a.rows, ((uint64_t)1 << 31) / a.per_row));
    };
    hipError_t e;
    const bool ragged = a.cols % P::VEC != 0;           // rows end inside a piece
    if (mode == QGEMM_QUANT_PER_MATRIX) {
        if (a.ld == a.cols && a.ldq == a.cols && (uint64_t)a.rows * a.cols < ((uint64_t)1 << 31)) {      // no gaps: one row
            a.cols *= a.rows;
            a.rows = a.rows ? 1 : 0;
        }
        number((a.cols + P::VEC - 1) / P::VEC);
        const uint64_t pieces = (uint64_t)a.rows * a.per_row;
        // (an empty matrix is for the forms that look whether a row has a piece: the others load without asking)
        const bool row_ends = a.cols == 0 || a.cols % P::VEC != 0, one_row = a.rows == 1;
        auto form = [&](auto one_ragged, auto one, auto rows_ragged, auto rows) { return one_row ? (row_ends ? one_ragged : one) : row_ends ? rows_ragged : rows; };
        const bool small = pieces * 16 <= (one_row ? kQuantSmallBytes : kQuantSmallRowsBytes), capturing = !small && stream_is_capturing(stream);
        if (small || (capturing && pieces * 16 <= kQuantSmallBytes)) {
            e = launch_kernel(form(quant_small_matrix_kernel<IN_DT, OUT_DT, true, true>, quant_small_matrix_kernel<IN_DT, OUT_DT, true, false>,
                                   quant_small_matrix_kernel<IN_DT, OUT_DT, false, true>, quant_small_matrix_kernel<IN_DT, OUT_DT, false, false>),
                              dim3((unsigned)std::max<uint64_t>(1, (pieces + 1023) / 1024)), dim3(1024), 0, stream, a);
            return e == hipSuccess ? QGEMM_OK : QGEMM_ERR_LAUNCH;
        }
        // two passes: partial maxima, one per workgroup, in the workspace
        const uint32_t slices = std::max<uint32_t>(1, (a.rows + a.rows_per_slice - 1) / a.rows_per_slice);
        const uint64_t turns = ((uint64_t)a.rows_per_slice * a.per_row + 256 * kQuantTurn - 1) / (256 * kQuantTurn);
        const uint32_t nblk = (uint32_t)std::max<uint64_t>(1, std::min<uint64_t>(1024, turns));
        const size_t room = (size_t)nblk * slices * sizeof(uint32_t);
        const uint64_t most = (uint64_t)std::min(g_ctx.num_cus, kQuantGroups) * 1024;        // lanes of a launch that fits the chip
        const bool whole_fits = one_row && pieces <= most * kQuantMostPieces && (uintptr_t)a.x % 4 == 0;
        Context::QuantStream *const place = g_ctx.quant_wait != -1 && whole_fits && !capturing ? may_exchange_maxima(stream) : nullptr;
        if (place) {
            const uint32_t whole = a.cols / P::VEC, each = (uint32_t)((whole + most - 1) / most);
            const uint32_t groups = std::max<uint32_t>(1, std::min<uint32_t>((uint32_t)(most / 1024), (whole + 1023) / 1024));
            a.share = (whole + groups - 1) / groups;
            // (captured, the same call makes two passes in the room that an eager one has left: one that needs none itself leaves it too)
            (void)grow_block(g_ctx.ws, room, kLeastBlock);
            if (++place->launches == 0) place->launches = 1;
            a.tag = place->launches;
            a.set = (uint32_t)(place - g_ctx.quant_streams) * (kQuantSets / 2) + a.tag % (kQuantSets / 2);
            a.wait = quant_wait_of(pieces * 16) * 100;
            e = launch_kernel(each <= 1 ? quant_whole_matrix_kernel<IN_DT, OUT_DT, 1> : each <= 2 ? quant_whole_matrix_kernel<IN_DT, OUT_DT, 2> :
                              each <= 4 ? quant_whole_matrix_kernel<IN_DT, OUT_DT, 4> : quant_whole_matrix_kernel<IN_DT, OUT_DT, kQuantMostPieces>,
                              dim3(groups), dim3(1024), 0, stream, a);
            return e == hipSuccess ? QGEMM_OK : QGEMM_ERR_LAUNCH;
        }
        a.npartial = nblk * slices;
        void *ws = nullptr;
        int st = ensure_workspace_locked(room, stream, &ws);
        if (st != QGEMM_OK) return st;
        a.partial = (uint32_t *)ws;
        e = launch_kernel(form(quant_amax_kernel<IN_DT, true, true>, quant_amax_kernel<IN_DT, true, false>,
                               quant_amax_kernel<IN_DT, false, true>, quant_amax_kernel<IN_DT, false, false>), dim3(nblk, slices), dim3(256), 0, stream, a);
        if (e != hipSuccess) return QGEMM_ERR_LAUNCH;
        const uint32_t nq = (uint32_t)std::max<uint64_t>(1, std::min<uint64_t>(2048, turns));
        e = launch_kernel(form(quant_matrix_kernel<IN_DT, OUT_DT, true, true>, quant_matrix_kernel<IN_DT, OUT_DT, true, false>,
                               quant_matrix_kernel<IN_DT, OUT_DT, false, true>, quant_matrix_kernel<IN_DT, OUT_DT, false, false>), dim3(nq, slices), dim3(256), 0, stream, a);
    } else if (mode == QGEMM_QUANT_BLOCK_1x128) {
        number((a.cols + 127) / 128);
        const RowBlockGrid g = row_block_grid(a.rows, a.per_row, 256 / P::LANES);
        a.rows_per_slice = g.rows_per_slice;
        if (g.slices > kMaxGridY) return QGEMM_ERR_TOO_LARGE;
        const dim3 grid(g.groups, g.slices);
        if ((uint64_t)g.rows_per_slice * a.per_row >= (uint64_t)kQuantManyGroups * (256 / P::LANES))
            e = launch_kernel(ragged ? quant_row_block_kernel<IN_DT, OUT_DT, true> : quant_row_block_kernel<IN_DT, OUT_DT, false>, grid, dim3(256), 0, stream, QGEMM_QUANT_HEAD_OF(a));
        else
            e = launch_kernel(ragged ? quant_few_blocks_kernel<IN_DT, OUT_DT, true> : quant_few_blocks_kernel<IN_DT, OUT_DT, false>, grid, dim3(256), 0, stream, a);
    } else {
        const uint64_t nblocks = (uint64_t)((a.rows + 127) / 128) * ((a.cols + 127) / 128);
        if (nblocks >= ((uint64_t)1 << 31)) return QGEMM_ERR_TOO_LARGE;
        if (a.rows <= kQuantFewRows)
            e = launch_kernel(ragged ? quant_low_block_kernel<IN_DT, OUT_DT, true> : quant_low_block_kernel<IN_DT, OUT_DT, false>, dim3((unsigned)nblocks), dim3(256), 0, stream, a);
        else
            e = launch_kernel(ragged ? quant_square_block_kernel<IN_DT, OUT_DT, true> : quant_square_block_kernel<IN_DT, OUT_DT, false>, dim3((unsigned)nblocks), dim3(256), 0, stream, QGEMM_QUANT_HEAD_OF(a));
    }
    return e == hipSuccess ? QGEMM_OK : QGEMM_ERR_LAUNCH;
}

}  // namespace

// ===========================================================================
extern "C" {

QGEMM_EXPORT int qgemm_device_count(void) {
    int n = 0;
    if (hipGetDeviceCount(&n) != hipSuccess) return 0;
    return n;
}

QGEMM_EXPORT int qgemm_init(void) {
    std::lock_guard<std::mutex> lock(g_ctx.mu);
    return ensure_init_locked();
}

QGEMM_EXPORT int qgemm_shutdown(void) {
    std::lock_guard<std::mutex> lock(g_ctx.mu);
    for (const WsBlock &b : g_ctx.ws_own)
        if (b.p) g_ctx.retired.push_back(b.p);
    if (g_ctx.ws.p) g_ctx.retired.push_back(g_ctx.ws.p);
    if (!g_ctx.retired.empty()) (void)hipDeviceSynchronize();
    for (void *p : g_ctx.retired) (void)hipFree(p);
    if (g_ctx.ws_event) (void)hipEventDestroy(g_ctx.ws_event);
    g_ctx.ws = WsBlock();
    for (WsBlock &b : g_ctx.ws_own) b = WsBlock();
    g_ctx.ws_owners = 0;
    g_ctx.ws_own_failed = false;
    g_ctx.retired.clear();
    g_ctx.ws_event = nullptr;
    g_ctx.ws_event_recorded = false;
    g_ctx.ready = false;
    return QGEMM_OK;
}

QGEMM_EXPORT const char *qgemm_status_string(int status) {
    switch (status) {
        case QGEMM_OK: return "ok";
        case QGEMM_ERR_INVALID_ARG: return "invalid argument";
        case QGEMM_ERR_UNSUPPORTED: return "unsupported dtype / layout combination";
        case QGEMM_ERR_NO_DEVICE: return "no HIP device";
        case QGEMM_ERR_LAUNCH: return "HIP call failed";
        case QGEMM_ERR_ALLOC: return "workspace allocation failed";
        case QGEMM_ERR_NOT_DIVISIBLE_M: return "M is not divisible by any predefined BLOCK_TILE_SIZE_M in the list";
        case QGEMM_ERR_NOT_DIVISIBLE_N: return "N is not divisible by any predefined BLOCK_TILE_SIZE_N in the list";
        case QGEMM_ERR_NOT_DIVISIBLE_K: return "K is not divisible by any predefined BLOCK_TILE_SIZE_K in the list";
        case QGEMM_ERR_TOO_LARGE: return "dimension or stride too large";
        case QGEMM_ERR_SCRATCH_TOO_SMALL: return "problem needs more than the static scratch (QGEMM_STATIC_SCRATCH_BYTES)";
    }
    return "unknown status";
}

QGEMM_EXPORT int qgemm_tile_map(uint32_t wg, uint32_t tiles_m, uint32_t tiles_n, uint32_t group_m, uint32_t *tile_m,
                   uint32_t *tile_n) {
    if (!tile_m || !tile_n || tiles_m == 0 || tiles_n == 0) return QGEMM_ERR_INVALID_ARG;
    if ((uint64_t)wg >= (uint64_t)tiles_m * tiles_n) return QGEMM_ERR_INVALID_ARG;
    tile_map(wg, make_tile_map(tiles_m, tiles_n, group_m), *tile_m, *tile_n);
    return QGEMM_OK;
}

QGEMM_EXPORT int qgemm_quantize_grid(int in_dtype, size_t rows, size_t cols, uint32_t *rows_per_slice, uint32_t *slices, uint32_t *groups) {
    if (in_dtype != QGEMM_DT_F32 && in_dtype != QGEMM_DT_BF16 && in_dtype != QGEMM_DT_F16) return QGEMM_ERR_UNSUPPORTED;
    if (!rows_per_slice || !slices || !groups || rows == 0 || cols == 0) return QGEMM_ERR_INVALID_ARG;
    if (rows >= ((size_t)1 << 31) || cols >= ((size_t)1 << 31)) return QGEMM_ERR_TOO_LARGE;
    const RowBlockGrid g = row_block_grid((uint32_t)rows, (uint32_t)((cols + 127) / 128), 256 / (in_dtype == QGEMM_DT_F32 ? Piece<QGEMM_DT_F32>::LANES : Piece<QGEMM_DT_BF16>::LANES));
    *rows_per_slice = g.rows_per_slice;
    *slices = g.slices;
    *groups = g.groups;
    return g.slices > kMaxGridY ? QGEMM_ERR_TOO_LARGE : QGEMM_OK;
}

QGEMM_EXPORT int qgemm_set_option(const char *key, long value) {
    if (!key) return QGEMM_ERR_INVALID_ARG;
    std::lock_guard<std::mutex> lock(g_ctx.mu);
    if (!std::strcmp(key, "force_config")) {
        if (value != -1) return QGEMM_ERR_INVALID_ARG;      // rows are named: qgemm_force_config; -1 returns to the heuristic
        g_ctx.force_config.clear();
    } else if (!std::strcmp(key, "force_split")) g_ctx.force_split = value;
    else if (!std::strcmp(key, "group_m")) g_ctx.force_group_m = value;
    else if (!std::strcmp(key, "kmajor")) g_ctx.kmajor = value;
    else if (!std::strcmp(key, "any_shape")) g_ctx.any_shape = value;
    else if (!std::strcmp(key, "stagger")) g_ctx.stagger = value;
    else if (!std::strcmp(key, "stagger_groups")) g_ctx.stagger_groups = value;
    else if (!std::strcmp(key, "c_plain")) g_ctx.c_plain = value;
    else if (!std::strcmp(key, "b_stream")) g_ctx.b_stream = value;
    else if (!std::strcmp(key, "k_rot")) g_ctx.k_rot = value;
    else if (!std::strcmp(key, "as_groups")) g_ctx.as_groups = value;
    else if (!std::strcmp(key, "small_tiles")) g_ctx.small_tiles = value;
    else if (!std::strcmp(key, "few_rows")) g_ctx.few_rows = value;
    else if (!std::strcmp(key, "quant_wait")) g_ctx.quant_wait = std::max(-2L, std::min(value, 1000000L));
    else if (!std::strcmp(key, "row_estimate")) g_ctx.row_estimate = value;
#if QGEMM_DEBUG_BUILD
    else if (!std::strcmp(key, "dbg_ptr")) g_ctx.dbg_ptr = value;
#endif
    else if (!std::strcmp(key, "row_split")) g_ctx.row_split = value;
    else return QGEMM_ERR_INVALID_ARG;
    return QGEMM_OK;
}

QGEMM_EXPORT int qgemm_force_config(const char *name) {
    std::lock_guard<std::mutex> lock(g_ctx.mu);
    if (!name || !*name) {
        g_ctx.force_config.clear();
        return QGEMM_OK;
    }
    // the name has to be a row of at least one family
    bool known = false;
    for (int arith = 0; arith < 4 && !known; ++arith)
        for (int block = 0; block < 2 && !known; ++block)
            for (int kmaj = 0; kmaj < 4 && !known; ++kmaj) {
                int count = 0;
                const Variant *tab = table_for(arith, block != 0, kmaj, &count);
                known = row_by_name(tab, count, name) >= 0;
            }
    if (!known) return QGEMM_ERR_INVALID_ARG;
    g_ctx.force_config = name;
    return QGEMM_OK;
}

QGEMM_EXPORT int qgemm_variant_count(int in_dtype, int scale_mode, int k_major) {
    int count = 0;
    const int arith = arith_of(in_dtype);
    if (arith < 0 || !table_for(arith, scale_mode == QGEMM_SCALE_BLOCK128, k_major, &count)) return 0;
    return count;
}

QGEMM_EXPORT int qgemm_variant_name(int in_dtype, int scale_mode, int k_major, int index, char *buf, size_t buflen) {
    if (!buf || buflen == 0) return QGEMM_ERR_INVALID_ARG;
    int count = 0;
    const int arith = arith_of(in_dtype);
    const Variant *tab = arith < 0 ? nullptr : table_for(arith, scale_mode == QGEMM_SCALE_BLOCK128, k_major, &count);
    if (!tab) return QGEMM_ERR_UNSUPPORTED;
    if (index < 0 || index >= count) return QGEMM_ERR_INVALID_ARG;
    std::snprintf(buf, buflen, "%s", tab[index].name);
    return QGEMM_OK;
}

QGEMM_EXPORT int qgemm_last_config(char *buf, size_t buflen) {
    if (!buf || buflen == 0) return QGEMM_ERR_INVALID_ARG;
    std::lock_guard<std::mutex> lock(g_ctx.mu);
    std::snprintf(buf, buflen, "%s", g_ctx.last_config.c_str());
    return QGEMM_OK;
}

QGEMM_EXPORT int qgemm_last_any_kernel(char *buf, size_t buflen) {
    if (!buf || buflen == 0) return QGEMM_ERR_INVALID_ARG;
    std::lock_guard<std::mutex> lock(g_ctx.mu);
    std::snprintf(buf, buflen, "%s", g_ctx.last_any_kernel);
    return QGEMM_OK;
}

QGEMM_EXPORT int qgemm_plan(int in_dtype, int scale_mode, int k_major, size_t M, size_t N, size_t K, char *buf,
                            size_t buflen) {
    return qgemm_plan_out(in_dtype, QGEMM_DT_BF16, scale_mode, k_major, M, N, K, buf, buflen);
}

QGEMM_EXPORT int qgemm_plan_out(int in_dtype, int out_dtype, int scale_mode, int k_major, size_t M, size_t N, size_t K, char *buf,
                                size_t buflen) {
    if (!buf || buflen == 0 || M == 0 || N == 0 || K == 0 || k_major < 0 || k_major > 3) return QGEMM_ERR_INVALID_ARG;
    const int arith = arith_of(in_dtype);
    if (arith < 0) return QGEMM_ERR_UNSUPPORTED;
    if (scale_mode != 0 && scale_mode != QGEMM_SCALE_PER_MATRIX && scale_mode != QGEMM_SCALE_BLOCK128)
        return QGEMM_ERR_INVALID_ARG;
    if (scale_mode == QGEMM_SCALE_BLOCK128 && arith != AR_F8 && arith != AR_I8) return QGEMM_ERR_UNSUPPORTED;
    if (!out_dtype_ok(in_dtype, out_dtype) || (scale_mode == QGEMM_SCALE_BLOCK128 && out_dtype == QGEMM_DT_I32)) return QGEMM_ERR_UNSUPPORTED;
    std::lock_guard<std::mutex> lock(g_ctx.mu);          // no device call below: 256 CUs are assumed before qgemm_init
    const size_t eb = (arith == AR_BF16 || arith == AR_F16) ? 2 : 1;
    NtProblem q = NtProblem();
    q.arith = arith;
    q.block = scale_mode == QGEMM_SCALE_BLOCK128;
    q.M = M;
    q.N = N;
    q.Kbytes = K * eb;
    q.lda_bytes = q.ldb_bytes = K * eb;
    q.ldc = N;
    q.out_dtype = out_dtype;
    std::string name;
    if (k_major) {
        const size_t lda = (k_major & 1) ? M * eb : K * eb, ldb = (k_major & 2) ? N * eb : K * eb;
        int rows = 0;
        const bool family = table_for(arith, q.block, k_major, &rows) != nullptr;
        if (family && kmajor_problem_ok(q, k_major, lda, ldb)) {
            q.kmaj = k_major;
            q.lda_bytes = lda;
            q.ldb_bytes = ldb;
        } else {
            name = "transpose+";
        }
    }
    if (!mfma_shape_ok(q)) {
        std::snprintf(buf, buflen, "strided_any_shape");
        return QGEMM_OK;
    }
    Plan pl;
    const int st = plan_nt(q, pl);
    if (st != QGEMM_OK) return st;
    if (q.block) {          // dense scales in the arrangement of the layout asked about
        const uint32_t KB = (uint32_t)((K + 127) / 128);
        if (k_major == 3) { q.as_ms = 1; q.as_ks = (uint32_t)M; }
        else { q.as_ms = KB; q.as_ks = 1; }
        (void)settle_scale_layout(q, pl);
    }
    name += std::string(pl.v->name) + kmaj_suffix(q.kmaj);
    if (pl.a.nsplit > 1) name += "_splitk" + std::to_string(pl.a.nsplit);
    if (pl.rest) {
        name += (pl.m_main ? "+" : "|") + std::string(pl.rest->v->name);
        if (pl.rest->a.nsplit > 1) name += "_splitk" + std::to_string(pl.rest->a.nsplit);
    }
    std::snprintf(buf, buflen, "%s", name.c_str());
    return QGEMM_OK;
}

QGEMM_EXPORT int qgemm_quantize(int in_dtype, int out_dtype, int mode, const void *x, size_t ld, size_t rows, size_t cols,
                                void *q, size_t ldq, float *scales, size_t scale_rs, size_t scale_cs, void *stream_) {
    if (in_dtype != QGEMM_DT_F32 && in_dtype != QGEMM_DT_BF16 && in_dtype != QGEMM_DT_F16) return QGEMM_ERR_UNSUPPORTED;
    if (out_dtype != QGEMM_DT_I8 && out_dtype != QGEMM_DT_F8E4M3) return QGEMM_ERR_UNSUPPORTED;
    if (mode != QGEMM_QUANT_PER_MATRIX && mode != QGEMM_QUANT_BLOCK_1x128 && mode != QGEMM_QUANT_BLOCK_128x128)
        return QGEMM_ERR_INVALID_ARG;
    if (!scales) return QGEMM_ERR_INVALID_ARG;
    if (rows >= ((size_t)1 << 31) || cols >= ((size_t)1 << 31)) return QGEMM_ERR_TOO_LARGE;
    std::lock_guard<std::mutex> lock(g_ctx.mu);
    int st = ensure_init_locked();
    if (st != QGEMM_OK) return st;
    hipStream_t stream = (hipStream_t)stream_;
    WorkspaceUse ws_use(stream);
    QuantArgs a;
    std::memset(&a, 0, sizeof(a));
    a.x = x;
    a.q = q;
    a.scales = scales;
    a.rows = (uint32_t)rows;
    a.cols = (uint32_t)cols;
    a.ld = ld;
    a.ldq = ldq;
    a.scale_rs = scale_rs;
    a.scale_cs = scale_cs;
    if (rows == 0 || cols == 0) {
        if (mode != QGEMM_QUANT_PER_MATRIX) return QGEMM_OK;
        // the scale of an empty matrix is the scale of a zero matrix: run the passes over nothing
        a.rows = a.cols = 0;
    } else if (!x || !q || ld < cols || ldq < cols) {
        return QGEMM_ERR_INVALID_ARG;
    }
    g_ctx.last_config = mode == QGEMM_QUANT_PER_MATRIX ? "quantize_per_matrix"
                        : (mode == QGEMM_QUANT_BLOCK_1x128 ? "quantize_1x128" : "quantize_128x128");
    const bool f8 = out_dtype == QGEMM_DT_F8E4M3;
    switch (in_dtype) {
        case QGEMM_DT_F32:
            return f8 ? quantize_t<QGEMM_DT_F32, QGEMM_DT_F8E4M3>(mode, a, stream) : quantize_t<QGEMM_DT_F32, QGEMM_DT_I8>(mode, a, stream);
        case QGEMM_DT_BF16:
            return f8 ? quantize_t<QGEMM_DT_BF16, QGEMM_DT_F8E4M3>(mode, a, stream) : quantize_t<QGEMM_DT_BF16, QGEMM_DT_I8>(mode, a, stream);
        default:
            return f8 ? quantize_t<QGEMM_DT_F16, QGEMM_DT_F8E4M3>(mode, a, stream) : quantize_t<QGEMM_DT_F16, QGEMM_DT_I8>(mode, a, stream);
    }
}

QGEMM_EXPORT int qgemm_transpose(int elem_bytes, const void *in, void *out, size_t M, size_t N, void *stream) {
    if (elem_bytes != 1 && elem_bytes != 2 && elem_bytes != 4) return QGEMM_ERR_UNSUPPORTED;
    if (M == 0 || N == 0) return QGEMM_OK;
    if (!in || !out) return QGEMM_ERR_INVALID_ARG;
    if (M >= ((size_t)1 << 31) || N >= ((size_t)1 << 31)) return QGEMM_ERR_TOO_LARGE;
    std::lock_guard<std::mutex> lock(g_ctx.mu);
    int st = ensure_init_locked();
    if (st != QGEMM_OK) return st;
    return launch_transpose(elem_bytes, in, out, M, N, (hipStream_t)stream);
}

QGEMM_EXPORT int qgemm_gemm(int in_dtype, int out_dtype, int layout_b, const void *A, size_t ldA, const void *B, size_t ldB,
               void *C, size_t ldC, size_t M, size_t N, size_t K, void *stream_) {
    const int arith = arith_of(in_dtype);
    if (arith < 0 || !out_dtype_ok(in_dtype, out_dtype)) return QGEMM_ERR_UNSUPPORTED;
    if (layout_b != QGEMM_B_KN && layout_b != QGEMM_B_NK) return QGEMM_ERR_INVALID_ARG;
    if (M == 0 || N == 0) return QGEMM_OK;
    if (!A || !B || !C || K == 0) return QGEMM_ERR_INVALID_ARG;
    if (ldA < K || ldC < N || ldB < (layout_b == QGEMM_B_KN ? N : K)) return QGEMM_ERR_INVALID_ARG;
    hipStream_t stream = (hipStream_t)stream_;
    std::lock_guard<std::mutex> lock(g_ctx.mu);
    int st = ensure_init_locked();
    if (st != QGEMM_OK) return st;
    WorkspaceUse ws_use(stream);

    const size_t eb = dtype_bytes(in_dtype);
    NtProblem q = NtProblem();
    q.arith = arith;
    q.block = false;
    q.A = A;
    q.C = C;
    q.lda_bytes = ldA * eb;
    q.ldc = ldC;
    q.M = M;
    q.N = N;
    q.Kbytes = K * eb;
    q.out_dtype = out_dtype;
    q.per_matrix = 0;
    q.split_k = 0;

    if (layout_b == QGEMM_B_NK) {
        q.B = B;
        q.ldb_bytes = ldB * eb;
        if (mfma_shape_ok(q) && aligned16(A) && aligned16(B)) return launch_nt(q, stream);
    } else if (eb == 2 && aligned16(A) && aligned16(B) && kmajor_problem_ok(q, 2, q.lda_bytes, ldB * eb)) {
        // "NN", 16-bit operands: the kernel takes B as it is stored (K x N), see GemmCfg::KMAJ
        q.kmaj = 2;
        q.B = B;
        q.ldb_bytes = ldB * eb;
        return launch_nt(q, stream);
    } else if (ldB == N) {
        // "NN" otherwise: bring B to N x K through the transpose utility (the route the reference's
        // v3.1 launcher sketches, sm80_gemm_kernel_v3.1.cu:277-279), then run the NT kernel.
        q.ldb_bytes = K * eb;
        if (mfma_shape_ok(q) && aligned16(A)) {
            Plan pl;
            st = plan_nt(q, pl);
            if (st != QGEMM_OK) return st;
            const size_t split_room = (pl.split_bytes + 255) / 256 * 256;
            void *ws = nullptr;
            st = ensure_workspace_locked(split_room + N * K * eb, stream, &ws);
            if (st != QGEMM_OK) return st;
            void *bt = (char *)ws + split_room;
            st = launch_transpose((int)eb, B, bt, K, N, stream);
            if (st != QGEMM_OK) return st;
            q.B = bt;
            return run_nt(q, pl, ws, stream);
        }
    }

    if (M >= ((size_t)1 << 32) || N >= ((size_t)1 << 32) || K >= ((size_t)1 << 32)) return QGEMM_ERR_TOO_LARGE;
    const SourceOperand a_src{A, ldA * eb, false}, b_src{B, ldB * eb, layout_b == QGEMM_B_KN};
    bool taken = false;
    st = launch_unaligned(q, in_dtype, a_src, b_src, K, stream, &taken);
    if (taken || st != QGEMM_OK) return st;
    st = launch_packed(q, in_dtype, a_src, b_src, K, stream, &taken);
    return taken ? st : launch_any(q, in_dtype, a_src, b_src, K, stream);
}

}  // extern "C"

namespace {

// Body of qgemm_scaled_gemm and qgemm_scaled_gemm_static; `use_static`: the workspace is the static scratch.
int scaled_gemm_entry(bool use_static, int in_dtype, int out_dtype, int scale_mode, int layout, const void *A, const void *B,
                      const float *a_scale, const float *b_scale, void *C, size_t ldC, size_t M, size_t N, size_t K,
                      int split_k, void *stream_) {
    if (in_dtype != QGEMM_DT_I8 && in_dtype != QGEMM_DT_F8E4M3) return QGEMM_ERR_UNSUPPORTED;
    if (!out_dtype_ok(in_dtype, out_dtype)) return QGEMM_ERR_UNSUPPORTED;
    if (scale_mode != QGEMM_SCALE_PER_MATRIX && scale_mode != QGEMM_SCALE_BLOCK128) return QGEMM_ERR_INVALID_ARG;
    // (int8 with block scales and int32 output: there is no int32 sum of scaled blocks)
    if (scale_mode == QGEMM_SCALE_BLOCK128 && out_dtype == QGEMM_DT_I32) return QGEMM_ERR_UNSUPPORTED;
    if (layout != QGEMM_LAYOUT_K_CONTIGUOUS && layout != QGEMM_LAYOUT_REFERENCE) return QGEMM_ERR_INVALID_ARG;
    if (split_k < 0) return QGEMM_ERR_INVALID_ARG;
    if (layout == QGEMM_LAYOUT_REFERENCE) {
        // dispatch contract of select_BLOCK_TILE_SIZE_{M,N,K}: hip_mix_gemm_kernel.cpp:442-505
        if (M % 32 != 0) return QGEMM_ERR_NOT_DIVISIBLE_M;
        if (N % 32 != 0) return QGEMM_ERR_NOT_DIVISIBLE_N;
        if (K % 32 != 0) return QGEMM_ERR_NOT_DIVISIBLE_K;
    }
    if (M == 0 || N == 0) return QGEMM_OK;
    if (!A || !B || !C || K == 0 || ldC < N) return QGEMM_ERR_INVALID_ARG;
    const bool raw_acc = out_dtype == QGEMM_DT_I32;
    if (!raw_acc && (!a_scale || !b_scale)) return QGEMM_ERR_INVALID_ARG;
    hipStream_t stream = (hipStream_t)stream_;
    std::lock_guard<std::mutex> lock(g_ctx.mu);
    int st = ensure_init_locked();
    if (st != QGEMM_OK) return st;
    struct StaticScope {        // every workspace request of this call goes to the static scratch
        explicit StaticScope(bool on) { g_ctx.static_call = on; }
        ~StaticScope() { g_ctx.static_call = false; }
    } scope(use_static);
    WorkspaceUse ws_use(stream);

    const bool block = scale_mode == QGEMM_SCALE_BLOCK128;
    const uint32_t KB = (uint32_t)((K + 127) / 128), NBLK = (uint32_t)((N + 127) / 128);
    NtProblem q = NtProblem();
    q.arith = arith_of(in_dtype);
    q.block = block;
    q.C = C;
    q.ldc = ldC;
    q.M = M;
    q.N = N;
    q.Kbytes = K;
    q.lda_bytes = K;
    q.ldb_bytes = K;
    q.as = a_scale;
    q.bs = b_scale;
    q.out_dtype = out_dtype;
    q.per_matrix = (!block && !raw_acc) ? 1 : 0;
    q.split_k = split_k;
    if (block) {
        if (layout == QGEMM_LAYOUT_K_CONTIGUOUS) {
            q.as_ms = KB; q.as_ks = 1; q.bs_ns = KB; q.bs_ks = 1;
        } else {   // a_scale[m + kb*M], b_scale[nb + kb*ceil(N/128)]: hip_mix_gemm_kernel.cpp:137,149,164
            q.as_ms = 1; q.as_ks = (uint32_t)M; q.bs_ns = 1; q.bs_ks = NBLK;
        }
    }

    if (layout == QGEMM_LAYOUT_K_CONTIGUOUS) {
        q.A = A;
        q.B = B;
        if (mfma_shape_ok(q) && aligned16(A) && aligned16(B)) return launch_nt(q, stream);
    } else if (block && aligned16(A) && aligned16(B) && kmajor_problem_ok(q, 3, M, N)) {
        // reference layout, block scales: A is K x M (M contiguous), B is K x N; the kernel reads both as stored
        q.kmaj = 3;
        q.A = A;
        q.B = B;
        q.lda_bytes = M;
        q.ldb_bytes = N;
        return launch_nt(q, stream);
    } else if (mfma_shape_ok(q)) {
        // reference layout otherwise: bring both to K-contiguous through the transpose utility, then run
        // the NT kernel.
        Plan pl;
        st = plan_nt(q, pl);
        if (st != QGEMM_OK) return st;
        const size_t split_room = (pl.split_bytes + 255) / 256 * 256;
        const size_t at_bytes = (M * K + 255) / 256 * 256;
        void *ws = nullptr;
        st = ensure_workspace_locked(split_room + at_bytes + N * K, stream, &ws);
        if (st != QGEMM_OK) return st;
        char *at = (char *)ws + split_room, *bt = at + at_bytes;
        // M, N, K are multiples of 32 here: both matrices qualify for the register-permute byte transpose
        if (aligned16(A) && aligned16(B) && K < ((size_t)1 << 31)) {
            Transpose2Args t;
            t.in[0] = (const uint8_t *)A; t.out[0] = (uint8_t *)at; t.M[0] = (uint32_t)K; t.N[0] = (uint32_t)M;
            t.in[1] = (const uint8_t *)B; t.out[1] = (uint8_t *)bt; t.M[1] = (uint32_t)K; t.N[1] = (uint32_t)N;
            const size_t tk = (K + 127) / 128;
            t.tiles_n[0] = (uint32_t)((M + 127) / 128);
            t.tiles_n[1] = (uint32_t)((N + 127) / 128);
            t.tiles0 = (uint32_t)(tk * t.tiles_n[0]);
            const size_t total = tk * ((size_t)t.tiles_n[0] + t.tiles_n[1]);
            if (total >= ((size_t)1 << 31)) return QGEMM_ERR_TOO_LARGE;
            HIP_TRY(launch_kernel(transpose_bytes2_kernel, dim3((unsigned)total), dim3(256), 0, stream, t));
        } else {
            st = launch_transpose(1, A, at, K, M, stream);
            if (st != QGEMM_OK) return st;
            st = launch_transpose(1, B, bt, K, N, stream);
            if (st != QGEMM_OK) return st;
        }
        q.A = at;
        q.B = bt;
        (void)settle_scale_layout(q, pl);            // (scales are rows-contiguous in this layout)
        return run_nt(q, pl, ws, stream);
    }

    if (M >= ((size_t)1 << 32) || N >= ((size_t)1 << 32) || K >= ((size_t)1 << 32)) return QGEMM_ERR_TOO_LARGE;
    const bool km = layout == QGEMM_LAYOUT_REFERENCE;
    const SourceOperand a_src{A, km ? M : K, km}, b_src{B, km ? N : K, km};
    bool taken = false;
    st = launch_unaligned(q, in_dtype, a_src, b_src, K, stream, &taken);
    if (taken || st != QGEMM_OK) return st;
    st = launch_packed(q, in_dtype, a_src, b_src, K, stream, &taken);
    return taken ? st : launch_any(q, in_dtype, a_src, b_src, K, stream);
}

}  // namespace

extern "C" {

QGEMM_EXPORT int qgemm_scaled_gemm(int in_dtype, int out_dtype, int scale_mode, int layout, const void *A, const void *B,
                      const float *a_scale, const float *b_scale, void *C, size_t ldC, size_t M, size_t N, size_t K,
                      int split_k, void *stream) {
    return scaled_gemm_entry(false, in_dtype, out_dtype, scale_mode, layout, A, B, a_scale, b_scale, C, ldC, M, N, K, split_k,
                             stream);
}

QGEMM_EXPORT int qgemm_scaled_gemm_static(int in_dtype, int out_dtype, int scale_mode, int layout, const void *A,
                                          const void *B, const float *a_scale, const float *b_scale, void *C, size_t ldC,
                                          size_t M, size_t N, size_t K, int split_k, void *stream) {
    return scaled_gemm_entry(true, in_dtype, out_dtype, scale_mode, layout, A, B, a_scale, b_scale, C, ldC, M, N, K, split_k,
                             stream);
}

QGEMM_EXPORT int qgemm_reserve_workspace(size_t bytes) {
    std::lock_guard<std::mutex> lock(g_ctx.mu);
    int st = ensure_init_locked();
    if (st != QGEMM_OK) return st;
    // (takes no stream, so it cannot tell whether one is being captured: the caller reserves before a capture)
    if (grow_block(g_ctx.ws, bytes, 0) != QGEMM_OK) return QGEMM_ERR_ALLOC;
    // calls that need no more than this allocate nothing from here on, on any stream
    for (WsBlock &b : g_ctx.ws_own) (void)make_own_block(b, std::min(bytes, kOwnBytes));
    return QGEMM_OK;
}

QGEMM_EXPORT int qgemm_workspace_info(void **base, size_t *bytes) {
    if (!base || !bytes) return QGEMM_ERR_INVALID_ARG;
    std::lock_guard<std::mutex> lock(g_ctx.mu);
    *base = g_ctx.ws.p;
    *bytes = g_ctx.ws.bytes;
    return QGEMM_OK;
}

// ---------------------------------------------------------------------------
// self test
// ---------------------------------------------------------------------------
namespace {

float host_decode(int arith, const uint8_t *p, int idx) {
    if (arith == AR_I8) return (float)((const int8_t *)p)[idx];
    if (arith == AR_F8) {
        const uint8_t b = p[idx];
        const int e = (b >> 3) & 15, m = b & 7;
        float mag = e == 0 ? (float)m / 512.0f : (1.0f + (float)m / 8.0f) * std::exp2((float)(e - 7));
        return (b & 0x80) ? -mag : mag;
    }
    uint16_t h;
    std::memcpy(&h, p + 2 * idx, 2);
    if (arith == AR_BF16) {
        uint32_t u = (uint32_t)h << 16;
        float f;
        std::memcpy(&f, &u, 4);
        return f;
    }
    // fp16: the probe only uses small integers, exactly representable
    const int e = (h >> 10) & 31, m = h & 1023;
    float mag = e == 0 ? (float)m / 16777216.0f : (1.0f + (float)m / 1024.0f) * std::exp2((float)(e - 15));
    return (h & 0x8000) ? -mag : mag;
}

// value v in [-4, 4] encoded in the family's element type
void host_encode_small(int arith, int v, uint8_t *p, int idx) {
    if (arith == AR_I8) { ((int8_t *)p)[idx] = (int8_t)v; return; }
    if (arith == AR_F8) {
        static const uint8_t code[5] = {0x00, 0x38, 0x40, 0x44, 0x48};   // 0, 1, 2, 3, 4
        p[idx] = (uint8_t)(code[v < 0 ? -v : v] | (v < 0 ? 0x80 : 0));
        return;
    }
    uint16_t h;
    if (arith == AR_BF16) {
        static const uint16_t code[5] = {0x0000, 0x3F80, 0x4000, 0x4040, 0x4080};
        h = (uint16_t)(code[v < 0 ? -v : v] | (v < 0 ? 0x8000 : 0));
    } else {
        static const uint16_t code[5] = {0x0000, 0x3C00, 0x4000, 0x4200, 0x4400};
        h = (uint16_t)(code[v < 0 ? -v : v] | (v < 0 ? 0x8000 : 0));
    }
    std::memcpy(p + 2 * idx, &h, 2);
}

}  // namespace

QGEMM_EXPORT int qgemm_selftest_layouts(char *buf, size_t buflen) {
    std::lock_guard<std::mutex> lock(g_ctx.mu);
    int st = ensure_init_locked();
    if (st != QGEMM_OK) return st;
    std::string rep;
    bool all_ok = true;
    char line[256];

    // ---- LDS DMA: lane l's 16 bytes land at lds_base + 16*l, for low and high LDS addresses;
    //      out-of-range lanes write zeros
    {
        const int nsrc = 4096;
        std::vector<uint8_t> hsrc(nsrc);
        for (int i = 0; i < nsrc; ++i) hsrc[i] = (uint8_t)((i * 7 + (i >> 8)) & 0xFF);
        std::vector<uint32_t> hoff(64);
        for (int l = 0; l < 64; ++l) hoff[l] = (uint32_t)(((63 - l) * 48) % 2048);   // a permutation-ish gather, 16-aligned
        hoff[5] = 4096 + 64;   // out of range
        hoff[40] = 0xFFFFFF00u;
        hoff[7] = 3488;        // in range alone, out of range once soffset = 1024 is added
        void *dsrc = nullptr, *doff = nullptr, *dout = nullptr;
        HIP_TRY(hipMalloc(&dsrc, nsrc + 4096));   // slack behind the 4096-byte buffer range the probe declares
        HIP_TRY(hipMalloc(&doff, 256));
        HIP_TRY(hipMalloc(&dout, 1024));
        HIP_TRY(hipMemcpy(dsrc, hsrc.data(), nsrc, hipMemcpyHostToDevice));
        HIP_TRY(hipMemcpy(doff, hoff.data(), 256, hipMemcpyHostToDevice));
        HIP_TRY(hipFuncSetAttribute((const void *)probe_lds_dma_kernel, hipFuncAttributeMaxDynamicSharedMemorySize,
                                    160 * 1024));
        const uint32_t bases[3] = {0, 72 * 1024, 159 * 1024};
        const uint32_t soffs[3] = {0, 1024, 16};
        for (int t = 0; t < 3; ++t) {
            HIP_TRY(launch_kernel(probe_lds_dma_kernel, dim3(1), dim3(64), 160 * 1024, nullptr, (const char *)dsrc,
                                  (const uint32_t *)doff, (uint32_t)nsrc, bases[t], soffs[t], (char *)dout));
            std::vector<uint8_t> hout(1024);
            HIP_TRY(hipMemcpy(hout.data(), dout, 1024, hipMemcpyDeviceToHost));
            int bad = 0, oob_zero = 0, oob_untouched = 0;
            for (int l = 0; l < 64; ++l) {
                const uint64_t off = (uint64_t)hoff[l] + soffs[t];
                if (l == 7 && off + 16 > (uint64_t)nsrc) {
                    bool z = true;
                    for (int j = 0; j < 16; ++j) z &= hout[l * 16 + j] == 0;
                    std::snprintf(line, sizeof(line), "lds_dma: soffset %s part of the buffer range check\n",
                                  z ? "IS" : "is NOT");
                    rep += line;
                    // tile rows past M or N are kept out of reach by the range check alone (the row block of a
                    // copy sits in the scalar offset in the simple pipeline)
                    if (!z) all_ok = false;
                    continue;
                }
                if (off + 16 > (uint64_t)nsrc) {
                    bool z = true, u = true;
                    for (int j = 0; j < 16; ++j) {
                        z &= hout[l * 16 + j] == 0;
                        u &= hout[l * 16 + j] == 0xA5;
                    }
                    oob_zero += z;
                    oob_untouched += u;
                    continue;
                }
                for (int j = 0; j < 16; ++j) bad += hout[l * 16 + j] != hsrc[off + j];
            }
            std::snprintf(line, sizeof(line), "lds_dma base=%u soffset=%u: mismatched_bytes=%d oob_lanes_zero=%d oob_lanes_untouched=%d\n",
                          bases[t], soffs[t], bad, oob_zero, oob_untouched);
            rep += line;
            if (bad) all_ok = false;
        }
        // 16-byte copies at 4-byte aligned offsets, the last ones across the end of the range: a_scale travels that way,
        // four K blocks of a row per lane, whatever the number of K blocks in a row
        for (int l = 0; l < 64; ++l) hoff[l] = (uint32_t)(l < 56 ? 4 * (7 * l % 1000) : nsrc - 4 * (l - 55));
        HIP_TRY(hipMemcpy(doff, hoff.data(), 256, hipMemcpyHostToDevice));
        HIP_TRY(launch_kernel(probe_lds_dma_kernel, dim3(1), dim3(64), 160 * 1024, nullptr, (const char *)dsrc, (const uint32_t *)doff,
                              (uint32_t)nsrc, 0u, 0u, (char *)dout));
        std::vector<uint8_t> hout(1024);
        HIP_TRY(hipMemcpy(hout.data(), dout, 1024, hipMemcpyDeviceToHost));
        int bad = 0;
        for (int l = 0; l < 64; ++l)
            for (int j = 0; j < 16; ++j) {
                const uint32_t off = hoff[l] + j;
                bad += hout[l * 16 + j] != (off < (uint32_t)nsrc ? hsrc[off] : 0);
            }
        std::snprintf(line, sizeof(line), "lds_dma at 4-byte alignment and across the end of the range: mismatched_bytes=%d\n", bad);
        rep += line;
        if (bad) all_ok = false;
        (void)hipFree(dsrc);
        (void)hipFree(doff);
        (void)hipFree(dout);
    }

    // ---- 8-byte buffer loads at 4-byte aligned offsets, and across the end of the buffer range: the twin kernels
    //      for K-contiguous a_scale (two K blocks per load) read rows with an odd number of K blocks that way
    {
        const int n_in = 60;                                 // floats inside the range; 64 are allocated
        std::vector<float> h(64);
        for (int i = 0; i < 64; ++i) h[i] = 100.0f + (float)i;
        void *d = nullptr, *o = nullptr;
        HIP_TRY(hipMalloc(&d, 64 * 4));
        HIP_TRY(hipMalloc(&o, 128 * 4));
        HIP_TRY(hipMemcpy(d, h.data(), 64 * 4, hipMemcpyHostToDevice));
        HIP_TRY(launch_kernel(probe_b64_load_kernel, dim3(1), dim3(64), 0, nullptr, (const float *)d, (uint32_t)(n_in * 4), (int *)o));
        std::vector<float> got(128);
        HIP_TRY(hipMemcpy(got.data(), o, 128 * 4, hipMemcpyDeviceToHost));
        int bad = 0;
        for (int l = 0; l + 1 < n_in; ++l) bad += got[2 * l] != h[l] || got[2 * l + 1] != h[l + 1];
        const bool per_dword = got[2 * (n_in - 1)] == h[n_in - 1] && got[2 * (n_in - 1) + 1] == 0.0f;
        bool beyond_zero = true;
        for (int l = n_in; l < 64; ++l) beyond_zero &= got[2 * l] == 0.0f && got[2 * l + 1] == 0.0f;
        std::snprintf(line, sizeof(line), "b64 buffer load: mismatched_pairs=%d (odd lanes are 4-byte aligned only), range check %s, past_range_zero=%d\n",
                      bad, per_dword ? "per dword" : "NOT per dword", (int)beyond_zero);
        rep += line;
        if (bad || !per_dword || !beyond_zero) all_ok = false;
        (void)hipFree(d);
        (void)hipFree(o);
    }

    // ---- MFMA operand / accumulator layout for the four families
    {
        void *dx = nullptr, *dy = nullptr, *dout = nullptr;
        HIP_TRY(hipMalloc(&dx, 2048));
        HIP_TRY(hipMalloc(&dy, 2048));
        HIP_TRY(hipMalloc(&dout, 1024));
        const char *names[4] = {"i8", "f8", "bf16", "f16"};
        for (int arith = 0; arith < 4; ++arith) {
            const int eb = arith <= AR_F8 ? 1 : 2;
            const int per_lane = 32 / eb;                    // elements per lane per operand
            std::vector<uint8_t> hx(2048), hy(2048);
            uint32_t rng = 12345u + arith;
            auto next = [&]() { rng = rng * 1664525u + 1013904223u; return (int)((rng >> 24) % 9) - 4; };
            for (int i = 0; i < 64 * per_lane; ++i) {
                host_encode_small(arith, next(), hx.data(), i);
                host_encode_small(arith, next(), hy.data(), i);
            }
            HIP_TRY(hipMemcpy(dx, hx.data(), 2048, hipMemcpyHostToDevice));
            HIP_TRY(hipMemcpy(dy, hy.data(), 2048, hipMemcpyHostToDevice));
            auto probe = arith == AR_I8 ? probe_mfma_kernel<AR_I8> : arith == AR_F8 ? probe_mfma_kernel<AR_F8>
                         : arith == AR_BF16 ? probe_mfma_kernel<AR_BF16> : probe_mfma_kernel<AR_F16>;
            HIP_TRY(launch_kernel(probe, dim3(1), dim3(64), 0, nullptr, (const char *)dx, (const char *)dy, (int *)dout));
            std::vector<int> hout(256);
            HIP_TRY(hipMemcpy(hout.data(), dout, 1024, hipMemcpyDeviceToHost));
            // assumed: operand lane l = row (l & 15), K group (l >> 4); the same element position of
            // the two operands meets in the contraction; accumulator lane l, register r =
            // D[first-operand row 4*(l >> 4) + r][second-operand row (l & 15)]
            int bad = 0;
            for (int l = 0; l < 64; ++l)
                for (int r = 0; r < 4; ++r) {
                    const int i = 4 * (l >> 4) + r, j = l & 15;
                    double sum = 0;
                    for (int g = 0; g < 4; ++g)
                        for (int e = 0; e < per_lane; ++e)
                            sum += (double)host_decode(arith, hx.data(), (g * 16 + i) * per_lane + e) *
                                   (double)host_decode(arith, hy.data(), (g * 16 + j) * per_lane + e);
                    double got;
                    if (arith == AR_I8) got = (double)hout[l * 4 + r];
                    else {
                        float f;
                        std::memcpy(&f, &hout[l * 4 + r], 4);
                        got = (double)f;
                    }
                    bad += got != sum;
                }
            std::snprintf(line, sizeof(line), "mfma %s: mismatched_accumulators=%d of 256\n", names[arith], bad);
            rep += line;
            if (bad) all_ok = false;
        }
        (void)hipFree(dx);
        (void)hipFree(dy);
        (void)hipFree(dout);
    }
    // ---- which XCD does workgroup i land on?  The tile raster assumes i % 8.
    {
        const int nwg = 64;
        void *dout = nullptr;
        HIP_TRY(hipMalloc(&dout, nwg * 8));
        HIP_TRY(launch_kernel(probe_xcc_kernel, dim3(nwg), dim3(64), 0, nullptr, (uint32_t *)dout));
        std::vector<uint32_t> h(nwg * 2);
        HIP_TRY(hipMemcpy(h.data(), dout, nwg * 8, hipMemcpyDeviceToHost));
        (void)hipFree(dout);
        int round_robin = 0;
        rep += "xcc of workgroups 0..31:";
        for (int i = 0; i < nwg; ++i) {
            if (i < 32) {
                std::snprintf(line, sizeof(line), " %u", h[i * 2] & 15u);
                rep += line;
            }
            round_robin += (int)(h[i * 2] & 15u) == i % kXcds;
        }
        std::snprintf(line, sizeof(line), "\nxcc round robin (wg %% 8): %d of %d workgroups\n", round_robin, nwg);
        rep += line;
    }
    if (buf && buflen) std::snprintf(buf, buflen, "%s", rep.c_str());
    return all_ok ? QGEMM_OK : QGEMM_ERR_UNSUPPORTED;
}

}  // extern "C"


// llm_accel.cpp -- C ABI of the resident decoder-layer path (host side).
//
// One context owns every device allocation: weights in the tile4x128
// layout, the norm table, the Q8.8 RoPE table, the paged KV cache, hidden
// pairs and scratch.  llm_task() validates a command in the controller's
// order, enqueues the sublayer's kernels on the context stream and returns
// the status record; nothing of the hidden state or KV cache crosses PCIe
// between tasks.
#include "llm_accel.h"

#include <hip/hip_runtime.h>

#include <algorithm>
#include <iterator>
#include <cmath>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <string>
#include <chrono>
#include <functional>
#include <thread>
#include <vector>

#include "attention.h"
#include "coherent.h"
#include "fixed_point.h"
#include "kernels.h"
#include "ops.h"
#include "prefill.h"

namespace {

thread_local std::string g_err;

int fail(int code, const std::string& msg) {
    g_err = msg;
    return code;
}

#define HIP_TRY(expr)                                                   \
    do {                                                                \
        hipError_t e_ = (expr);                                         \
        if (e_ != hipSuccess)                                           \
            return fail(LLM_E_HIP, std::string(#expr) + ": " +          \
                                       hipGetErrorString(e_));          \
    } while (0)

// Stream synchronisation of a context, then the check that no wait
// between workgroups of a launch gave up since the last one.
#define SYNC_TRY(c)                                                     \
    do {                                                                \
        HIP_TRY(hipStreamSynchronize((c)->stream));                     \
        if (int rc_ = check_waits(c)) return rc_;                       \
    } while (0)

}  // namespace

namespace llm {
int set_last_error(int code, const char* msg) { return fail(code, msg); }
}  // namespace llm

namespace {

uint32_t round_up(uint32_t v, uint32_t m) { return (v + m - 1) / m * m; }
uint64_t cdiv(uint64_t a, uint64_t b) { return (a + b - 1) / b; }

// One weight matrix in the tile4x128 layout.
struct Matrix {
    int16_t* d = nullptr;
    uint32_t n = 0, k = 0, n_pad = 0, k_pad = 0, steps = 0;
    // matrix-core copy: byte-plane records and (sum hi, sum lo) per output
    int8_t* mf = nullptr;
    int32_t* ms = nullptr;
    uint32_t nc = 0, kq = 0;
    int32_t* ctx_part = nullptr;     // the context's split scratch
    uint32_t* ctx_count = nullptr;
    int maxw[3] = {0, 0, 0};  // per stored projection (qkv keeps three)
    // 12-bit copy: p12_ok once every stored projection (Q, K, V of the
    // Q|K|V matrix, else one) is loaded with weights in [-2048, 2047]
    uint8_t* p12 = nullptr;
    bool p12_fit[3] = {false, true, true};
    bool p12_ok = false;
    // held in 12 bits only (no 16-bit copy, no byte planes) until a weight
    // outside [-2048, 2047] arrives (widen_matrix)
    bool p12_only = false;
    // corrections of the 12-bit copy (kCorrSlots words per output row,
    // allocated with the first weight outside 12 bits; see ProjArgs)
    uint32_t* corr = nullptr;
    bool corr_any = false;
    // gate <-> up and Q|K|V <-> O: read together (gate|up in one launch,
    // Q|K|V and O in the fused attention sublayer), so held in the same
    // layout
    Matrix* partner = nullptr;
    int L = 16;               // int32 widening interval in k-steps
    size_t elems() const { return (size_t)n_pad * k_pad; }
};

enum { M_QKV = 0, M_O = 1, M_GATE = 2, M_UP = 3, M_DOWN = 4, M_COUNT = 5 };

// Largest int32 accumulation interval (k-steps of 8 products per lane)
// that cannot overflow for any int16 activation: 8 * L * 32768 * max|w|
// < 2^31.  0 selects the per-product int64 path.
int widening_interval(int maxw) {
    if (maxw == 0) return 16;
    const int64_t lim = ((int64_t)1 << 31) - 1;
    const int64_t per_step = (int64_t)8 * 32768 * maxw;
    const int64_t allowed = lim / per_step;
    for (int L : {16, 8, 4, 1})
        if (allowed >= L) return L;
    return 0;
}

}  // namespace

struct llm_ctx {
    llm_shape_t s{};
    int device = 0;
    hipStream_t stream = nullptr;
    uint32_t H = 0, I = 0, Hq = 0, Hkv = 0, d = 0, G = 0, Ckv = 0, L = 0;
    uint32_t max_seq = 0, tiles = 0, Hp = 0, Ip = 0, Nqkv = 0;
    int32_t qk_scale = 0;
    int16_t* arena = nullptr;          // all weights
    std::vector<Matrix> mats;          // [layer][M_COUNT]
    std::vector<bool> loaded;          // [layer][7]
    bool norms_loaded = false;
    int16_t* norms = nullptr;
    int16_t* rope = nullptr;
    int16_t* exp8 = nullptr;
    uint32_t* silu8 = nullptr;  // per exp8 entry e: e | fx_recip(256 + e) << 16
    int16_t* exp14 = nullptr;
    int16_t* kcache = nullptr;
    int16_t* vcache = nullptr;
    std::vector<int16_t*> pairs;       // [8][Hp]
    int16_t* xn_attn = nullptr;        // [8][Hp] attention-norm output
    int16_t* xn_ffn = nullptr;         // [8][Hp] FFN-norm output
    int16_t* qkv = nullptr;            // [8][Nqkv]
    int16_t* attn = nullptr;           // [8][Hp]
    int16_t* act = nullptr;            // [8][Ip]
    // attention split-path scratch
    uint32_t chunk_tiles = 4;
    int32_t* c_flag = nullptr;
    int32_t* c_tsum = nullptr;
    int32_t* c_sum = nullptr;
    int16_t* s_scores = nullptr;
    int16_t* s_tmax = nullptr;
    int32_t* s_tsum = nullptr;
    int16_t* s_tval = nullptr;
    uint32_t* counters = nullptr;
    size_t counter_bytes = 0, rht_words = 0;
    // fused attention sublayer: arrival counters (growing across launches)
    // and the host-visible word a kernel sets when one of its waits gave up
    uint32_t* sync = nullptr;
    uint32_t* host_abort = nullptr;
    bool fused = true;                 // LLM_ACCEL_FUSED=0 disables it
    bool gqa = true;                   // GQA tile path; LLM_ACCEL_GQA=0 disables it
    // contexts of at least this many tiles take the GQA tile path (shorter
    // ones run faster with a workgroup per query head and tile);
    // LLM_ACCEL_GQA_MIN_TILES overrides it
    uint32_t gqa_min_tiles = 64;
    // blocks of kMfMinRows or more rows take the GQA path from 5 tiles: the
    // one-launch per-head tile grid (rows x heads x tiles workgroups) no
    // longer fits the device there and the two-launch pair is slower
    // (configs[4] prompt: 58.8 -> 57.6 us per 8-row block and layer); one
    // or two rows keep the per-head tile path below 64 tiles (decode at
    // ~1.1k positions: 42.2 against 45.8 us per forward)
    uint32_t gqa_min_tiles_block = 5;
    // the tile path (5-64 tiles) in one launch when the grid fits on the
    // device at once; LLM_ACCEL_TILE_FUSED=0 keeps its two launches
    bool tile_fused = true;
    // 12-bit copies of the weight matrices for single decode rows (weights
    // in [-2048, 2047]); LLM_ACCEL_P12=0 keeps the 16-bit copies only
    bool p12 = true;
    // the matrix-core path reads the 12-bit copies where every matrix of a
    // launch has one; LLM_ACCEL_MF12=0 keeps it on the byte planes
    bool mf12 = true;
    int32_t* s_tmax32 = nullptr;       // tile maxima published in that launch
    int32_t* s_gmax32 = nullptr;       // GQA path: tagged tile maxima
    uint32_t gqa_epoch = 0;            // epoch of the last GQA launch
    // GQA scores and PV in one launch when the grid fits on the device;
    // LLM_ACCEL_GQA_FUSED=0 keeps three launches
    bool gqa_fused = true;
    // LLM_ACCEL_COOP=1: the one-launch attention kernels go through the
    // cooperative launch, which refuses a grid the device cannot hold at
    // once (then the separate launches run).  Off by default: measured at
    // +19 us per one-layer decode forward (40.7 -> 59.8 us at 320
    // positions); the bounded waits and llm_generate's wait-free re-run
    // cover the same case without that cost.
    bool coop = false;
    // ... with the run-sum scan as workgroups of that launch (tagged tile
    // sums in s_gsum64); LLM_ACCEL_GQA_SCAN_FUSED=0 keeps it a launch
    uint64_t* s_gsum64 = nullptr;
    bool gqa_scan_fused = true;
    uint32_t sync_qkv[32] = {};        // QKV arrivals per line so far, mod 2^32
    uint32_t sync_attn = 0;            // attention arrivals per line, mod 2^32
    // bound of one wait (100 MHz ticks); LLM_ACCEL_WAIT_LIMIT overrides it
    // (tests force the time-out path with a tiny value)
    uint32_t wait_limit = 0;
    // residency of the fused launch per (rows - 1, QKV epilogue is the
    // input norm): -1 until first needed
    int sub_cap[2][2] = {{-1, -1}, {-1, -1}};
    // the one-launch tile path and O in one launch for decode rows at 5-64
    // tiles; LLM_ACCEL_TILE_O=0 keeps them two launches
    bool tile_o = true;
    int tile_o_cap[2][5] = {{-1, -1, -1, -1, -1}, {-1, -1, -1, -1, -1}};  // rows x variant
    int cus = 0;
    // RMSNorm gain: > 0 when it is the same for every row (hidden >= 128:
    // fm_t(hidden) saturates, recip() returns 0, the mean square is 0 and
    // the gain is rsqrt(0)); 0 selects the per-row reduction.
    int32_t const_gain = 0;
    // Normalised copies of a pair computed in a producing epilogue: valid
    // while that pair is not written again.  pair < 0 means empty.
    struct NormCache { int pair = -1; uint32_t layer = 0; };
    NormCache attn_cache, ffn_cache;
    // Final RMSNorm of pair `pair` (the last layer's FFN output, `rows`
    // rows) held in xn_final, whose rows rows..7 are those of pair `src`
    // (that layer's FFN input): a Task 20 from `pair` into `src` with the
    // same row count becomes an exchange of buffers.
    struct FinalCache { int pair = -1, src = -1; uint32_t rows = 0; };
    FinalCache final_cache;
    int16_t* xn_final = nullptr;        // [8][Hp]
    // Operator-level commands (llm_op): the context's own in / aux / out
    // port buffers and the 8-row projection staging, allocated on first use.
    bool ports_ready = false, port_out = false;
    int16_t* ports[3] = {nullptr, nullptr, nullptr};
    size_t port_n = 0;                  // elements per port
    int16_t* op_stage = nullptr;        // [8][max(Hp, Ip)]
    int32_t* op_tsum = nullptr;         // tile sums of the operator-level flash attention
    // partial sums / arrival counters of the split matrix-core projection
    int32_t* mf_part = nullptr;
    uint32_t* mf_count = nullptr;
    // Pairs whose device address was handed out keep their buffer.
    std::vector<char> exported;
    std::vector<void*> allocations;
    std::vector<hipEvent_t> events;
    // per-launch timing (measurement only)
    bool timing = false;
    std::vector<hipEvent_t> ev_pool;
    struct Timed { int kid; hipEvent_t a, b; };
    std::vector<Timed> pending;
    double kernel_ms[LLM_K_COUNT] = {};
    uint64_t kernel_n[LLM_K_COUNT] = {};

    // LM head [vocab][hidden] (tile4x128) and the argmax keys of 8 rows
    Matrix lm;
    uint32_t lm_vocab = 0;
    unsigned long long* lm_keys = nullptr;

    // Request loop (llm_generate): pinned staging of the embedding rows of
    // one request (copied to the device asynchronously, one forward's
    // rows at a time), pinned argmax keys, stream events, the optional line
    // sink, and counts of host <-> device transfers over the context's life.
    int16_t* stage = nullptr;
    size_t stage_rows = 0;
    unsigned long long* keys_host = nullptr;
    std::vector<hipEvent_t> gen_events;
    llm_log_fn log_fn = nullptr;
    void* log_user = nullptr;
    // Layer-major prompt path (prefill.h) of llm_generate: its buffers, one
    // allocation sized for `rows` rows (a multiple of kPfRowPad), made by the
    // first prompt that takes it and replaced by a larger one when a longer
    // prompt comes.  Where the device has no room for it, or it would pass
    // LLM_ACCEL_PROMPT_BYTES, fewer rows run at a time, or the prompt in
    // blocks; LLM_ACCEL_PROMPT=0 keeps every prompt in blocks
    struct Prompt {
        uint32_t rows = 0;
        uint8_t* base = nullptr;
        int16_t *in = nullptr, *ha = nullptr, *hb = nullptr, *qkv = nullptr;
        int8_t *xn = nullptr, *xa = nullptr, *act = nullptr, *qp = nullptr, *kp = nullptr,
               *vp = nullptr;
        int32_t *kbias = nullptr, *rowsum = nullptr;
        uint32_t *kvflag = nullptr, *qflag = nullptr, *count = nullptr;
        int64_t* part = nullptr;
        size_t part_bytes = 0;
    } pf;
    bool prompt_path = true;
    size_t prompt_bytes = SIZE_MAX;
    // Transfers of rows and keys with the host: pinned staging (in: host to
    // device, out: device to host), the pinned word a transfer's kernel sets
    // to its number once its values are visible, and a device word for its
    // workgroups' arrivals.  `busy`: what has been enqueued since a transfer
    // or synchronisation was last seen to complete (not relied on once the
    // stream was handed out; from then on no copy into a pair or port is left
    // under way either, so that no other call has to wait on a stream that
    // the caller may be capturing).
    int16_t *io_in = nullptr, *io_out = nullptr;
    size_t io_elems = 0;
    uint32_t* io_flag = nullptr;
    uint32_t* io_count = nullptr;
    uint32_t io_seq = 0;
    enum Busy { QUIET, COPIES_IN, WORK };
    Busy busy = WORK;
    bool stream_out = false;
    bool copies_open = false;  // a copy into a pair or port may be under way
    size_t io_used = 0;   // of io_in, by copies not known to be complete
    uint64_t n_h2d_rows = 0;   // hidden-row uploads (calls)
    uint64_t n_d2h_rows = 0;   // hidden-row downloads (calls)
    uint64_t n_kv_moves = 0;   // KV reads / writes (calls)
    uint64_t n_argmax = 0;     // argmax key read-backs (calls)
    uint64_t n_wait_reruns = 0;  // forwards re-run without waits (llm_generate)
    // Stream-event times of the profiled forwards (a line sink set), summed
    // over the context's life: the reference's coarse_* report fields.
    double coarse_active_ms = 0, coarse_input_ms = 0, coarse_host_ms = 0;

    Matrix& mat(uint32_t layer, int m) { return mats[layer * M_COUNT + m]; }
};

namespace {

// Brackets one kernel launch with events when timing is enabled.
struct TimedScope {
    llm_ctx* c;
    int kid;
    hipEvent_t a = nullptr;
    TimedScope(llm_ctx* ctx, int k) : c(ctx), kid(k) {
        if (!c->timing) return;
        a = take();
        (void)hipEventRecord(a, c->stream);
    }
    ~TimedScope() {
        if (!c->timing || !a) return;
        hipEvent_t b = take();
        (void)hipEventRecord(b, c->stream);
        c->pending.push_back({kid, a, b});
    }
    hipEvent_t take() {
        if (c->ev_pool.empty()) {
            hipEvent_t e;
            (void)hipEventCreate(&e);
            return e;
        }
        hipEvent_t e = c->ev_pool.back();
        c->ev_pool.pop_back();
        return e;
    }
};

void harvest_timing(llm_ctx* c) {
    (void)hipStreamSynchronize(c->stream);
    for (auto& t : c->pending) {
        float ms = 0;
        if (hipEventElapsedTime(&ms, t.a, t.b) == hipSuccess) {
            c->kernel_ms[t.kid] += ms;
            c->kernel_n[t.kid] += 1;
        }
        c->ev_pool.push_back(t.a);
        c->ev_pool.push_back(t.b);
    }
    c->pending.clear();
}

// After a synchronisation: a fused launch whose wait gave up (bounded
// waits end the kernel instead of hanging) left its counters behind and
// invalid results; clear both.  Returns whether there was one.
bool clear_waits(llm_ctx* c) {
    if (!c->host_abort || __atomic_load_n(c->host_abort, __ATOMIC_ACQUIRE) == 0) return false;
    (void)hipMemsetAsync(c->sync, 0, llm::kSyncWords * 4, c->stream);
    // counters a workgroup that left a wait early did not reset
    (void)hipMemsetAsync(c->counters, 0, c->counter_bytes, c->stream);
    // and flags of the one-launch tile path a workgroup did not clear
    (void)hipMemsetAsync(c->s_tmax32, 0, c->rht_words * 4, c->stream);
    (void)hipMemsetAsync(c->s_tsum, 0, c->rht_words * 4, c->stream);
    (void)hipStreamSynchronize(c->stream);
    std::fill(std::begin(c->sync_qkv), std::end(c->sync_qkv), 0u);
    c->sync_attn = 0;
    __atomic_store_n(c->host_abort, 0u, __ATOMIC_RELEASE);
    return true;
}

// The same, reported as an error of the call that synchronised.
int late_error();
int check_waits(llm_ctx* c) { return clear_waits(c) ? late_error() : 0; }

int io_wait(llm_ctx* c, uint32_t seq);
int ensure_keys_host(llm_ctx* c);

// Everything enqueued so far has completed; `late` receives whether a
// bounded wait gave up since the last time that was seen.
int quiesce(llm_ctx* c, bool* late) {
    *late = false;
    if (c->busy == llm_ctx::QUIET && !c->stream_out) return 0;
    const uint32_t seq = ++c->io_seq;  // an empty transfer
    HIP_TRY(llm::launch_io_rows(nullptr, 0, nullptr, 0, 0, 0, c->io_count, c->io_flag, seq,
                                c->stream));
    if (int rc = io_wait(c, seq)) return rc;
    *late = clear_waits(c);
    return 0;
}
int late_error() {
    return fail(LLM_E_HIP, "a wait between workgroups of a fused launch timed out; "
                           "results since the last synchronisation are invalid");
}

// One port holds the largest tensor an operator exchanges: 8 feature rows
// of the hidden or intermediate width, every KV head's K / V panel of 64
// positions, or 64 scores per query head.
size_t port_elems(const llm_ctx* c) {
    return std::max({(size_t)8 * c->Hp, (size_t)8 * c->Ip, (size_t)64 * c->Hq, (size_t)64 * c->Ckv});
}

// Staging of at least `elems` int16 each way (made for the ports' size when
// the context is created).
int io_buffers(llm_ctx* c, size_t elems) {
    if (c->io_elems >= elems) return 0;
    HIP_TRY(hipStreamSynchronize(c->stream));  // a transfer may still read it
    if (c->io_in) (void)hipHostFree(c->io_in);
    c->io_in = c->io_out = nullptr;
    c->io_elems = 0;
    elems = (2 * elems + 2047) / 2048 * 2048;  // the two operands of a command
    if (hipHostMalloc((void**)&c->io_in, 2 * elems * 2, hipHostMallocDefault) != hipSuccess)
        return fail(LLM_E_NOMEM, "hipHostMalloc failed");
    c->io_out = c->io_in + elems;
    c->io_elems = elems;
    return 0;
}

// Waits until transfer `seq` (the last work enqueued) is complete: polls
// its word for a while, then leaves the wait to the runtime.
int io_wait(llm_ctx* c, uint32_t seq) {
    for (uint32_t i = 0; i < 200000; i++) {
        if (__atomic_load_n(c->io_flag, __ATOMIC_ACQUIRE) == seq) {
            c->busy = llm_ctx::QUIET;
            c->copies_open = false;
            return 0;
        }
        __builtin_ia32_pause();
    }
    HIP_TRY(hipStreamSynchronize(c->stream));
    if (__atomic_load_n(c->io_flag, __ATOMIC_ACQUIRE) != seq)
        return fail(LLM_E_HIP, "a transfer to the host did not complete");
    c->busy = llm_ctx::QUIET;
    c->copies_open = false;
    return 0;
}

// Every copy into a pair or port has completed: before the caller receives
// an address or the stream, through which it can reach the values without a
// call that waits for them.  Leaves `busy` and a wait that gave up to the
// next call that reports it.
int finish_copies(llm_ctx* c) {
    if (!c->copies_open) return 0;
    HIP_TRY(hipStreamSynchronize(c->stream));
    c->copies_open = false;
    return 0;
}

// Rows of `cols` values from host memory into device rows: staged, the copy
// enqueued and, unless `wait` or the stream was handed out, not waited for.
int rows_in(llm_ctx* c, const int16_t* host, int16_t* dev, uint32_t ld_dev, uint32_t cols,
            uint32_t rows, bool wait) {
    bool late = false;
    const size_t n = (size_t)rows * cols;
    if (c->busy == llm_ctx::COPIES_IN && !c->stream_out && c->io_used + n <= c->io_elems) {
        // only such copies are under way, and the staging has room
    } else {
        if (int rc = quiesce(c, &late)) return rc;
        c->io_used = 0;
    }
    if (n) {
        if (int rc = io_buffers(c, n)) return rc;
        int16_t* from = c->io_in + c->io_used;
        std::memcpy(from, host, n * 2);
        c->io_used += (n + 7) / 8 * 8;
        HIP_TRY(llm::launch_io_rows(from, cols, dev, ld_dev, cols, rows, nullptr, nullptr, 0,
                                    c->stream));
        c->busy = llm_ctx::COPIES_IN;
        c->copies_open = true;
        if (wait || c->stream_out)
            if (int rc = finish_copies(c)) return rc;
    }
    return late ? late_error() : 0;
}

// The same from the device, complete on return, with everything enqueued
// before it.
int rows_out(llm_ctx* c, const int16_t* dev, uint32_t ld_dev, int16_t* host, uint32_t cols,
             uint32_t rows) {
    if (rows && cols) {
        if (int rc = io_buffers(c, (size_t)rows * cols)) return rc;
        const uint32_t seq = ++c->io_seq;
        HIP_TRY(llm::launch_io_rows(dev, ld_dev, c->io_out, cols, cols, rows, c->io_count,
                                    c->io_flag, seq, c->stream));
        if (int rc = io_wait(c, seq)) return rc;
        std::memcpy(host, c->io_out, (size_t)rows * cols * 2);
        return check_waits(c);
    }
    bool late;
    if (int rc = quiesce(c, &late)) return rc;
    return late ? late_error() : 0;
}

// While in scope, the context enqueues only launches whose workgroups never
// wait for one another (separate QKV / attention / O launches, the
// two-launch tile and GQA paths): the request loop re-runs with it what a
// bounded wait that gave up invalidated.  The reference's controller either
// completes a command or returns a status code
// (kernel/control_cache_8x64.cpp:5892-5957); a device shared with other
// work can leave a one-launch kernel's workgroups without a slot, which is
// the case this covers.
struct WaitFreeScope {
    llm_ctx* c;
    bool fused, tile_fused, gqa_fused, tile_o;
    explicit WaitFreeScope(llm_ctx* ctx)
        : c(ctx), fused(ctx->fused), tile_fused(ctx->tile_fused), gqa_fused(ctx->gqa_fused),
          tile_o(ctx->tile_o) {
        c->fused = c->tile_fused = c->gqa_fused = c->tile_o = false;
    }
    ~WaitFreeScope() {
        c->fused = fused;
        c->tile_fused = tile_fused;
        c->gqa_fused = gqa_fused;
        c->tile_o = tile_o;
    }
};

int dev_alloc(llm_ctx* c, void** p, size_t bytes) {
    hipError_t e = hipMalloc(p, bytes);
    if (e != hipSuccess) {
        (void)hipGetLastError();  // not the next launch's
        return fail(LLM_E_NOMEM, "hipMalloc(" + std::to_string(bytes) +
                                     "): " + hipGetErrorString(e));
    }
    c->allocations.push_back(*p);
    // the fill runs behind the call, on the null stream, which the context's
    // non-blocking stream does not wait for
    e = hipMemset(*p, 0, bytes);
    if (e == hipSuccess) e = hipStreamSynchronize(nullptr);
    if (e != hipSuccess) return fail(LLM_E_HIP, hipGetErrorString(e));
    return 0;
}

// Nearest integer to v * 2^bits, v >= 0 (an AP_RND table constant).
int64_t table_const(long double v, int bits) {
    return (int64_t)floorl(ldexpl(v, bits) + 0.5L);
}

// hls::exp on ap_fixed<16,8>: the Q8.8 exponential of SiLU and of the
// Q8.8 softmax / flash operators (golden_exp, host/host_qwen_8x64.cpp:
// 578-586; cu_exp_approx, kernel/compute_stream.cpp:50-55).  The
// reference's HLS build instantiates it as three ROM lookups and two
// products (ROMs exp_x_msb_1_table, exp_x_msb_2_m_1_table, f_x_lsb_table;
// a 5-bit msb_2 field of weights 2^-2..2^-6; 25x18- and 25x25-bit
// multipliers -- results/qwen3b-e2e-20260820/build.raw.log:1469-1471,
// :1506-1516).  For x split into m1 (bits >= 2^-1, two's complement),
// m2 (bits 2^-2..2^-6) and l (bits 2^-7, 2^-8):
//   e^x ~= E1 (1 + E2)(1 + L),  E1 = e^m1 rounded at 2^-14,
//   E2 = e^m2 - 1 rounded at 2^-26, L = l + (e^l - 1 - l) rounded at 2^-24,
// truncated to Q8.8.  These widths reproduce the reference's published
// post-FFN fingerprint and final-hidden checksums; the result differs
// from floor(e^x * 256) at 13 inputs in [-8, 0].
int16_t hls_exp_q8_8(int x) {
    const int m1 = x & ~127, m2 = (x - m1) & ~3, l = (x - m1) & 3;
    const __int128 e1 = table_const(expl((long double)m1 / 256.0L), 14);
    const __int128 e2 = table_const(expm1l((long double)m2 / 256.0L), 26);
    const long double lf = (long double)l / 256.0L;
    const __int128 lt = ((__int128)l << 16) + table_const(expm1l(lf) - lf, 24);
    // (1 + E2)(1 + L) in units of 2^-50, then E1 * that in units of 2^-64.
    const __int128 f = ((__int128)1 << 50) + (e2 << 24) + (lt << 26) + e2 * lt;
    const __int128 y = (e1 * f) >> 56;
    return y > 32767 ? (int16_t)32767 : (int16_t)y;
}

// exp tables for x = -2048/256 .. 0: the Q8.8 one above, and the Q2.14
// probabilities floor(e^x * 2^14) (hls::exp on ap_fixed<18,4>,
// host/host_qwen_8x64.cpp:588-596).
void build_exp_tables(int16_t* q8_8, int16_t* q2_14) {
    for (int x = -2048; x <= 0; x++) {
        q8_8[x + 2048] = hls_exp_q8_8(x);
        long double e = expl((long double)x / 256.0L);
        q2_14[x + 2048] = (int16_t)floorl(e * 16384.0L);
    }
}

int16_t quantize_fix16(double v) {  // host/host_qwen_8x64.cpp:496-505
    double s = std::round(v * 256.0);
    if (s > 32767.0) return 32767;
    if (s < -32768.0) return -32768;
    return (int16_t)s;
}

// Rows [row0, row0 + rows) of matrix m get row-major weights w[rows][k].
// Runs fn(i) for i in [0, n) on up to 16 host threads (weight repacking).
template <typename F>
void parallel_for(uint32_t n, F fn) {
    const uint32_t T = std::max(1u, std::min({16u, std::thread::hardware_concurrency(), n}));
    if (T <= 1) {
        for (uint32_t i = 0; i < n; i++) fn(i);
        return;
    }
    std::vector<std::thread> th;
    for (uint32_t t = 0; t < T; t++)
        th.emplace_back([&, t] {
            for (uint32_t i = t; i < n; i += T) fn(i);
        });
    for (auto& x : th) x.join();
}

// Rows [0, rows) of w[rows][k] in the tile4x128 layout, rows padded to a
// whole block; maxw receives the largest |w|.
std::vector<int16_t> tile_rows(const Matrix& m, uint32_t rows, const int16_t* w, int* maxw) {
    const uint32_t rows_pad = round_up(rows, llm::kBlockRows);
    const uint32_t S = m.steps;
    std::vector<int16_t> buf((size_t)rows_pad * m.k_pad, 0);
    std::vector<int> row_max(rows, 0);
    parallel_for(rows, [&](uint32_t n) {
        const uint32_t b = n / 4, i = n % 4;
        const int16_t* src = w + (size_t)n * m.k;
        int mx = 0;
        for (uint32_t k = 0; k < m.k; k++) {
            const uint32_t s = k / 128, j = (k % 128) / 8, e = k % 8;
            const int16_t v = src[k];
            buf[(((size_t)b * S + s) * 4 + i) * 128 + j * 8 + e] = v;
            mx = std::max(mx, std::abs((int)v));
        }
        row_max[n] = mx;
    });
    int mw = 0;
    for (int v : row_max) mw = std::max(mw, v);
    if (maxw) *maxw = mw;
    return buf;
}

// The 12-bit copy (layout in kernels.hip, proj_p12_kernel) of the tile
// rows buf, from row row0 on (every weight in [-2048, 2047]).
int upload_p12(Matrix& m, uint32_t row0, const std::vector<int16_t>& buf) {
    const uint32_t S = m.steps;
    const size_t nsteps = buf.size() / 512;
    std::vector<uint8_t> pk(nsteps * llm::kP12Step, 0);
    parallel_for((uint32_t)nsteps, [&](uint32_t bs) {
        const int16_t* t = &buf[(size_t)bs * 512];  // [4 rows][16 lanes][8]
        uint8_t* o = &pk[(size_t)bs * llm::kP12Step];
        for (uint32_t ln = 0; ln < 64; ln++) {
            uint32_t word = 0;
            for (uint32_t e = 0; e < 8; e++) {
                const uint32_t u = (uint32_t)(t[ln * 8 + e] + 2048);
                o[8 * ln + e] = (uint8_t)(u & 255);
                word |= (u >> 8) << ((e & 1) * 16 + (e >> 1) * 4);
            }
            std::memcpy(o + 512 + 4 * ln, &word, 4);
        }
    });
    HIP_TRY(hipMemcpy(m.p12 + (size_t)(row0 / 4) * S * llm::kP12Step, pk.data(), pk.size(),
                      hipMemcpyHostToDevice));
    return 0;
}

// Byte-plane records (when the matrix holds them) and the per-output byte
// sums (always: the matrix-core kernels over either layout use them) of
// the 16-output chunks that rows [row0, row0 + rows) cover.
int upload_planes(Matrix& m, uint32_t row0, uint32_t rows, const int16_t* w) {
    if (row0 % llm::kMfRows != 0) return fail(LLM_E_ARG, "projection rows not aligned to 16");
    const uint32_t c0 = row0 / llm::kMfRows;
    const uint32_t c1 = (uint32_t)cdiv(row0 + rows, llm::kMfRows);
    const uint32_t KQ = m.kq;
    std::vector<int8_t> rec(m.mf ? (size_t)(c1 - c0) * KQ * llm::kMfRecord : 0);
    std::vector<int32_t> sums((size_t)(c1 - c0) * llm::kMfRows * 2, 0);
    parallel_for(c1 - c0, [&](uint32_t ci) {
        const uint32_t cc = c0 + ci;
        for (uint32_t jj = 0; jj < llm::kMfRows; jj++) {
            const uint32_t local = cc * llm::kMfRows + jj - row0;
            const bool valid = local < rows;
            int32_t* sm = &sums[((size_t)ci * llm::kMfRows + jj) * 2];
            for (uint32_t q = 0; q < KQ; q++)
                for (uint32_t g = 0; g < 4; g++)
                    for (uint32_t b = 0; b < 16; b++) {
                        const uint32_t k = q * llm::kMfCols + 16 * g + b;
                        const int32_t v = valid && k < m.k ? w[(size_t)local * m.k + k] : 0;
                        const int8_t hi = (int8_t)(v >> 8);
                        const int8_t lo = (int8_t)((v & 255) ^ 0x80);
                        if (m.mf) {
                            const size_t o = ((size_t)ci * KQ + q) * llm::kMfRecord +
                                             (16 * g + jj) * 16 + b;
                            rec[o] = hi;
                            rec[o + 1024] = lo;
                        }
                        sm[0] += hi;
                        sm[1] += lo;
                    }
        }
    });
    if (m.mf)
        HIP_TRY(hipMemcpy(m.mf + (size_t)c0 * KQ * llm::kMfRecord, rec.data(), rec.size(),
                          hipMemcpyHostToDevice));
    HIP_TRY(hipMemcpy(m.ms + (size_t)c0 * llm::kMfRows * 2, sums.data(),
                      sums.size() * sizeof(int32_t), hipMemcpyHostToDevice));
    return 0;
}

int dev_free(llm_ctx* c, void* p) {
    auto it = std::find(c->allocations.begin(), c->allocations.end(), p);
    if (it != c->allocations.end()) c->allocations.erase(it);
    HIP_TRY(hipFree(p));
    return 0;
}

// A matrix held in 12 bits only gets a weight outside [-2048, 2047]: it
// moves to the 16-bit copy and the byte planes, rebuilt for the rows loaded
// so far from the 12-bit copy (which is exact for them), and the 12-bit
// copy is released.
int widen_matrix(llm_ctx* c, Matrix& m) {
    HIP_TRY(hipStreamSynchronize(c->stream));
    const uint32_t S = m.steps;
    std::vector<uint8_t> pk((size_t)(m.n_pad / 4) * S * llm::kP12Step);
    HIP_TRY(hipMemcpy(pk.data(), m.p12, pk.size(), hipMemcpyDeviceToHost));
    std::vector<uint32_t> cw(m.corr_any ? (size_t)m.n_pad * llm::kCorrSlots : 0);
    if (m.corr_any)
        HIP_TRY(hipMemcpy(cw.data(), m.corr, cw.size() * 4, hipMemcpyDeviceToHost));
    std::vector<int16_t> w((size_t)m.n * m.k);
    parallel_for(m.n, [&](uint32_t n) {
        const uint32_t b = n / 4, i = n % 4;
        for (uint32_t k = 0; k < m.k; k++) {
            const uint32_t s = k / 128, j = (k % 128) / 8, e = k % 8, ln = 16 * i + j;
            const uint8_t* rec = &pk[((size_t)b * S + s) * llm::kP12Step];
            uint32_t word;
            std::memcpy(&word, rec + 512 + 4 * ln, 4);
            const uint32_t h = (word >> ((e & 1) * 16 + (e >> 1) * 4)) & 15;
            w[(size_t)n * m.k + k] = (int16_t)((int)(256 * h + rec[8 * ln + e]) - 2048);
        }
        // the weights the copy holds clamped
        for (uint32_t q = 0; q < (cw.empty() ? 0u : llm::kCorrSlots); q++) {
            const uint32_t e = cw[(size_t)n * llm::kCorrSlots + q];
            const int32_t d = (int16_t)(e & 0xffff);
            if (d) {
                int16_t& v = w[(size_t)n * m.k + (e >> 16)];
                v = (int16_t)(v + d);
            }
        }
    });
    int rc;
    if ((rc = dev_alloc(c, (void**)&m.d, m.elems() * sizeof(int16_t))) ||
        (rc = dev_alloc(c, (void**)&m.mf, (size_t)m.nc * m.kq * llm::kMfRecord)))
        return rc;
    const std::vector<int16_t> buf = tile_rows(m, m.n, w.data(), nullptr);
    HIP_TRY(hipMemcpy(m.d, buf.data(), buf.size() * sizeof(int16_t), hipMemcpyHostToDevice));
    if ((rc = upload_planes(m, 0, m.n, w.data()))) return rc;
    if ((rc = dev_free(c, m.p12))) return rc;
    m.p12 = nullptr;
    m.p12_ok = false;
    m.p12_only = false;
    if (m.corr && (rc = dev_free(c, m.corr))) return rc;
    m.corr = nullptr;
    m.corr_any = false;
    return 0;
}

int upload_rows(llm_ctx* c, Matrix& m, uint32_t row0, uint32_t rows,
                const int16_t* w, int which) {
    if (row0 % llm::kBlockRows != 0)
        return fail(LLM_E_ARG, "projection rows not aligned to 4");
    const uint32_t S = m.steps;
    int maxw = 0;
    std::vector<int16_t> buf = tile_rows(m, rows, w, &maxw);
    bool fits = true;
    for (size_t q = 0; fits && q < buf.size(); q++) fits = buf[q] >= -2048 && buf[q] <= 2047;
    int rc;
    // A matrix held in 12 bits keeps rows with at most kCorrSlots weights
    // outside the range: the copy holds them clamped and the row's
    // correction words the differences (exact: the kernels add
    // x[k] * delta to the row's sum).  More, and the matrix is widened.
    std::vector<int16_t> clamped;
    std::vector<uint32_t> cw;
    if (m.p12_only && !fits) {
        cw.assign((size_t)rows * llm::kCorrSlots, 0);
        bool sparse = true;
        for (uint32_t n = 0; sparse && n < rows; n++) {
            uint32_t q = 0;
            for (uint32_t k = 0; k < m.k; k++) {
                const int v = w[(size_t)n * m.k + k];
                if (v >= -2048 && v <= 2047) continue;
                if (q == llm::kCorrSlots) {
                    sparse = false;
                    break;
                }
                const int d = v - std::clamp(v, -2048, 2047);
                cw[(size_t)n * llm::kCorrSlots + q++] = (k << 16) | (uint16_t)(int16_t)d;
            }
        }
        if (sparse) {
            clamped.assign(w, w + (size_t)rows * m.k);
            for (auto& v : clamped) v = (int16_t)std::clamp((int)v, -2048, 2047);
            w = clamped.data();
            buf = tile_rows(m, rows, w, nullptr);
            fits = true;
            if (!m.corr && (rc = dev_alloc(c, (void**)&m.corr,
                                           (size_t)m.n_pad * llm::kCorrSlots * 4)))
                return rc;
            m.corr_any = true;
        } else {
            cw.clear();
            if ((rc = widen_matrix(c, m))) return rc;
            if (m.partner && m.partner->p12_only && (rc = widen_matrix(c, *m.partner))) return rc;
        }
    }
    if (m.corr) {
        // this part's rows: their corrections, or none
        if (cw.empty()) cw.assign((size_t)rows * llm::kCorrSlots, 0);
        HIP_TRY(hipMemcpy(m.corr + (size_t)row0 * llm::kCorrSlots, cw.data(), cw.size() * 4,
                          hipMemcpyHostToDevice));
    }
    if (m.d)
        HIP_TRY(hipMemcpy(m.d + (size_t)(row0 / 4) * S * 512, buf.data(),
                          buf.size() * sizeof(int16_t), hipMemcpyHostToDevice));
    if (m.p12) {
        m.p12_fit[which] = fits;
        m.p12_ok = m.p12_fit[0] && m.p12_fit[1] && m.p12_fit[2];
        if (fits && (rc = upload_p12(m, row0, buf))) return rc;
    }
    if (m.ms && (rc = upload_planes(m, row0, rows, w))) return rc;
    m.maxw[which] = maxw;
    m.L = widening_interval(std::max({m.maxw[0], m.maxw[1], m.maxw[2]}));
    return 0;
}

// Controller schedule counters for one accepted command
// (kernel/control_cache_8x64.cpp:5974-6481, attention tasks :5764,
// vector tasks :1856-1929).
void fill_counters(const llm_ctx* c, uint32_t op, uint32_t R, uint32_t pos,
                   llm_status_t* st) {
    const uint32_t vt = (R > 0 ? 1u : 0u) + (R > 4 ? 1u : 0u);
    const uint32_t hp = R * (uint32_t)cdiv(c->H, 16);
    const uint32_t ip = R * (uint32_t)cdiv(c->I, 16);
    if (op == LLM_OP_FINAL_NORM) {
        st->vector_tasks = vt;
        st->completed_packets = hp;
        return;
    }
    uint32_t waves = 0, mm = 0, vec = vt, pk = hp;
    const uint32_t begin = op == LLM_OP_FFN_SUBLAYER ? 4 : 0;
    const uint32_t end = op == LLM_OP_ATTENTION_SUBLAYER ? 4 : 7;
    for (uint32_t step = begin; step < end; step++) {
        const uint32_t out_dim = (step == 1 || step == 2) ? c->Ckv
                               : (step == 4 || step == 5) ? c->I : c->H;
        if (step == 3) {
            const uint32_t ow = (uint32_t)cdiv(c->d, 64);
            uint32_t at = 0;
            for (uint32_t t = 0; t < R; t++)
                at += 2 * (uint32_t)cdiv(pos + t + 1, 64) * (1 + ow);
            mm += at;
            pk += at * 32;
            waves += at / 2;
        }
        const uint32_t w = (uint32_t)cdiv(out_dim, 128);
        waves += w;
        mm += 2 * w;
        pk += 2 * w * 32;
        if (step == 3) {
            vec += vt;
            pk += hp;
            if (op != LLM_OP_ATTENTION_SUBLAYER) {
                vec += vt;
                pk += hp;
            }
        } else if (step == 5) {
            vec += vt;
            pk += ip;
        } else if (step == 6) {
            vec += vt;
            pk += hp;
        }
    }
    st->output_waves = waves;
    st->mm_tasks = mm;
    st->vector_tasks = vec;
    st->completed_packets = pk;
}

// A write to `pair` (task output, upload, device-pointer hand-out) drops
// every normalised copy derived from it.
void invalidate_pair(llm_ctx* c, int pair) {
    if (c->attn_cache.pair == pair) c->attn_cache.pair = -1;
    if (c->ffn_cache.pair == pair) c->ffn_cache.pair = -1;
    if (c->final_cache.pair == pair || c->final_cache.src == pair)
        c->final_cache.pair = c->final_cache.src = -1;
}

int check_layer_loaded(llm_ctx* c, uint32_t layer, bool attn, bool ffn) {
    if (!c->norms_loaded) return fail(LLM_E_STATE, "norm table not loaded");
    for (uint32_t p = 0; p < 7; p++) {
        const bool need = p < 4 ? attn : ffn;
        if (need && !c->loaded[layer * 7 + p])
            return fail(LLM_E_STATE, "layer " + std::to_string(layer) +
                                         " projection " + std::to_string(p) +
                                         " not loaded");
    }
    return 0;
}

// Matrix-core copies of the matrix (and of the up matrix for gate|up).
void set_mf(const llm_ctx* c, llm::ProjArgs& a, const Matrix& m, const Matrix* m2 = nullptr) {
    a.mf_p12 = c->mf12;
    a.corr0 = m.corr_any ? m.corr : nullptr;
    if (m2) a.corr1 = m2->corr_any ? m2->corr : nullptr;
    a.mf_part = m.ctx_part;
    a.mf_count = m.ctx_count;
    a.mf0 = m.mf;
    a.ms0 = m.ms;
    a.kq = m.kq;
    a.nc = m.nc;
    if (m2) {
        a.mf1 = m2->mf;
        a.ms1 = m2->ms;
    }
}

int enqueue_attention_sublayer(llm_ctx* c, uint32_t layer, uint32_t R,
                               uint32_t pos, int in_pair, int out_pair) {
    hipStream_t st = c->stream;
    const int16_t* in = c->pairs[in_pair];
    int16_t* out = c->pairs[out_pair];
    const bool cached = c->const_gain > 0 && c->attn_cache.pair == in_pair &&
                        c->attn_cache.layer == layer;
    // With a constant gain the projection normalises the raw rows itself
    // as it loads them.
    const bool norm_in = !cached && c->const_gain > 0;
    if (!cached && !norm_in) {
        TimedScope ts(c, LLM_K_RMSNORM);
        HIP_TRY(llm::launch_rmsnorm(in, c->Hp,
                                    c->norms + (size_t)(2 * layer) * c->H, c->H,
                                    c->xn_attn, c->Hp, R, c->const_gain, st));
    }
    const Matrix& mq = c->mat(layer, M_QKV);
    llm::ProjArgs a{};
    a.w0 = mq.d;
    a.steps = mq.steps;
    a.x = norm_in ? in : c->xn_attn;
    a.ldx = c->Hp;
    a.out = c->qkv;
    a.ldo = c->Nqkv;
    a.n = mq.n;
    a.rows = R;
    set_mf(c, a, mq);
    if (mq.p12_ok) a.p0 = mq.p12;  // single rows outside the fused launch
    if (norm_in) {
        a.in_gamma = c->norms + (size_t)(2 * layer) * c->H;
        a.in_gain = c->const_gain;
        a.in_cols = c->H;
    }
    const int qkv_epi = norm_in ? llm::EPI_STORE_NORM_IN : llm::EPI_STORE;
    llm::AttnArgs at{};
    at.qkv = c->qkv;
    at.ldqkv = c->Nqkv;
    at.rope = c->rope;
    const size_t layer_off = (size_t)layer * c->Hkv * c->tiles * llm::kTile * c->d;
    at.kcache = c->kcache + layer_off;
    at.vcache = c->vcache + layer_off;
    at.tiles = c->tiles;
    at.pos0 = pos;
    at.num_heads = c->Hq;
    at.num_kv_heads = c->Hkv;
    at.group = c->G;
    at.head_dim = c->d;
    at.qk_scale = c->qk_scale;
    at.exp14 = c->exp14;
    at.out = c->attn;
    at.ldo = c->Hp;
    at.chunk_tiles = c->chunk_tiles;
    const uint32_t gqa_from = R >= llm::kMfMinRows ? c->gqa_min_tiles_block : c->gqa_min_tiles;
    at.use_gqa = c->gqa && (uint32_t)cdiv(pos + R, llm::kTile) >= gqa_from ? 1u : 0u;
    at.max_tiles = c->tiles;
    at.tile_fused = c->tile_fused ? 1u : 0u;
    at.s_tmax32 = c->s_tmax32;
    at.s_gmax32 = c->s_gmax32;
    at.s_gsum64 = c->gqa_scan_fused ? c->s_gsum64 : nullptr;
    if (at.use_gqa && c->gqa_fused) {
        // a fresh epoch for the GQA path's tagged maxima and sums; past the
        // last one both are cleared (stream-ordered before this launch)
        if (++c->gqa_epoch > llm::kGqaEpochMax) {
            HIP_TRY(hipMemsetAsync(c->s_gmax32, 0, c->rht_words * 4, c->stream));
            HIP_TRY(hipMemsetAsync(c->s_gsum64, 0, c->rht_words * 8, c->stream));
            c->gqa_epoch = 1;
        }
        at.epoch = c->gqa_epoch;
    }

    at.abort = c->sync + llm::kSyncAbort;
    at.host_abort = c->host_abort;
    at.wait_limit = c->wait_limit;
    at.cus = (uint32_t)c->cus;
    at.coop = c->coop ? 1u : 0u;
    at.s_scores = c->s_scores;
    at.s_tmax = c->s_tmax;
    at.s_tsum = c->s_tsum;
    at.s_tval = c->s_tval;
    at.counters = c->counters;
    at.max_chunks = (uint32_t)cdiv(c->tiles, c->chunk_tiles);
    at.c_flag = c->c_flag;
    at.c_tsum = c->c_tsum;
    at.c_sum = c->c_sum;
    const uint32_t last_tiles = (uint32_t)cdiv(pos + R, llm::kTile);
    static_assert(llm::kTile == 64, "attention tiles are 64 positions");
    if (c->chunk_tiles == 0 || c->chunk_tiles > llm::kMaxChunkTiles)
        return fail(LLM_E_STATE, "attention chunk must be 1..8 tiles");
    const uint32_t chunks = (uint32_t)cdiv(last_tiles, c->chunk_tiles);
    const Matrix& mo = c->mat(layer, M_O);
    llm::ProjArgs o{};
    o.w0 = mo.d;
    o.steps = mo.steps;
    o.x = c->attn;
    o.ldx = c->Hp;
    o.out = out;
    o.ldo = c->Hp;
    o.res = in;
    o.ldr = c->Hp;
    o.n = mo.n;
    o.rows = R;
    set_mf(c, o, mo);
    if (mo.p12_ok) o.p0 = mo.p12;
    if (c->const_gain > 0) {  // FFN norm of this sublayer's output
        o.norm_out = c->xn_ffn;
        o.ldn = c->Hp;
        o.norm_gamma = c->norms + (size_t)(2 * layer + 1) * c->H;
        o.norm_gain = c->const_gain;
    }
    llm::SublayerArgs sub{};
    sub.qkv = a;
    sub.o = o;
    sub.at = at;
    sub.nq = llm::sublayer_qkv_workgroups(mq.n_pad / 4);
    sub.na = R * c->Hq;
    sub.no = llm::sublayer_o_workgroups(mo.n_pad / 4);
    sub.sync = c->sync;
    std::copy(std::begin(c->sync_qkv), std::end(c->sync_qkv), sub.qkv_base);
    sub.attn_base = c->sync_attn;
    sub.host_abort = c->host_abort;
    sub.wait_limit = c->wait_limit;
    int cap = 0;
    if (c->fused && R <= 2) {
        int& cc = c->sub_cap[R - 1][qkv_epi == llm::EPI_STORE_NORM_IN];
        if (cc < 0) cc = llm::sublayer_capacity(c->d, R, qkv_epi, c->cus);
        cap = cc;
    }
    if (c->fused && !llm::proj_uses_mfma(a, qkv_epi) && !llm::proj_uses_mfma(o, llm::EPI_RESID) &&
        llm::sublayer_fused_ok(sub, R, qkv_epi, mq.L, mo.L, cap)) {
        TimedScope ts(c, LLM_K_ATTN_SUBLAYER);
        HIP_TRY(llm::launch_attention_sublayer(sub, R, qkv_epi, std::min(mq.L, mo.L), st));
        // counter values after this launch
        for (uint32_t l = 0; l < llm::kSyncQkvLines; l++)
            c->sync_qkv[l] += sub.nq / llm::kSyncQkvLines + (l < sub.nq % llm::kSyncQkvLines);
        c->sync_attn += sub.na;
    } else {
        {
            TimedScope ts(c, LLM_K_QKV);
            HIP_TRY(llm::launch_proj(a, qkv_epi, mq.L, mq.n_pad / 4, st));
        }
        llm::TileOArgs to{};
        bool tile_o = false;
        if (c->tile_o && R <= 2 && !llm::proj_uses_mfma(o, llm::EPI_RESID)) {
            const int var = llm::tile_o_variant(o, mo.L);
            int& cc = c->tile_o_cap[R - 1][var];
            if (cc < 0) cc = llm::tile_o_capacity(c->d, R, var, c->cus);
            to.at = at;
            to.o = o;
            to.sync = c->sync;
            to.attn_base = c->sync_attn;
            to.host_abort = c->host_abort;
            to.wait_limit = c->wait_limit;
            tile_o = llm::tile_o_prepare(to, R, cc);
        }
        if (tile_o) {
            TimedScope ts(c, LLM_K_ATTENTION);
            HIP_TRY(llm::launch_attention_tile_o(to, R, mo.L, st));
            c->sync_attn += to.arrivals;  // counter values after this launch
        } else {
            {
                TimedScope ts(c, LLM_K_ATTENTION);
                HIP_TRY(llm::launch_attention(at, R, c->Hkv, chunks, st));
            }
            {
                TimedScope ts(c, LLM_K_OPROJ);
                HIP_TRY(llm::launch_proj(o, llm::EPI_RESID, mo.L, mo.n_pad / 4, st));
            }
        }
    }
    invalidate_pair(c, out_pair);
    if (c->const_gain > 0) c->ffn_cache = {out_pair, layer};
    return 0;
}

int enqueue_ffn_sublayer(llm_ctx* c, uint32_t layer, uint32_t R, int in_pair,
                         int out_pair) {
    hipStream_t st = c->stream;
    const int16_t* in = c->pairs[in_pair];
    int16_t* out = c->pairs[out_pair];
    const bool cached = c->const_gain > 0 && c->ffn_cache.pair == in_pair &&
                        c->ffn_cache.layer == layer;
    if (!cached) {
        TimedScope ts(c, LLM_K_RMSNORM);
        HIP_TRY(llm::launch_rmsnorm(in, c->Hp,
                                    c->norms + (size_t)(2 * layer + 1) * c->H,
                                    c->H, c->xn_ffn, c->Hp, R, c->const_gain, st));
    }
    const Matrix& mg = c->mat(layer, M_GATE);
    const Matrix& mu = c->mat(layer, M_UP);
    llm::ProjArgs a{};
    a.w0 = mg.d;
    a.w1 = mu.d;
    a.steps = mg.steps;
    a.x = c->xn_ffn;
    a.ldx = c->Hp;
    a.out = c->act;
    a.ldo = c->Ip;
    a.n = mg.n;
    a.rows = R;
    a.exp8 = c->exp8;
    a.silu8 = c->silu8;
    set_mf(c, a, mg, &mu);
    if (mg.p12_ok && mu.p12_ok) {
        a.p0 = mg.p12;
        a.p1 = mu.p12;
    }
    {
        TimedScope ts(c, LLM_K_GATEUP);
        HIP_TRY(llm::launch_proj(a, llm::EPI_SILU, std::min(mg.L, mu.L),
                                 mg.n_pad / 4, st));
    }
    const Matrix& md = c->mat(layer, M_DOWN);
    llm::ProjArgs dn{};
    dn.w0 = md.d;
    dn.steps = md.steps;
    dn.x = c->act;
    dn.ldx = c->Ip;
    dn.out = out;
    dn.ldo = c->Hp;
    dn.res = in;
    dn.ldr = c->Hp;
    dn.n = md.n;
    dn.rows = R;
    set_mf(c, dn, md);
    if (md.p12_ok) dn.p0 = md.p12;
    const bool next = c->const_gain > 0 && layer + 1 < c->L;
    if (c->const_gain > 0) {
        dn.ldn = c->Hp;
        dn.norm_gain = c->const_gain;
        if (next) {  // attention norm of the next layer
            dn.norm_out = c->xn_attn;
            dn.norm_gamma = c->norms + (size_t)(2 * (layer + 1)) * c->H;
        }
        // final norm (row 2L): a Task 20 may follow any layer's FFN
        // (run_composed_decoder_stack, host/host_qwen_8x64.cpp:1258-1445)
        dn.final_out = c->xn_final;
        dn.final_gamma = c->norms + (size_t)(2 * c->L) * c->H;
    }
    {
        TimedScope ts(c, LLM_K_DOWN);
        HIP_TRY(llm::launch_proj(dn, llm::EPI_RESID, md.L, md.n_pad / 4, st));
    }
    invalidate_pair(c, out_pair);
    if (next) c->attn_cache = {out_pair, layer + 1};
    if (c->const_gain > 0) c->final_cache = {out_pair, in_pair, R};
    return 0;
}

}  // namespace

extern "C" {

const char* llm_last_error(void) { return g_err.c_str(); }

int llm_ctx_create(const llm_shape_t* shape, int device, uint32_t num_pairs,
                   llm_ctx_t** out) {
    if (!shape || !out) return fail(LLM_E_ARG, "null argument");
    *out = nullptr;
    const llm_shape_t& s = *shape;
    if (s.hidden_size == 0 || s.intermediate_size == 0 || s.num_layers == 0 ||
        s.num_heads == 0 || s.num_kv_heads == 0 || s.max_seq_len == 0 ||
        s.hidden_size % s.num_heads != 0 || s.num_heads % s.num_kv_heads != 0)
        return fail(LLM_E_ARG, "inconsistent shape");
    const uint32_t d = s.hidden_size / s.num_heads;
    const uint32_t G = s.num_heads / s.num_kv_heads;
    if (d % 16 != 0 || d > 128 || G > 16 || G * d > 2048)
        return fail(LLM_E_ARG,
                    "head_dim must be a multiple of 16 and <= 128, group <= 16");
    if (s.hidden_size % 8 || s.intermediate_size % 4)
        return fail(LLM_E_ARG, "hidden must be a multiple of 8, intermediate of 4");
    if (num_pairs < 2) return fail(LLM_E_ARG, "need at least two hidden pairs");
    int ndev = 0;
    if (hipGetDeviceCount(&ndev) != hipSuccess || ndev == 0)
        return fail(LLM_E_HIP, "no HIP device available");
    if (device < 0 || device >= ndev) return fail(LLM_E_ARG, "bad device id");
    HIP_TRY(hipSetDevice(device));

    llm_ctx* c = new llm_ctx();
    c->s = s;
    c->device = device;
    c->H = s.hidden_size;
    c->I = s.intermediate_size;
    c->Hq = s.num_heads;
    c->Hkv = s.num_kv_heads;
    c->d = d;
    c->G = G;
    c->Ckv = s.num_kv_heads * d;
    c->L = s.num_layers;
    c->max_seq = s.max_seq_len;
    c->tiles = (uint32_t)cdiv(s.max_seq_len, llm::kTile);
    c->Hp = round_up(c->H, llm::kStepCols);
    c->Ip = round_up(c->I, llm::kStepCols);
    c->Nqkv = c->H + 2 * c->Ckv;
    c->qk_scale = (int32_t)std::floor(256.0 / std::sqrt((double)d) + 0.5);

    auto cleanup = [&](int code) {
        llm_ctx_destroy(c);
        return code;
    };
    if (hipStreamCreateWithFlags(&c->stream, hipStreamNonBlocking) != hipSuccess)
        return cleanup(fail(LLM_E_HIP, "hipStreamCreate failed"));

    // weights
    if (const char* e = std::getenv("LLM_ACCEL_P12")) c->p12 = std::strcmp(e, "0") != 0;
    if (const char* e = std::getenv("LLM_ACCEL_MF12")) c->mf12 = std::strcmp(e, "0") != 0;
    if (const char* e = std::getenv("LLM_ACCEL_TILE_O")) c->tile_o = std::strcmp(e, "0") != 0;
    c->mats.resize((size_t)c->L * M_COUNT);
    c->loaded.assign((size_t)c->L * 7, false);
    for (uint32_t l = 0; l < c->L; l++) {
        const uint32_t dims[M_COUNT][2] = {{c->Nqkv, c->H}, {c->H, c->H},
                                           {c->I, c->H}, {c->I, c->H},
                                           {c->H, c->I}};
        for (int m = 0; m < M_COUNT; m++) {
            Matrix& mt = c->mat(l, m);
            mt.n = dims[m][0];
            mt.k = dims[m][1];
            mt.n_pad = round_up(mt.n, llm::kBlockRows);
            mt.k_pad = round_up(mt.k, llm::kStepCols);
            mt.steps = mt.k_pad / llm::kStepCols;
        }
    }
    // A matrix whose shape every 12-bit kernel serves is held in 12 bits
    // only (1.5 bytes per weight) until a weight outside [-2048, 2047]
    // arrives; the others hold the 16-bit copy and the byte planes (and a
    // 12-bit copy for as long as their weights fit).
    auto p12_shape = [&](const Matrix& mt, int m) {
        return c->p12 && c->mf12 && mt.steps <= llm::kP12MaxSteps &&
               (m != M_QKV || (c->H % llm::kMfRows == 0 && c->Ckv % llm::kMfRows == 0));
    };
    for (uint32_t l = 0; l < c->L; l++) {
        c->mat(l, M_GATE).partner = &c->mat(l, M_UP);
        c->mat(l, M_UP).partner = &c->mat(l, M_GATE);
        c->mat(l, M_QKV).partner = &c->mat(l, M_O);
        c->mat(l, M_O).partner = &c->mat(l, M_QKV);
    }
    size_t wide_total = 0;
    for (int idx = 0; idx < (int)c->mats.size(); idx++) {
        Matrix& mt = c->mats[idx];
        mt.p12_only = p12_shape(mt, idx % M_COUNT);
        if (!mt.p12_only) wide_total += mt.elems();
    }
    int rc;
    if (wide_total && (rc = dev_alloc(c, (void**)&c->arena, wide_total * sizeof(int16_t))))
        return cleanup(rc);
    size_t off = 0;
    for (int idx = 0; idx < (int)c->mats.size(); idx++) {
        Matrix& mt = c->mats[idx];
        if (!mt.p12_only) {
            mt.d = c->arena + off;
            off += mt.elems();
        }
        if (idx % M_COUNT == M_QKV) mt.p12_fit[1] = mt.p12_fit[2] = false;
        if (c->p12)
            if ((rc = dev_alloc(c, (void**)&mt.p12, mt.elems() / 512 * llm::kP12Step)))
                return cleanup(rc);
        if (mt.p12_only) {
            // weights not loaded yet are 0 in the 12-bit image, as in the
            // 16-bit one
            if (llm::launch_p12_zero(mt.p12, mt.elems() / 512, c->stream) != hipSuccess)
                return cleanup(fail(LLM_E_HIP, "p12 initialisation"));
            mt.p12_fit[0] = mt.p12_fit[1] = mt.p12_fit[2] = true;
            mt.p12_ok = true;
        }
        // byte sums for both matrix-core layouts, byte planes for the
        // matrices held in 16 bits
        mt.nc = (uint32_t)cdiv(mt.n, llm::kMfRows);
        mt.kq = (uint32_t)cdiv(mt.k, llm::kMfCols);
        if (!mt.p12_only &&
            (rc = dev_alloc(c, (void**)&mt.mf, (size_t)mt.nc * mt.kq * llm::kMfRecord)))
            return cleanup(rc);
        if ((rc = dev_alloc(c, (void**)&mt.ms, (size_t)mt.nc * llm::kMfRows * 2 * 4)))
            return cleanup(rc);
        if (mt.p12_only) {
            // byte sums of all-zero rows: sum (w >> 8) = 0, sum ((w & 255) - 128)
            // = -128 per input of the padded K
            std::vector<int32_t> zs((size_t)mt.nc * llm::kMfRows * 2, 0);
            for (size_t q = 1; q < zs.size(); q += 2) zs[q] = -128 * (int32_t)(mt.kq * llm::kMfCols);
            if (hipMemcpy(mt.ms, zs.data(), zs.size() * 4, hipMemcpyHostToDevice) != hipSuccess)
                return cleanup(fail(LLM_E_HIP, "weight sums initialisation"));
        }
    }
    if (hipStreamSynchronize(c->stream) != hipSuccess)
        return cleanup(fail(LLM_E_HIP, "weight image initialisation"));
    // tables
    // norm table + one k-step of padding: the fused-norm projections read
    // gammas in whole k-steps
    if ((rc = dev_alloc(c, (void**)&c->norms,
                        ((size_t)(2 * c->L + 1) * c->H + c->Hp) * sizeof(int16_t))) ||
        (rc = dev_alloc(c, (void**)&c->rope,
                        (size_t)c->max_seq * d * sizeof(int16_t))) ||
        (rc = dev_alloc(c, (void**)&c->exp8, 2056 * sizeof(int16_t))) ||
        (rc = dev_alloc(c, (void**)&c->silu8, 2056 * sizeof(uint32_t))) ||
        (rc = dev_alloc(c, (void**)&c->exp14, 2056 * sizeof(int16_t))))
        return cleanup(rc);
    {
        // aux1 RoPE table exactly as initialize_persistent_auxiliary_data
        // (host/host_qwen_8x64.cpp:2159-2189): [cos d/2 | sin d/2] per pos.
        std::vector<int16_t> rope((size_t)c->max_seq * d);
        std::vector<double> inv_freq(d / 2);
        for (uint32_t i = 0; i < d / 2; i++)
            inv_freq[i] = 1.0 / std::pow(s.rope_theta, double(2 * i) / d);
        for (uint32_t p = 0; p < c->max_seq; p++)
            for (uint32_t i = 0; i < d / 2; i++) {
                const double angle = p * inv_freq[i];
                rope[(size_t)p * d + i] = quantize_fix16(std::cos(angle));
                rope[(size_t)p * d + d / 2 + i] = quantize_fix16(std::sin(angle));
            }
        if (hipMemcpy(c->rope, rope.data(), rope.size() * 2, hipMemcpyHostToDevice))
            return cleanup(fail(LLM_E_HIP, "rope upload"));
        int16_t e8[2049], e14[2049];
        build_exp_tables(e8, e14);
        // the SiLU epilogues' reciprocal recip(256 + e), formed here by the
        // same Newton steps instead of per output on the device
        uint32_t s8[2049];
        for (int i = 0; i < 2049; i++)
            s8[i] = (uint32_t)(uint16_t)e8[i] | (uint32_t)(uint16_t)fx_recip(256 + e8[i]) << 16;
        if (hipMemcpy(c->exp8, e8, sizeof(e8), hipMemcpyHostToDevice) ||
            hipMemcpy(c->silu8, s8, sizeof(s8), hipMemcpyHostToDevice) ||
            hipMemcpy(c->exp14, e14, sizeof(e14), hipMemcpyHostToDevice))
            return cleanup(fail(LLM_E_HIP, "exp table upload"));
    }
    // KV cache: pages of 64 positions per (layer, kv head); tile t of
    // (layer, head) is page (layer * Hkv + head) * tiles + t.
    const size_t pages = (size_t)c->L * c->Hkv * c->tiles;
    if ((rc = dev_alloc(c, (void**)&c->kcache, pages * llm::kTile * d * 2)) ||
        (rc = dev_alloc(c, (void**)&c->vcache, pages * llm::kTile * d * 2)))
        return cleanup(rc);
    // hidden pairs and scratch
    c->pairs.resize(num_pairs);
    for (auto& p : c->pairs)
        if ((rc = dev_alloc(c, (void**)&p, (size_t)8 * c->Hp * 2)))
            return cleanup(rc);
    const size_t rht = (size_t)8 * c->Hkv * c->tiles * c->G;  // rows*heads*tiles*group
    c->counter_bytes = std::max(llm::counter_words(c->Hq, c->tiles), (size_t)8 * c->Hkv) * 4;
    c->rht_words = rht;
    c->exported.assign(num_pairs, 0);
    if ((rc = dev_alloc(c, (void**)&c->xn_attn, (size_t)8 * c->Hp * 2)) ||
        (rc = dev_alloc(c, (void**)&c->xn_final, (size_t)8 * c->Hp * 2)) ||
        (rc = dev_alloc(c, (void**)&c->xn_ffn, (size_t)8 * c->Hp * 2)) ||
        (rc = dev_alloc(c, (void**)&c->qkv, (size_t)8 * c->Nqkv * 2)) ||
        (rc = dev_alloc(c, (void**)&c->attn, (size_t)8 * c->Hp * 2)) ||
        (rc = dev_alloc(c, (void**)&c->act, (size_t)8 * c->Ip * 2)) ||
        (rc = dev_alloc(c, (void**)&c->s_scores, rht * llm::kTile * 2)) ||
        (rc = dev_alloc(c, (void**)&c->s_tmax, rht * 2)) ||
        (rc = dev_alloc(c, (void**)&c->s_tsum, rht * 4)) ||
        (rc = dev_alloc(c, (void**)&c->s_tval, rht * d * 2)) ||
        (rc = dev_alloc(c, (void**)&c->counters, c->counter_bytes)) ||
        (rc = dev_alloc(c, (void**)&c->s_tmax32, rht * 4)) ||
        (rc = dev_alloc(c, (void**)&c->s_gmax32, rht * 4)) ||
        (rc = dev_alloc(c, (void**)&c->s_gsum64, rht * 8)) ||

        (rc = dev_alloc(c, (void**)&c->sync, (size_t)llm::kSyncWords * 4)))
        return cleanup(rc);
    if (hipHostMalloc((void**)&c->host_abort, 64, hipHostMallocDefault) != hipSuccess)
        return cleanup(fail(LLM_E_NOMEM, "hipHostMalloc failed"));
    *c->host_abort = 0;
    c->io_flag = c->host_abort + 8;  // a word of the same 64 bytes
    *c->io_flag = 0;
    if ((rc = dev_alloc(c, (void**)&c->io_count, 256)) || (rc = io_buffers(c, port_elems(c))) ||
        (rc = ensure_keys_host(c)))
        return cleanup(rc);
    if (const char* e = std::getenv("LLM_ACCEL_FUSED")) c->fused = std::strcmp(e, "0") != 0;
    if (const char* e = std::getenv("LLM_ACCEL_PROMPT"))
        c->prompt_path = std::strcmp(e, "0") != 0;
    if (const char* e = std::getenv("LLM_ACCEL_PROMPT_BYTES"))
        c->prompt_bytes = (size_t)std::strtoull(e, nullptr, 10);
    if (const char* e = std::getenv("LLM_ACCEL_GQA")) c->gqa = std::strcmp(e, "0") != 0;
    if (const char* e = std::getenv("LLM_ACCEL_TILE_FUSED"))
        c->tile_fused = std::strcmp(e, "0") != 0;
    if (const char* e = std::getenv("LLM_ACCEL_GQA_MIN_TILES"))
        c->gqa_min_tiles = c->gqa_min_tiles_block = (uint32_t)std::strtoul(e, nullptr, 10);
    if (const char* e = std::getenv("LLM_ACCEL_GQA_FUSED"))
        c->gqa_fused = std::strcmp(e, "0") != 0;
    if (const char* e = std::getenv("LLM_ACCEL_GQA_SCAN_FUSED"))
        c->gqa_scan_fused = std::strcmp(e, "0") != 0;
    if (const char* e = std::getenv("LLM_ACCEL_COOP")) c->coop = std::strcmp(e, "1") == 0;
    // the GQA path's epoch before the first launch (tests start it just
    // below kGqaEpochMax so that it wraps within a few launches)
    if (const char* e = std::getenv("LLM_ACCEL_GQA_EPOCH_START"))
        c->gqa_epoch = std::min<uint32_t>((uint32_t)std::strtoul(e, nullptr, 0), llm::kGqaEpochMax);
    if (hipDeviceGetAttribute(&c->cus, hipDeviceAttributeMultiprocessorCount, c->device) !=
        hipSuccess)
        return cleanup(fail(LLM_E_HIP, "device attribute query failed"));
    c->wait_limit = llm::kWaitLimitTicks;
    if (const char* e = std::getenv("LLM_ACCEL_WAIT_LIMIT"))
        c->wait_limit = (uint32_t)std::strtoul(e, nullptr, 10);
    // Test hook: every arrival counter (and the host's copy) starts at
    // LLM_ACCEL_SYNC_START instead of 0, e.g. just below 2^32 so that the
    // counters wrap within a few launches.
    if (const char* e = std::getenv("LLM_ACCEL_SYNC_START")) {
        const uint32_t v = (uint32_t)std::strtoul(e, nullptr, 0);
        std::vector<uint32_t> init(llm::kSyncWords, 0);
        for (uint32_t l = 0; l < llm::kSyncQkvLines; l++) init[l * llm::kSyncStride] = v;
        for (uint32_t l = 0; l < llm::kSyncAttnLines; l++)
            init[llm::kSyncAttn + l * llm::kSyncStride] = v;
        if (hipMemcpy(c->sync, init.data(), init.size() * 4, hipMemcpyHostToDevice) != hipSuccess)
            return cleanup(fail(LLM_E_HIP, "counter initialisation failed"));
        std::fill(std::begin(c->sync_qkv), std::end(c->sync_qkv), v);
        c->sync_attn = v;
    }
    {
        const size_t rhc = (size_t)8 * c->Hkv * cdiv(c->tiles, c->chunk_tiles) * c->G;
        if ((rc = dev_alloc(c, (void**)&c->c_flag, rhc * 4)) ||
            (rc = dev_alloc(c, (void**)&c->c_tsum, rhc * 4)) ||
            (rc = dev_alloc(c, (void**)&c->c_sum, rhc * d * 4)))
            return cleanup(rc);
    }
    {
        // split matrix-core scratch: the largest (chunks x parts x record)
        size_t words = 0, chunks = 0;
        for (uint32_t m = 0; m < M_COUNT; m++) {
            const Matrix& mt = c->mat(0, m);
            // either kernel of the matrix-core path
            const uint32_t nm = (m == M_GATE || m == M_UP) ? 2 : 1;
            // the operator-level commands launch row ranges of a matrix,
            // whose fewer chunks may split K into more parts
            for (uint32_t n2 = 1; n2 <= mt.nc; n2++) {
                const uint32_t parts = std::max(llm::mf_split(n2, mt.kq).parts,
                                                llm::mf12_split(n2, mt.steps, nm).parts);
                words = std::max(words, (size_t)n2 * parts * llm::mf_part_words(nm));
            }
            chunks = std::max(chunks, (size_t)mt.nc);
        }
        if ((rc = dev_alloc(c, (void**)&c->mf_part, words * 4)) ||
            (rc = dev_alloc(c, (void**)&c->mf_count, chunks * 4)))
            return cleanup(rc);
        for (auto& mt : c->mats) {
            mt.ctx_part = c->mf_part;
            mt.ctx_count = c->mf_count;
        }
    }
    if (fx_recip(fx_sat16((int64_t)c->H * 256)) == 0)
        c->const_gain = fx_rmsnorm_gain(0, c->H);
    // the fused norms form gain * gamma with 24-bit multiplies (the gain is
    // 6623 raw); a gain beyond that keeps the separate norm kernel
    if (c->const_gain >= (1 << 23)) c->const_gain = 0;
    *out = c;
    return 0;
}

void llm_ctx_destroy(llm_ctx_t* c) {
    if (!c) return;
    (void)hipSetDevice(c->device);
    if (c->stream) (void)hipStreamSynchronize(c->stream);
    for (auto e : c->events) (void)hipEventDestroy(e);
    for (auto e : c->ev_pool) (void)hipEventDestroy(e);
    for (auto& t : c->pending) {
        (void)hipEventDestroy(t.a);
        (void)hipEventDestroy(t.b);
    }
    for (void* p : c->allocations) (void)hipFree(p);
    if (c->host_abort) (void)hipHostFree(c->host_abort);
    if (c->stage) (void)hipHostFree(c->stage);
    if (c->io_in) (void)hipHostFree(c->io_in);
    if (c->keys_host) (void)hipHostFree(c->keys_host);
    for (auto e : c->gen_events) (void)hipEventDestroy(e);
    if (c->stream) (void)hipStreamDestroy(c->stream);
    delete c;
}

int llm_load_projection(llm_ctx_t* c, uint32_t layer, uint32_t proj,
                        const int16_t* w) {
    if (!c || !w || layer >= c->L || proj > LLM_PROJ_DOWN)
        return fail(LLM_E_ARG, "bad projection load arguments");
    HIP_TRY(hipSetDevice(c->device));
    int rc;
    switch (proj) {
    case LLM_PROJ_Q:
        rc = upload_rows(c, c->mat(layer, M_QKV), 0, c->H, w, 0);
        break;
    case LLM_PROJ_K:
        rc = upload_rows(c, c->mat(layer, M_QKV), c->H, c->Ckv, w, 1);
        break;
    case LLM_PROJ_V:
        rc = upload_rows(c, c->mat(layer, M_QKV), c->H + c->Ckv, c->Ckv, w, 2);
        break;
    case LLM_PROJ_O:
        rc = upload_rows(c, c->mat(layer, M_O), 0, c->H, w, 0);
        break;
    case LLM_PROJ_GATE:
        rc = upload_rows(c, c->mat(layer, M_GATE), 0, c->I, w, 0);
        break;
    case LLM_PROJ_UP:
        rc = upload_rows(c, c->mat(layer, M_UP), 0, c->I, w, 0);
        break;
    default:
        rc = upload_rows(c, c->mat(layer, M_DOWN), 0, c->H, w, 0);
        break;
    }
    if (rc == 0) c->loaded[layer * 7 + proj] = true;
    return rc;
}

int llm_load_packed_shards(llm_ctx_t* c, const int16_t* const shards[16],
                           uint64_t shard_words) {
    if (!c || !shards) return fail(LLM_E_ARG, "null argument");
    for (int i = 0; i < 16; i++)
        if (!shards[i]) return fail(LLM_E_ARG, "null shard");
    // projection_spec / projection_weight_raw (host:325-376, :899-935)
    uint64_t tiles[7], base[7], layer_tiles = 0;
    uint32_t in_dims[7], out_dims[7];
    for (uint32_t p = 0; p < 7; p++) {
        in_dims[p] = p == LLM_PROJ_DOWN ? c->I : c->H;
        out_dims[p] = (p == LLM_PROJ_K || p == LLM_PROJ_V) ? c->Ckv
                    : (p == LLM_PROJ_GATE || p == LLM_PROJ_UP) ? c->I : c->H;
        tiles[p] = cdiv(out_dims[p], 16) * cdiv(in_dims[p], 16);
        base[p] = layer_tiles;
        layer_tiles += tiles[p];
    }
    if (shard_words < cdiv((uint64_t)c->L * layer_tiles, 2))
        return fail(LLM_E_ARG, "shard_words too small for the shape");
    std::vector<int16_t> w;
    for (uint32_t l = 0; l < c->L; l++) {
        for (uint32_t p = 0; p < 7; p++) {
            const uint32_t N = out_dims[p], K = in_dims[p];
            const uint64_t in_tiles = cdiv(K, 16);
            w.assign((size_t)N * K, 0);
            for (uint32_t n = 0; n < N; n++)
                for (uint32_t k = 0; k < K; k++) {
                    const uint64_t tile = (uint64_t)l * layer_tiles + base[p] +
                                          (uint64_t)(n / 16) * in_tiles + k / 16;
                    const uint32_t lane_in_tile = (n % 16) * 16 + k % 16;
                    const uint32_t shard = (uint32_t)(tile & 1) * 8 + lane_in_tile / 32;
                    w[(size_t)n * K + k] =
                        shards[shard][(tile >> 1) * 32 + lane_in_tile % 32];
                }
            int rc = llm_load_projection(c, l, p, w.data());
            if (rc) return rc;
        }
    }
    return 0;
}

// Bytes of the file at `path`, or -1 when it cannot be opened.
static long long file_bytes(const std::string& path) {
    FILE* f = std::fopen(path.c_str(), "rb");
    if (!f) return -1;
    long long n = -1;
    if (std::fseek(f, 0, SEEK_END) == 0) n = std::ftell(f);
    std::fclose(f);
    return n;
}

// The whole file into dst, which must be exactly `bytes` long
// (load_exact_file, host/host_qwen_8x64.cpp:736-763).
static int load_exact(const std::string& path, void* dst, size_t bytes, const char* what) {
    const long long actual = file_bytes(path);
    if (actual != (long long)bytes)
        return fail(LLM_E_ARG, std::string(what) + " size mismatch: " + path +
                                   " expected=" + std::to_string(bytes) +
                                   " actual=" + std::to_string(actual < 0 ? 0 : actual));
    FILE* f = std::fopen(path.c_str(), "rb");
    if (!f) return fail(LLM_E_ARG, "failed to read " + path);
    const size_t got = std::fread(dst, 1, bytes, f);
    std::fclose(f);
    if (got != bytes) return fail(LLM_E_ARG, "failed to read " + path);
    return 0;
}

int llm_load_checkpoint_dir(llm_ctx_t* c, const char* dir, uint32_t flags,
                            int16_t* embedding) {
    if (!c || !dir) return fail(LLM_E_ARG, "null argument");
    if (flags & ~(uint32_t)(LLM_CKPT_TIE_EMBEDDINGS | LLM_CKPT_REQUIRE_LM_HEAD))
        return fail(LLM_E_ARG, "unknown checkpoint flags");
    const std::string d(dir);
    const size_t vocab = c->s.vocab_size, emb_vals = vocab * c->H;
    const size_t norm_vals = (size_t)(2 * c->L + 1) * c->H;
    // weight_shard_words (host/host_qwen_8x64.cpp:165-187): 16x16 tiles of
    // every projection of every layer, two tiles per 64-byte word
    uint64_t layer_tiles = 0;
    for (uint32_t p = 0; p < 7; p++) {
        const uint32_t K = p == LLM_PROJ_DOWN ? c->I : c->H;
        const uint32_t N = (p == LLM_PROJ_K || p == LLM_PROJ_V) ? c->Ckv
                         : (p == LLM_PROJ_GATE || p == LLM_PROJ_UP) ? c->I : c->H;
        layer_tiles += cdiv(N, 16) * cdiv(K, 16);
    }
    const uint64_t shard_words = cdiv((uint64_t)c->L * layer_tiles, 2);
    const bool tie = flags & LLM_CKPT_TIE_EMBEDDINGS;
    // every size first, in the reference's order (embedding, norms, shards,
    // LM head), so that a bad directory loads nothing
    std::vector<std::string> shard_paths(16);
    for (int i = 0; i < 16; i++) {
        char name[64];
        std::snprintf(name, sizeof name, "/layer_weights_shard%02d.fix16.bin", i);
        shard_paths[i] = d + name;
    }
    const std::string emb_path = d + "/token_embedding.fix16.bin";
    const std::string norm_path = d + "/norm_weights.fix16.bin";
    const std::string lm_path = d + "/lm_head.fix16.bin";
    auto check = [&](const std::string& path, size_t bytes, const char* what) {
        const long long actual = file_bytes(path);
        if (actual == (long long)bytes) return 0;
        return fail(LLM_E_ARG, std::string(what) + " size mismatch: " + path +
                                   " expected=" + std::to_string(bytes) +
                                   " actual=" + std::to_string(actual < 0 ? 0 : actual));
    };
    int rc;
    if ((rc = check(emb_path, emb_vals * 2, "embedding"))) return rc;
    if ((rc = check(norm_path, norm_vals * 2, "norm weights"))) return rc;
    for (int i = 0; i < 16; i++)
        if ((rc = check(shard_paths[i], shard_words * 64, "weight shard"))) return rc;
    const bool have_lm = !tie && file_bytes(lm_path) >= 0;
    if (have_lm && (rc = check(lm_path, emb_vals * 2, "LM head"))) return rc;
    if (!tie && !have_lm && (flags & LLM_CKPT_REQUIRE_LM_HEAD))
        return fail(LLM_E_ARG, "generate mode requires lm_head.fix16.bin or tied embeddings");
    HIP_TRY(hipSetDevice(c->device));
    {
        std::vector<int16_t> norms(norm_vals);
        if ((rc = load_exact(norm_path, norms.data(), norm_vals * 2, "norm weights")) ||
            (rc = llm_load_norms(c, norms.data())))
            return rc;
    }
    {
        std::vector<std::vector<int16_t>> shards(16);
        const int16_t* ptrs[16];
        for (int i = 0; i < 16; i++) {
            shards[i].resize((size_t)shard_words * 32);
            if ((rc = load_exact(shard_paths[i], shards[i].data(), shard_words * 64,
                                 "weight shard")))
                return rc;
            ptrs[i] = shards[i].data();
        }
        if ((rc = llm_load_packed_shards(c, ptrs, shard_words))) return rc;
    }
    std::vector<int16_t> own;
    int16_t* emb = embedding;
    if (!emb && tie) {
        own.resize(emb_vals);
        emb = own.data();
    }
    if (emb && (rc = load_exact(emb_path, emb, emb_vals * 2, "embedding"))) return rc;
    if (tie) return llm_load_lm_head(c, emb, (uint32_t)vocab);
    if (have_lm) {
        std::vector<int16_t> lm(emb_vals);
        if ((rc = load_exact(lm_path, lm.data(), emb_vals * 2, "LM head"))) return rc;
        return llm_load_lm_head(c, lm.data(), (uint32_t)vocab);
    }
    return 0;
}

int llm_load_norms(llm_ctx_t* c, const int16_t* norms) {
    if (!c || !norms) return fail(LLM_E_ARG, "null argument");
    HIP_TRY(hipSetDevice(c->device));
    HIP_TRY(hipMemcpy(c->norms, norms, (size_t)(2 * c->L + 1) * c->H * 2,
                      hipMemcpyHostToDevice));
    c->norms_loaded = true;
    return 0;
}

int llm_hidden_upload(llm_ctx_t* c, uint32_t pair, const int16_t* rows,
                      uint32_t n) {
    if (!c || !rows || pair >= c->pairs.size() || n > 8)
        return fail(LLM_E_ARG, "bad hidden upload arguments");
    HIP_TRY(hipSetDevice(c->device));
    invalidate_pair(c, (int)pair);
    c->n_h2d_rows++;
    // a pair whose address was handed out may be read on another stream
    return rows_in(c, rows, c->pairs[pair], c->Hp, c->H, n, c->exported[pair]);
}

int llm_hidden_download(llm_ctx_t* c, uint32_t pair, int16_t* rows,
                        uint32_t n) {
    if (!c || !rows || pair >= c->pairs.size() || n > 8)
        return fail(LLM_E_ARG, "bad hidden download arguments");
    HIP_TRY(hipSetDevice(c->device));
    c->n_d2h_rows++;
    return rows_out(c, c->pairs[pair], c->Hp, rows, c->H, n);
}

int llm_hidden_upload_ports(llm_ctx_t* c, uint32_t pair, const int16_t* port0,
                            const int16_t* port1, uint32_t n,
                            uint32_t stride_words) {
    if (!c || !port0 || (n > 4 && !port1) || n > 8 ||
        (size_t)stride_words * 32 < c->H)
        return fail(LLM_E_ARG, "bad port upload arguments");
    std::vector<int16_t> rows((size_t)n * c->H);
    for (uint32_t t = 0; t < n; t++) {
        const int16_t* src = (t < 4 ? port0 : port1) + (size_t)(t % 4) * stride_words * 32;
        std::memcpy(&rows[(size_t)t * c->H], src, (size_t)c->H * 2);
    }
    return llm_hidden_upload(c, pair, rows.data(), n);
}

int llm_hidden_download_ports(llm_ctx_t* c, uint32_t pair, int16_t* port0,
                              int16_t* port1, uint32_t n,
                              uint32_t stride_words) {
    if (!c || !port0 || (n > 4 && !port1) || n > 8 ||
        (size_t)stride_words * 32 < c->H)
        return fail(LLM_E_ARG, "bad port download arguments");
    std::vector<int16_t> rows((size_t)n * c->H);
    int rc = llm_hidden_download(c, pair, rows.data(), n);
    if (rc) return rc;
    for (uint32_t t = 0; t < n; t++) {
        int16_t* dst = (t < 4 ? port0 : port1) + (size_t)(t % 4) * stride_words * 32;
        std::memcpy(dst, &rows[(size_t)t * c->H], (size_t)c->H * 2);
    }
    return 0;
}

int llm_task(llm_ctx_t* c, uint32_t op, uint32_t layer, uint32_t token_count,
             uint32_t position, uint32_t tile_len, uint32_t in_pair,
             uint32_t out_pair, llm_status_t* status) {
    llm_status_t local;
    llm_status_t* st = status ? status : &local;
    std::memset(st, 0, sizeof(*st));
    if (!c) return fail(LLM_E_ARG, "null context");
    if (in_pair >= c->pairs.size() || out_pair >= c->pairs.size())
        return fail(LLM_E_ARG, "bad pair id");
    // control_cache_8x64_dual_core (kernel/control_cache_8x64.cpp:5882-5957)
    if (tile_len != 0) token_count &= 0xffffu;
    st->op = LLM_OP_NOP;
    st->token_count = token_count;
    st->last_task = 1;
    auto reject = [&](uint32_t code) {
        st->code = code;
        return (int)code;
    };
    if (token_count > 8) return reject(LLM_STATUS_BAD_TOKEN_COUNT);
    st->op = op;
    if (op > LLM_OP_FINAL_NORM) return reject(LLM_STATUS_BAD_OPERATOR);
    if (op == LLM_OP_NOP) return LLM_STATUS_OK;
    if (layer >= c->L) return reject(LLM_STATUS_BAD_LAYER);
    c->busy = llm_ctx::WORK;
    const int ip = (int)in_pair, opr = (int)out_pair;
    if (hipSetDevice(c->device) != hipSuccess)
        return fail(LLM_E_HIP, "hipSetDevice failed");
    if (op == LLM_OP_FINAL_NORM) {
        const int16_t* in = c->pairs[in_pair];
        int16_t* out = c->pairs[out_pair];
        if (token_count == 0) return reject(LLM_STATUS_BAD_TOKEN_COUNT);
        if (!c->norms_loaded) return fail(LLM_E_STATE, "norm table not loaded");
        const auto& fc = c->final_cache;
        if (fc.pair == ip && fc.src == opr && fc.rows == token_count &&
            !c->exported[opr]) {
            // xn_final already holds what the norm would leave in out_pair
            std::swap(c->pairs[opr], c->xn_final);
        } else {
            TimedScope ts(c, LLM_K_RMSNORM);
            HIP_TRY(llm::launch_rmsnorm(in, c->Hp,
                                        c->norms + (size_t)(2 * c->L) * c->H,
                                        c->H, out, c->Hp, token_count,
                                        c->const_gain, c->stream));
        }
        invalidate_pair(c, opr);
        fill_counters(c, op, token_count, position, st);
        return LLM_STATUS_OK;
    }
    if (op == LLM_OP_DECODER_LAYER || op == LLM_OP_ATTENTION_SUBLAYER ||
        op == LLM_OP_FFN_SUBLAYER) {
        if (token_count == 0) return reject(LLM_STATUS_BAD_TOKEN_COUNT);
        if (position >= c->max_seq || position + token_count > c->max_seq)
            return reject(LLM_STATUS_BAD_POSITION);
        int rc = check_layer_loaded(c, layer, op != LLM_OP_FFN_SUBLAYER,
                                    op != LLM_OP_ATTENTION_SUBLAYER);
        if (rc) return rc;
        if (op == LLM_OP_ATTENTION_SUBLAYER) {
            rc = enqueue_attention_sublayer(c, layer, token_count, position, ip, opr);
        } else if (op == LLM_OP_FFN_SUBLAYER) {
            rc = enqueue_ffn_sublayer(c, layer, token_count, ip, opr);
        } else {
            rc = enqueue_attention_sublayer(c, layer, token_count, position, ip, opr);
            if (rc == 0) rc = enqueue_ffn_sublayer(c, layer, token_count, opr, opr);
        }
        if (rc) return rc;
        fill_counters(c, op, token_count, position, st);
        return LLM_STATUS_OK;
    }
    // The resident-layer image carries no per-operator scheduler
    // (kernel/control_cache_8x64.cpp:6483-6494).
    return reject(LLM_STATUS_BAD_OPERATOR);
}

}  // extern "C"

namespace {

// ---------------------------------------------------------------------
// Operator-level commands: the per-operator scheduler of the controller's
// full image (kernel/control_cache_8x64.cpp:6497-7500), driven by the
// reference host's run_feature / run_attention /
// run_prefill_attention_block (host/host_qwen_8x64.cpp:1088-1133,
// :1556-1675).
// ---------------------------------------------------------------------

int ensure_ports(llm_ctx* c) {
    if (c->ports_ready) return 0;
    const size_t n = port_elems(c);
    for (int i = 0; i < 3; i++)
        if (!c->ports[i])
            if (int rc = dev_alloc(c, (void**)&c->ports[i], n * 2)) return rc;
    if (!c->op_stage)
        if (int rc = dev_alloc(c, (void**)&c->op_stage,
                               (size_t)8 * std::max(c->Hp, c->Ip) * 2))
            return rc;
    if (!c->op_tsum)
        if (int rc = dev_alloc(c, (void**)&c->op_tsum, c->rht_words * 4)) return rc;
    c->port_n = n;
    c->ports_ready = true;
    return 0;
}

// The controller's status counters for an operator-level command
// (kernel/control_cache_8x64.cpp:6715-6723, :6825-6832, :7110-7113,
// :7163-7169, :7251-7258, :7339-7342, :7489-7495): two 8x64 cores, waves
// of 128 outputs, 32 packets per MM task, 16-lane vector packets, PV waves
// of 64 head elements.
void fill_op_counters(const llm_ctx* c, uint32_t op, uint32_t T, uint32_t pos,
                      uint32_t tile_len, llm_status_t* st) {
    const uint32_t pv_waves = (uint32_t)cdiv(c->d, 64);
    auto mm = [&](uint32_t waves, uint32_t tasks) {
        st->output_waves = waves;
        st->mm_tasks = tasks;
        st->completed_packets = tasks * 32;
    };
    if (op >= 1 && op <= 7) {
        const uint32_t out_dim = (op == 2 || op == 3) ? c->Ckv
                               : (op == 5 || op == 6) ? c->I : c->H;
        const uint32_t w = (uint32_t)cdiv(out_dim, 128);
        mm(w, 2 * w);
    } else if (op >= 8 && op <= 10) {
        const uint32_t blocks = (uint32_t)cdiv(op == 9 ? c->I : c->H, 16);
        const uint32_t c0 = std::min(T, 4u), c1 = T > 4 ? T - 4 : 0;
        st->vector_tasks = (c0 > 0) + (c1 > 0);
        st->completed_packets = (c0 + c1) * blocks;
    } else if (op == 11) {
        mm(1, 2);
    } else if (op == 12) {
        mm(pv_waves, 2 * pv_waves);
    } else if (op == 13) {
        st->vector_tasks = 2;
        st->completed_packets = 2 * c->G * (uint32_t)cdiv(tile_len, 16);
    } else if (op == 14 || op == 15) {
        mm(pv_waves, 2 * (uint32_t)cdiv(pos + 1, 64) * (1 + pv_waves));
    } else if (op == 17) {
        mm(pv_waves, 2 * (uint32_t)cdiv(pos + T, 64) * c->G * (1 + pv_waves));
    }
}

// One projection (0 = Q .. 6 = down) of `T` rows without epilogue.  Q, K
// and V are row ranges of the stored Q | K | V matrix.  The rows are
// staged into 8 rows padded to whole k-steps: the projection kernels read
// whole k-steps, and the matrix-core kernel all 8 rows (rows past T only
// reach outputs that are not stored).
int enqueue_op_projection(llm_ctx* c, uint32_t layer, uint32_t proj, uint32_t T,
                          const int16_t* in, int16_t* out) {
    static const int mat_of[7] = {M_QKV, M_QKV, M_QKV, M_O, M_GATE, M_UP, M_DOWN};
    const Matrix& m = c->mat(layer, mat_of[proj]);
    const uint32_t row0 = proj == 1 ? c->H : proj == 2 ? c->H + c->Ckv : 0;
    const uint32_t n = proj == 0 ? c->H : (proj <= 2 ? c->Ckv : m.n);
    if (T == 0) return 0;
    // the kernels read whole k-steps and, for 3 rows on, all 8 rows: the
    // context's own port holds those where its tight rows are whole steps;
    // otherwise the rows are staged
    const bool direct = in == c->ports[LLM_PORT_IN] && m.k == m.k_pad &&
                        (out + (size_t)T * n <= in || out >= in + c->port_n);
    if (direct) {
    } else if (m.k % 8 == 0 && (uintptr_t)in % 16 == 0)  // what the copy kernel's loads need
        HIP_TRY(llm::launch_io_rows(in, m.k, c->op_stage, m.k_pad, m.k, T, nullptr, nullptr, 0,
                                    c->stream));
    else
        HIP_TRY(hipMemcpy2DAsync(c->op_stage, (size_t)m.k_pad * 2, in, (size_t)m.k * 2,
                                 (size_t)m.k * 2, T, hipMemcpyDeviceToDevice, c->stream));
    llm::ProjArgs a{};
    a.w0 = m.d ? m.d + (size_t)row0 * m.k_pad : nullptr;
    a.steps = m.steps;
    a.x = direct ? in : c->op_stage;
    a.ldx = m.k_pad;
    a.out = out;
    a.ldo = n;
    a.n = n;
    a.rows = T;
    if (m.p12_ok) a.p0 = m.p12 + (size_t)(row0 / llm::kBlockRows) * m.steps * llm::kP12Step;
    // the matrix-core records and sums cover 16 outputs each (matrices held
    // in 12 bits only have Q, K and V on 16-row boundaries)
    if (row0 % llm::kMfRows == 0) {
        set_mf(c, a, m);
        if (a.mf0) a.mf0 += (size_t)(row0 / llm::kMfRows) * m.kq * llm::kMfRecord;
        a.ms0 += (size_t)2 * row0;
        a.nc = (uint32_t)cdiv(n, llm::kMfRows);
    }
    if (m.corr_any) a.corr0 = m.corr + (size_t)row0 * llm::kCorrSlots;
    HIP_TRY(llm::launch_proj(a, llm::EPI_STORE, m.L, (uint32_t)cdiv(n, 4), c->stream));
    return 0;
}

}  // namespace

extern "C" {

int llm_port(llm_ctx_t* c, uint32_t port, void** dev, size_t* elems) {
    if (!c || port > LLM_PORT_OUT) return fail(LLM_E_ARG, "bad port arguments");
    HIP_TRY(hipSetDevice(c->device));
    if (int rc = ensure_ports(c)) return rc;
    if (dev) {
        if (int rc = finish_copies(c)) return rc;
        *dev = c->ports[port];
        c->port_out = true;  // from here on port writes are complete on return
    }
    if (elems) *elems = c->port_n;
    return 0;
}

int llm_port_write(llm_ctx_t* c, uint32_t port, const int16_t* host, size_t elems) {
    if (!c || port > LLM_PORT_OUT || (!host && elems)) return fail(LLM_E_ARG, "bad port arguments");
    HIP_TRY(hipSetDevice(c->device));
    if (int rc = ensure_ports(c)) return rc;
    if (elems > c->port_n) return fail(LLM_E_ARG, "port write exceeds the port");
    return rows_in(c, host, c->ports[port], (uint32_t)elems, (uint32_t)elems, 1, c->port_out);
}

int llm_port_read(llm_ctx_t* c, uint32_t port, int16_t* host, size_t elems) {
    if (!c || port > LLM_PORT_OUT || (!host && elems)) return fail(LLM_E_ARG, "bad port arguments");
    HIP_TRY(hipSetDevice(c->device));
    if (int rc = ensure_ports(c)) return rc;
    if (elems > c->port_n) return fail(LLM_E_ARG, "port read exceeds the port");
    return rows_out(c, c->ports[port], (uint32_t)elems, host, (uint32_t)elems, 1);
}

int llm_op(llm_ctx_t* c, uint32_t op, uint32_t layer, uint32_t token_count,
           uint32_t position, uint32_t tile_len, const int16_t* in,
           const int16_t* aux, int16_t* out, llm_status_t* status) {
    llm_status_t local;
    llm_status_t* st = status ? status : &local;
    std::memset(st, 0, sizeof(*st));
    if (!c) return fail(LLM_E_ARG, "null context");
    // argument decoding and the checks shared by every operator
    // (kernel/control_cache_8x64.cpp:5882-5957)
    if (tile_len != 0) token_count &= 0xffffu;
    st->op = LLM_OP_NOP;
    st->token_count = token_count;
    st->last_task = 1;
    auto reject = [&](uint32_t code) {
        st->code = code;
        return (int)code;
    };
    if (token_count > 8) return reject(LLM_STATUS_BAD_TOKEN_COUNT);
    st->op = op;
    if (op > LLM_OP_FINAL_NORM) return reject(LLM_STATUS_BAD_OPERATOR);
    if (op == LLM_OP_NOP) return LLM_STATUS_OK;
    if (op == LLM_OP_DECODER_LAYER || op >= LLM_OP_ATTENTION_SUBLAYER) {
        st->op = LLM_OP_NOP;
        return fail(LLM_E_ARG, "operator " + std::to_string(op) +
                                   " is a resident-layer task: use llm_task");
    }
    if (layer >= c->L) return reject(LLM_STATUS_BAD_LAYER);
    const uint32_t T = token_count, G = c->G, D = c->d;
    // per-operator checks in the controller's order (:6497-6531,
    // :6729-6750, :7018-7027)
    if (op == LLM_OP_ATTN_PREFILL_BLOCK) {
        if (T == 0) return reject(LLM_STATUS_BAD_TOKEN_COUNT);
        if (position >= c->max_seq || position + T > c->max_seq)
            return reject(LLM_STATUS_BAD_POSITION);
    } else if (op == LLM_OP_ATTN_FLASH || op == LLM_OP_DECODE_SMOKE) {
        if (T != G) return reject(LLM_STATUS_BAD_TOKEN_COUNT);
        if (position >= c->max_seq) return reject(LLM_STATUS_BAD_POSITION);
        if (tile_len > 64) return reject(LLM_STATUS_BAD_TILE_LENGTH);
    } else if (op >= LLM_OP_ATTN_QK && op <= LLM_OP_SOFTMAX) {
        if (tile_len == 0 || tile_len > 64) return reject(LLM_STATUS_BAD_TILE_LENGTH);
    } else if (op <= LLM_OP_FFN_DOWN && tile_len != 0) {
        // run_mm_wave_profile's encoding (host/host_qwen_8x64.cpp:1495-1554)
        st->op = LLM_OP_NOP;
        return fail(LLM_E_ARG, "the MM wave-profile encoding (tile_len != 0 on a "
                               "projection) selects FPGA cores and stream stages; "
                               "it is not supported");
    }
    HIP_TRY(hipSetDevice(c->device));
    if (int rc = ensure_ports(c)) return rc;
    if (!in) in = c->ports[LLM_PORT_IN];
    if (!aux) aux = c->ports[LLM_PORT_AUX];
    if (!out) out = c->ports[LLM_PORT_OUT];
    c->busy = llm_ctx::WORK;
    hipStream_t s = c->stream;
    const size_t layer_off = (size_t)layer * c->Hkv * c->tiles * llm::kTile * D;
    if (op <= LLM_OP_FFN_DOWN) {
        if (!c->loaded[layer * 7 + op - 1])
            return fail(LLM_E_STATE, "layer " + std::to_string(layer) + " projection " +
                                         std::to_string(op - 1) + " not loaded");
        if (int rc = enqueue_op_projection(c, layer, op - 1, T, in, out)) return rc;
    } else if (op == LLM_OP_RMSNORM) {
        if (T) HIP_TRY(llm::launch_rmsnorm(in, c->H, aux, c->H, out, c->H, T,
                                           c->const_gain, s));
    } else if (op == LLM_OP_SILU_MUL) {
        HIP_TRY(llm::launch_op_silu_mul(in, aux, T * c->I, c->exp8, out, s));
    } else if (op == LLM_OP_RESIDUAL_ADD) {
        HIP_TRY(llm::launch_op_residual(in, aux, T * c->H, out, s));
    } else if (op == LLM_OP_ATTN_QK) {
        HIP_TRY(llm::launch_op_qk(in, aux, c->Hkv, G, D, tile_len, c->qk_scale, out, s));
    } else if (op == LLM_OP_ATTN_PV) {
        HIP_TRY(llm::launch_op_pv(in, aux, c->Hkv, G, D, tile_len, out, s));
    } else if (op == LLM_OP_SOFTMAX) {
        HIP_TRY(llm::launch_op_softmax(in, c->Hkv * G, tile_len, c->exp8, out, s));
    } else {
        const bool block = op == LLM_OP_ATTN_PREFILL_BLOCK;
        if (op == LLM_OP_DECODE_SMOKE)  // aux = K rows, then V rows, of every KV head
            HIP_TRY(llm::launch_op_kv_append(c->kcache + layer_off, c->vcache + layer_off,
                                             c->tiles, c->Hkv, D, position, aux,
                                             aux + (size_t)c->Hkv * D, s));
        llm::OpFlashArgs fa{};
        fa.q = in;
        fa.kcache = c->kcache + layer_off;
        fa.vcache = c->vcache + layer_off;
        fa.tiles = c->tiles;
        fa.kv_heads = c->Hkv;
        fa.tokens = block ? T : 1;
        fa.group = G;
        fa.head_dim = D;
        fa.pos0 = position;
        fa.qk_scale = c->qk_scale;
        fa.exp8 = c->exp8;
        fa.exp14 = c->exp14;
        fa.legacy = block ? 0 : 1;
        fa.out = out;
        fa.s_scores = c->s_scores;
        fa.s_tmax = c->s_tmax;
        fa.s_tsum = c->op_tsum;
        fa.s_tval = c->s_tval;
        HIP_TRY(llm::launch_op_flash(fa, s));
    }
    fill_op_counters(c, op, T, position, tile_len, st);
    return LLM_STATUS_OK;
}

}  // extern "C"

namespace {

// Cache pages hold 64 positions of one (layer, KV head): K as rows [64][d]
// with every row's elements in the bank-paired order [0 4 1 5 2 6 3 7] of
// each group of 8, V transposed [d][64] with positions in that order.
uint32_t paired_index(uint32_t e) {
    static const uint32_t slot[8] = {0, 2, 4, 6, 1, 3, 5, 7};
    return (e & ~7u) | slot[e & 7u];
}

// Copy positions [pos0, pos0 + n) between host rows [n][d] and the pages;
// to_device selects the direction.  Works page by page through a host
// staging copy of each touched page.
int kv_transfer(llm_ctx* c, uint32_t layer, uint32_t h, uint32_t pos0,
                uint32_t n, int16_t* k, int16_t* v, bool to_device) {
    const uint32_t d = c->d;
    std::vector<int16_t> page((size_t)64 * d);
    for (uint32_t p = pos0; p < pos0 + n;) {
        const uint32_t tile = p / 64, slot0 = p % 64;
        const uint32_t cnt = std::min(64 - slot0, pos0 + n - p);
        const size_t pg = ((size_t)layer * c->Hkv + h) * c->tiles + tile;
        for (int which = 0; which < 2; which++) {
            int16_t* rows = which == 0 ? k : v;
            if (!rows) continue;
            int16_t* dev = (which == 0 ? c->kcache : c->vcache) + pg * 64 * d;
            HIP_TRY(hipMemcpy(page.data(), dev, page.size() * 2, hipMemcpyDeviceToHost));
            for (uint32_t s = slot0; s < slot0 + cnt; s++) {
                int16_t* row = rows + (size_t)(tile * 64 + s - pos0) * d;
                for (uint32_t e = 0; e < d; e++) {
                    int16_t& cell = which == 0 ? page[(size_t)s * d + paired_index(e)]
                                               : page[(size_t)e * 64 + paired_index(s)];
                    if (to_device) cell = row[e];
                    else row[e] = cell;
                }
            }
            if (to_device)
                HIP_TRY(hipMemcpy(dev, page.data(), page.size() * 2,
                                  hipMemcpyHostToDevice));
        }
        p += cnt;
    }
    return 0;
}

}  // namespace

extern "C" {

int llm_kv_read(llm_ctx_t* c, uint32_t layer, uint32_t h, uint32_t pos0,
                uint32_t n, int16_t* k, int16_t* v) {
    if (!c || layer >= c->L || h >= c->Hkv || pos0 + n > c->max_seq)
        return fail(LLM_E_ARG, "bad KV read arguments");
    HIP_TRY(hipSetDevice(c->device));
    SYNC_TRY(c);
    c->n_kv_moves++;
    return kv_transfer(c, layer, h, pos0, n, k, v, false);
}

int llm_kv_write(llm_ctx_t* c, uint32_t layer, uint32_t h, uint32_t pos0,
                 uint32_t n, const int16_t* k, const int16_t* v) {
    if (!c || layer >= c->L || h >= c->Hkv || pos0 + n > c->max_seq)
        return fail(LLM_E_ARG, "bad KV write arguments");
    HIP_TRY(hipSetDevice(c->device));
    SYNC_TRY(c);
    c->n_kv_moves++;
    return kv_transfer(c, layer, h, pos0, n, const_cast<int16_t*>(k),
                       const_cast<int16_t*>(v), true);
}

int llm_kv_clear(llm_ctx_t* c) {
    if (!c) return fail(LLM_E_ARG, "null context");
    c->busy = llm_ctx::WORK;
    HIP_TRY(hipSetDevice(c->device));
    const size_t bytes = (size_t)c->L * c->Hkv * c->tiles * 64 * c->d * 2;
    HIP_TRY(hipMemsetAsync(c->kcache, 0, bytes, c->stream));
    HIP_TRY(hipMemsetAsync(c->vcache, 0, bytes, c->stream));
    SYNC_TRY(c);
    return 0;
}

void* llm_pair_device_ptr(llm_ctx_t* c, uint32_t pair) {
    if (!c || pair >= c->pairs.size()) return nullptr;
    if (hipSetDevice(c->device) != hipSuccess) return nullptr;
    if (finish_copies(c) != 0) return nullptr;
    invalidate_pair(c, (int)pair);  // the caller may write through it
    c->exported[pair] = 1;          // and keeps using this address
    return c->pairs[pair];
}

void* llm_stream(llm_ctx_t* c) {
    if (!c) return nullptr;
    if (hipSetDevice(c->device) != hipSuccess) return nullptr;
    if (finish_copies(c) != 0) return nullptr;
    c->stream_out = true;  // the caller may enqueue on it
    return (void*)c->stream;
}

int llm_sync(llm_ctx_t* c) {
    if (!c) return fail(LLM_E_ARG, "null context");
    HIP_TRY(hipSetDevice(c->device));
    bool late;
    if (int rc = quiesce(c, &late)) return rc;
    return late ? late_error() : 0;
}

int llm_event_record(llm_ctx_t* c, uint32_t slot) {
    if (!c || slot >= 1024) return fail(LLM_E_ARG, "bad event slot");
    c->busy = llm_ctx::WORK;
    HIP_TRY(hipSetDevice(c->device));
    if (c->events.empty()) {
        c->events.resize(1024);
        for (auto& e : c->events) HIP_TRY(hipEventCreate(&e));
    }
    HIP_TRY(hipEventRecord(c->events[slot], c->stream));
    return 0;
}

int llm_event_elapsed_ms(llm_ctx_t* c, uint32_t a, uint32_t b, float* ms) {
    if (!c || !ms || a >= c->events.size() || b >= c->events.size())
        return fail(LLM_E_ARG, "bad event slots");
    HIP_TRY(hipEventSynchronize(c->events[b]));
    HIP_TRY(hipEventElapsedTime(ms, c->events[a], c->events[b]));
    return 0;
}

int llm_kernel_timing(llm_ctx_t* c, int enable) {
    if (!c) return fail(LLM_E_ARG, "null context");
    c->busy = llm_ctx::WORK;
    HIP_TRY(hipSetDevice(c->device));
    harvest_timing(c);
    for (int k = 0; k < LLM_K_COUNT; k++) c->kernel_ms[k] = 0, c->kernel_n[k] = 0;
    c->timing = enable != 0;
    return 0;
}

int llm_kernel_stats(llm_ctx_t* c, uint32_t kernel, uint64_t* launches,
                     double* total_ms) {
    if (!c || kernel >= LLM_K_COUNT) return fail(LLM_E_ARG, "bad kernel id");
    HIP_TRY(hipSetDevice(c->device));
    harvest_timing(c);
    if (launches) *launches = c->kernel_n[kernel];
    if (total_ms) *total_ms = c->kernel_ms[kernel];
    return 0;
}

int llm_bench_projection(llm_ctx_t* c, uint32_t kernel, uint32_t rows,
                         uint32_t layers, uint32_t iters, float* avg_us) {
    if (!c || !avg_us || rows == 0 || rows > 8 || layers == 0 ||
        layers > c->L || iters == 0)
        return fail(LLM_E_ARG, "bad projection benchmark arguments");
    if (kernel != LLM_K_QKV && kernel != LLM_K_OPROJ &&
        kernel != LLM_K_GATEUP && kernel != LLM_K_DOWN)
        return fail(LLM_E_ARG, "not a projection kernel");
    c->busy = llm_ctx::WORK;
    HIP_TRY(hipSetDevice(c->device));
    auto launch = [&](uint32_t layer) -> hipError_t {
        llm::ProjArgs a{};
        a.rows = rows;
        int epi = llm::EPI_STORE, L = 16;
        uint32_t blocks = 0;
        if (kernel == LLM_K_QKV) {
            const Matrix& m = c->mat(layer, M_QKV);
            a.w0 = m.d; a.steps = m.steps; a.x = c->xn_attn; a.ldx = c->Hp;
            a.out = c->qkv; a.ldo = c->Nqkv; a.n = m.n; L = m.L; blocks = m.n_pad / 4;
            set_mf(c, a, m);
            if (m.p12_ok) a.p0 = m.p12;
        } else if (kernel == LLM_K_OPROJ || kernel == LLM_K_DOWN) {
            const Matrix& m = c->mat(layer, kernel == LLM_K_OPROJ ? M_O : M_DOWN);
            a.w0 = m.d; a.steps = m.steps;
            a.x = kernel == LLM_K_OPROJ ? c->attn : c->act;
            a.ldx = kernel == LLM_K_OPROJ ? c->Hp : c->Ip;
            // output into a buffer the launch does not read
            a.out = c->qkv; a.ldo = c->Nqkv; a.res = c->xn_ffn; a.ldr = c->Hp;
            a.n = m.n; L = m.L; blocks = m.n_pad / 4; epi = llm::EPI_RESID;
            set_mf(c, a, m);
            if (m.p12_ok) a.p0 = m.p12;
        } else {
            const Matrix& g = c->mat(layer, M_GATE);
            const Matrix& u = c->mat(layer, M_UP);
            a.w0 = g.d; a.w1 = u.d; a.steps = g.steps; a.x = c->xn_ffn;
            a.ldx = c->Hp; a.out = c->act; a.ldo = c->Ip; a.n = g.n;
            a.exp8 = c->exp8; a.silu8 = c->silu8;
            L = std::min(g.L, u.L); blocks = g.n_pad / 4;
            epi = llm::EPI_SILU;
            set_mf(c, a, g, &u);
            if (g.p12_ok && u.p12_ok) {
                a.p0 = g.p12;
                a.p1 = u.p12;
            }
        }
        return llm::launch_proj(a, epi, L, blocks, c->stream);
    };
    hipEvent_t e0, e1;
    HIP_TRY(hipEventCreate(&e0));
    HIP_TRY(hipEventCreate(&e1));
    hipError_t e = launch(0);  // warm the instruction cache
    (void)hipEventRecord(e0, c->stream);
    for (uint32_t i = 0; i < iters && e == hipSuccess; i++) e = launch(i % layers);
    (void)hipEventRecord(e1, c->stream);
    (void)hipEventSynchronize(e1);
    float ms = 0;
    (void)hipEventElapsedTime(&ms, e0, e1);
    (void)hipEventDestroy(e0);
    (void)hipEventDestroy(e1);
    // scratch rows were overwritten: drop derived norm copies
    c->attn_cache.pair = c->ffn_cache.pair = -1;
    if (e != hipSuccess) return fail(LLM_E_HIP, hipGetErrorString(e));
    *avg_us = ms * 1000.0f / iters;
    return 0;
}

int llm_weight_bytes(llm_ctx_t* c, uint64_t* bytes, uint32_t* wide_matrices) {
    if (!c || !bytes || !wide_matrices) return fail(LLM_E_ARG, "null argument");
    uint64_t b = 0;
    uint32_t wide = 0;
    for (const Matrix& m : c->mats) {
        if (m.d) b += m.elems() * sizeof(int16_t), wide++;
        if (m.p12) b += m.elems() / 512 * llm::kP12Step;
        if (m.mf) b += (uint64_t)m.nc * m.kq * llm::kMfRecord;
        if (m.ms) b += (uint64_t)m.nc * llm::kMfRows * 2 * sizeof(int32_t);
        if (m.corr) b += (uint64_t)m.n_pad * llm::kCorrSlots * 4;
    }
    *bytes = b;
    *wide_matrices = wide;
    return 0;
}

int llm_bench_copy(llm_ctx_t* c, uint64_t bytes, uint32_t iters, float* ms) {
    if (!c || !ms || bytes < 16 || iters == 0)
        return fail(LLM_E_ARG, "bad copy arguments");
    c->busy = llm_ctx::WORK;
    HIP_TRY(hipSetDevice(c->device));
    const size_t n16 = bytes / 16;
    void *src = nullptr, *dst = nullptr;
    HIP_TRY(hipMalloc(&src, n16 * 16));
    if (hipMalloc(&dst, n16 * 16) != hipSuccess) {
        (void)hipFree(src);
        return fail(LLM_E_NOMEM, "copy buffer");
    }
    (void)hipMemsetAsync(src, 1, n16 * 16, c->stream);
    hipEvent_t a, b;
    (void)hipEventCreate(&a);
    (void)hipEventCreate(&b);
    hipError_t e = llm::launch_copy((const uint4*)src, (uint4*)dst, n16, c->stream);
    (void)hipEventRecord(a, c->stream);
    for (uint32_t i = 0; i < iters && e == hipSuccess; i++)
        e = llm::launch_copy((const uint4*)src, (uint4*)dst, n16, c->stream);
    (void)hipEventRecord(b, c->stream);
    (void)hipEventSynchronize(b);
    float t = 0;
    (void)hipEventElapsedTime(&t, a, b);
    *ms = t / iters;
    (void)hipEventDestroy(a);
    (void)hipEventDestroy(b);
    (void)hipFree(src);
    (void)hipFree(dst);
    if (e != hipSuccess) return fail(LLM_E_HIP, hipGetErrorString(e));
    return 0;
}

int llm_exp_tables(int16_t* q8_8, int16_t* q2_14) {
    int16_t a[2049], b[2049];
    build_exp_tables(a, b);
    if (q8_8) std::memcpy(q8_8, a, sizeof(a));
    if (q2_14) std::memcpy(q2_14, b, sizeof(b));
    return 0;
}

}  // extern "C"

namespace {

int64_t key_score(unsigned long long k) {
    return (int64_t)(k >> 18) - ((int64_t)1 << 45);
}
uint32_t key_token(unsigned long long k) {
    return llm::kArgmaxVocabMax - (uint32_t)(k & llm::kArgmaxVocabMax);
}

double ms_since(std::chrono::steady_clock::time_point t) {
    return std::chrono::duration<double, std::milli>(
               std::chrono::steady_clock::now() - t).count();
}

// Stream events of the request loop: at least n of them.
int gen_events(llm_ctx* c, size_t n) {
    while (c->gen_events.size() < n) {
        hipEvent_t e;
        HIP_TRY(hipEventCreate(&e));
        c->gen_events.push_back(e);
    }
    return 0;
}

float event_ms(hipEvent_t a, hipEvent_t b) {
    float ms = 0;
    return hipEventElapsedTime(&ms, a, b) == hipSuccess ? ms : 0.0f;
}

void emit(llm_ctx* c, const std::string& line) {
    if (c->log_fn) c->log_fn(line.c_str(), c->log_user);
}

std::string fmt_ms(double v) {
    char b[32];
    std::snprintf(b, sizeof b, "%.6f", v);
    return b;
}

// One forward of `rows` rows at `position` through layers [0, layer_count)
// (run_composed_decoder_stack, host/host_qwen_8x64.cpp:1258-1445): the
// rows (pinned host memory) into pair 1 by a copy kernel, Task 18
// (1 -> 0) and 19 (0 -> 1) per layer, Task 20 (1 -> 0) when `final_norm`.
// Nothing is waited for, unless a line sink is set: then the forward is
// bracketed by stream events per task, synchronised, and reported as the
// reference reports its coarse tasks (COARSE_TASK_PROGRESS per task, then
// one COARSE_TASK_PREFILL_BLOCK or COARSE_TASK_STACK line).
int run_stack(llm_ctx_t* c, const int16_t* rows_host, uint32_t rows, uint32_t position,
              uint32_t layer_count, bool final_norm, bool prompt_block,
              uint32_t* tasks) {
    const bool prof = c->log_fn != nullptr;
    const uint32_t ntask = 2 * layer_count + (final_norm ? 1u : 0u);
    if (prof)
        if (int rc = gen_events(c, 2 + ntask)) return rc;
    const auto host0 = std::chrono::steady_clock::now();
    auto enqueue = [&]() -> int {
        if (prof) HIP_TRY(hipEventRecord(c->gen_events[0], c->stream));
        invalidate_pair(c, 1);
        HIP_TRY(llm::launch_io_rows(rows_host, c->H, c->pairs[1], c->Hp, c->H, rows, nullptr,
                                    nullptr, 0, c->stream));
        c->n_h2d_rows++;
        if (prof) HIP_TRY(hipEventRecord(c->gen_events[1], c->stream));
        llm_status_t st;
        uint32_t done = 0;
        auto task = [&](uint32_t op, uint32_t layer, uint32_t in, uint32_t out) {
            const int r = llm_task(c, op, layer, rows, position, 0, in, out, &st);
            if (r < 0) return r;
            if (r != 0 || st.op != op || !st.last_task)
                return fail(LLM_E_STATE, "controller status failure: op " +
                                             std::to_string(op) + " code " +
                                             std::to_string(st.code));
            if (prof) HIP_TRY(hipEventRecord(c->gen_events[2 + done], c->stream));
            done++;
            return 0;
        };
        int rc;
        for (uint32_t layer = 0; layer < layer_count; layer++) {
            if ((rc = task(LLM_OP_ATTENTION_SUBLAYER, layer, 1, 0))) return rc;
            if ((rc = task(LLM_OP_FFN_SUBLAYER, layer, 0, 1))) return rc;
        }
        if (final_norm && (rc = task(LLM_OP_FINAL_NORM, 0, 1, 0))) return rc;
        return 0;
    };
    if (int rc = enqueue()) return rc;
    *tasks += ntask;
    if (!prof) return 0;
    HIP_TRY(hipStreamSynchronize(c->stream));
    if (clear_waits(c)) {
        // a bounded wait gave up: this forward again, without such waits
        // (its K/V rows are rewritten from the same rows)
        WaitFreeScope wf(c);
        c->n_wait_reruns++;
        if (int rc = enqueue()) return rc;
        SYNC_TRY(c);
    }
    const double host_ms = ms_since(host0);
    double phase_ms[3] = {0, 0, 0};  // attention, FFN, final norm
    for (uint32_t k = 0; k < ntask; k++) {
        const bool fin = final_norm && k + 1 == ntask;
        const uint32_t ph = fin ? 2 : k % 2;
        const double ms = event_ms(c->gen_events[1 + k], c->gen_events[2 + k]);
        phase_ms[ph] += ms;
        static const char* names[3] = {"attention", "ffn", "final_norm"};
        static const uint32_t ops[3] = {LLM_OP_ATTENTION_SUBLAYER, LLM_OP_FFN_SUBLAYER,
                                        LLM_OP_FINAL_NORM};
        emit(c, "COARSE_TASK_PROGRESS completed=" + std::to_string(k + 1) +
                    " total=" + std::to_string(ntask) + " op=" + std::to_string(ops[ph]) +
                    " phase=" + names[ph] + " layer=" + std::to_string(fin ? 0 : k / 2) +
                    " position=" + std::to_string(position) +
                    " query_tokens=" + std::to_string(rows) + " controller_ms=" + fmt_ms(ms));
    }
    const double input_ms = event_ms(c->gen_events[0], c->gen_events[1]);
    const double active_ms = event_ms(c->gen_events[1], c->gen_events[1 + ntask]);
    std::string line =
        std::string(prompt_block ? "COARSE_TASK_PREFILL_BLOCK" : "COARSE_TASK_STACK") +
        " layers=" + std::to_string(layer_count) + " tasks=" + std::to_string(ntask);
    if (prompt_block)
        line += " position_begin=" + std::to_string(position) +
                " query_tokens=" + std::to_string(rows) +
                " position_end=" + std::to_string(position + rows - 1);
    else
        line += " position=" + std::to_string(position);
    line += " event_timing_domain=hip_stream_event attention_controller_ms=" +
            fmt_ms(phase_ms[0]) + " ffn_controller_ms=" + fmt_ms(phase_ms[1]) +
            " final_norm_controller_ms=" + fmt_ms(phase_ms[2]) +
            " kernel_active_ms=" + fmt_ms(active_ms) + " input_migration_ms=" +
            fmt_ms(input_ms) +
            " auxiliary_migration_ms=0 status_kernel_ms=0 status_migration_ms=0"
            " output_migration_ms=0 profiled_sequence_ms=" +
            fmt_ms(input_ms + active_ms) + " host_elapsed_ms=" + fmt_ms(host_ms);
    if (prompt_block) line += std::string(" output_materialized=") + (final_norm ? "1" : "0");
    line += " intermediate_host_copy=0";
    if (prompt_block) line += " kv_cache_owner=controller";
    c->coarse_active_ms += active_ms;
    c->coarse_input_ms += input_ms;
    c->coarse_host_ms += host_ms;
    emit(c, line);
    return 0;
}

// Rows of a prompt that go through a layer at once (its workspace is bounded
// by them), and the blocks from which that is the faster way: one layer takes
// ~128 us for up to 32 rows at once on config B (91 at hidden 896, 70 at 480,
// 57 at 256), and in blocks of 8 or 5 rows 180 / 115 / 93 / 91 us for four of
// them, 136 / 88 / 71 / 69 for three; in one-row blocks 139 / 81 / 70 / 64 for
// four.  Every launch whose matrices have corrections adds ~15 us to a layer
// (all four, hidden 2,048 / 896 / 512 / 256: 163 / 130 / 104 / 86 against 163
// / 113 / 92 / 87 for four blocks of 8, 210 / 143 / 117 / 112 for five, and
// 206 / 125 / 103 / 92 for five of two; one of the four, hidden 896: 105
// against 112 for four): from two launches a layer on one block more.  With
// matrices held in 16 bits 183 / 124 / 93 / 75 against 195 / 110 / 86 / 83
// for four blocks: six.
constexpr uint32_t kPfMaxRows = 2048;
constexpr uint32_t pf_min_blocks(uint32_t block, bool corr, bool wide) {
    return (block > 1 ? 4 : 5) + (wide ? 2 : (corr ? 1 : 0));
}
// Split-K scratch of its products: at most 256 workgroup parts of 128 x 128
// 64-bit sums, and their arrival counters.
constexpr size_t kPfPartBytes = (size_t)256 * 128 * 128 * 8;
constexpr uint32_t kPfMaxTiles = 256;

// Whether every matrix of layers [0, layer_count) has a layout that the
// layer-major prompt path reads.
bool prompt_path_ok(llm_ctx* c, uint32_t n_prompt, uint32_t block, uint32_t layer_count) {
    const uint32_t blocks = cdiv(n_prompt, block);
    if (!c->prompt_path || c->const_gain <= 0 || c->log_fn || blocks < pf_min_blocks(block, false, false))
        return false;
    bool wide = false;
    uint32_t corr = 0;  // launches with corrections
    for (uint32_t l = 0; l < layer_count; l++) {
        for (int m = 0; m < M_COUNT; m++) {
            const Matrix& mt = c->mat(l, m);
            if (mt.steps > llm::kP12MaxSteps || (!mt.p12_ok && !mt.mf)) return false;
            wide |= !mt.p12_ok;
        }
        const Matrix &g = c->mat(l, M_GATE), &u = c->mat(l, M_UP);
        if (!(g.p12_ok && u.p12_ok) && !(g.mf && u.mf)) return false;
        corr += c->mat(l, M_QKV).corr_any + c->mat(l, M_O).corr_any +
                (g.corr_any || u.corr_any) + c->mat(l, M_DOWN).corr_any;
    }
    return blocks >= pf_min_blocks(block, corr > layer_count, wide);
}

// Places the buffers for p.rows rows from p.base on (nowhere while that is
// null); returns their bytes.
size_t place_prompt_buffers(const llm_ctx* c, llm_ctx::Prompt& p) {
    size_t at = 0;
    auto take = [&](auto*& ptr, size_t bytes) {
        ptr = p.base ? (std::remove_reference_t<decltype(ptr)>)(p.base + at) : nullptr;
        at += (bytes + 255) / 256 * 256;
    };
    const size_t R = p.rows, np = round_up(c->Nqkv, 128);
    take(p.in, R * c->H * 2);
    take(p.ha, R * c->Hp * 2);
    take(p.hb, R * c->Hp * 2);
    take(p.qkv, R * np * 2);
    take(p.xn, llm::pf_xp_bytes(p.rows, c->Hp));
    take(p.xa, llm::pf_xp_bytes(p.rows, c->Hp));
    take(p.act, llm::pf_xp_bytes(p.rows, c->Ip));
    take(p.qp, llm::pf_qp_bytes(p.rows, c->Hq, c->d));
    take(p.kp, llm::pf_kp_bytes(c->Hkv, c->tiles, c->d));
    take(p.vp, llm::pf_vp_bytes(c->Hkv, c->tiles, c->d));
    take(p.kbias, (size_t)c->Hkv * c->tiles * 64 * 4);
    take(p.rowsum, R * 4);
    take(p.kvflag, (size_t)2 * c->Hkv * c->tiles * 4);
    take(p.qflag, (size_t)c->Hq * (R / 32) * 4);
    take(p.count, kPfMaxTiles * 4);
    take(p.part, kPfPartBytes);
    p.part_bytes = kPfPartBytes;
    return at;
}

// Buffers for `rows` rows at a time or, where there is no room for them, for
// as many (half, a quarter, ...) as there is: c->pf.rows, 0 if for none.  The
// buffers in hand are given up only for larger ones.
int prompt_buffers(llm_ctx* c, uint32_t rows) {
    const uint32_t pad = llm::kPfRowPad;
    for (uint32_t R = round_up(rows, pad); R > c->pf.rows; R = R > pad ? round_up(R / 2, pad) : 0) {
        llm_ctx::Prompt p{};
        p.rows = R;
        const size_t bytes = place_prompt_buffers(c, p);
        if (bytes > c->prompt_bytes) continue;
        const int rc = dev_alloc(c, (void**)&p.base, bytes);
        if (rc == LLM_E_NOMEM) continue;
        if (rc) return rc;
        place_prompt_buffers(c, p);
        if (c->pf.base) {
            HIP_TRY(hipStreamSynchronize(c->stream));
            if (int r = dev_free(c, c->pf.base)) return r;
        }
        c->pf = p;
        // attention outputs past the heads' width stay 0 (the attention
        // writes whole heads only)
        HIP_TRY(llm::launch_pf_init(p.in, R, 0, c->Hp, c->norms, c->const_gain, p.ha, p.xa,
                                    c->stream));
        break;
    }
    return 0;
}

// Prompt rows [0, n) (pinned host memory) through layers [0, layer_count),
// layer by layer over as many rows at a time as the buffers hold, at most
// kPfMaxRows: K/V rows, hidden pairs and final norm as the blocks of `block`
// rows leave them.
int run_prompt_layers(llm_ctx* c, const int16_t* rows_host, uint32_t n, uint32_t block,
                      uint32_t layer_count) {
    hipStream_t st = c->stream;
    auto& p = c->pf;
    // whole blocks, unless it is all
    const uint32_t cap = std::min(p.rows, kPfMaxRows), chunk = n <= cap ? n : cap / block * block;
    auto gemm = [&](const int8_t* x, uint32_t m, const Matrix& w, const Matrix* w2, int epi,
                    const int16_t* res, int16_t* out, int8_t* xp, const int16_t* gamma) -> int {
        llm::PfGemmArgs a{};
        a.x = x;
        a.m = m;
        a.steps = w.steps;
        a.n = w.n;
        a.kq = w.kq;
        a.ms0 = w.ms;
        a.ms1 = w2 ? w2->ms : nullptr;
        if (w.p12_ok && (!w2 || w2->p12_ok)) {
            a.p0 = w.p12;
            a.p1 = w2 ? w2->p12 : nullptr;
            a.corr0 = w.corr_any ? w.corr : nullptr;
            a.corr1 = w2 && w2->corr_any ? w2->corr : nullptr;
        } else {
            a.mf0 = w.mf;
            a.mf1 = w2 ? w2->mf : nullptr;
            HIP_TRY(llm::launch_pf_rowsum(x, m, w.steps, p.rowsum, st));
            a.rowsum = p.rowsum;
        }
        a.res = res;
        a.out = out;
        a.xp_out = xp;
        a.norm_gamma = gamma;
        a.norm_gain = c->const_gain;
        a.silu8 = c->silu8;
        a.part = p.part;
        a.part_bytes = p.part_bytes;
        a.count = p.count;
        a.max_tiles = kPfMaxTiles;
        HIP_TRY(llm::launch_pf_gemm(a, epi, st));
        return 0;
    };
    for (uint32_t c0 = 0; c0 < n; c0 += chunk) {
        const uint32_t m = std::min(chunk, n - c0);
        HIP_TRY(hipMemcpyAsync(p.in, rows_host + (size_t)c0 * c->H, (size_t)m * c->H * 2,
                               hipMemcpyHostToDevice, st));
        c->n_h2d_rows += cdiv(m, block);  // counted per block of rows
        HIP_TRY(llm::launch_pf_init(p.in, m, c->H, c->Hp, c->norms, c->const_gain, p.ha, p.xn, st));
        for (uint32_t l = 0; l < layer_count; l++) {
            int rc = check_layer_loaded(c, l, true, true);
            if (rc) return rc;
            const int16_t* gf = c->norms + (size_t)(2 * l + 1) * c->H;
            const int16_t* gn = c->norms + (size_t)(2 * l + 2) * c->H;
            {
                TimedScope ts(c, LLM_K_QKV);
                if ((rc = gemm(p.xn, m, c->mat(l, M_QKV), nullptr, llm::EPI_STORE, nullptr, p.qkv,
                               nullptr, nullptr)))
                    return rc;
            }
            llm::PfAttnArgs at{};
            at.qkv = p.qkv;
            at.qkv_nt = round_up(c->Nqkv, 128) / 32;
            at.m = m;
            at.pos0 = c0;
            at.rope = c->rope;
            const size_t layer_off = (size_t)l * c->Hkv * c->tiles * llm::kTile * c->d;
            at.kcache = c->kcache + layer_off;
            at.vcache = c->vcache + layer_off;
            at.tiles = c->tiles;
            at.num_heads = c->Hq;
            at.num_kv_heads = c->Hkv;
            at.group = c->G;
            at.head_dim = c->d;
            at.qk_scale = c->qk_scale;
            at.exp14 = c->exp14;
            at.qp = p.qp;
            at.kp = p.kp;
            at.vp = p.vp;
            at.kbias = p.kbias;
            at.kvflag = p.kvflag;
            at.qflag = p.qflag;
            at.xp_out = p.xa;
            at.out_steps = c->Hp / 128;
            {
                TimedScope ts(c, LLM_K_ROPE);
                HIP_TRY(llm::launch_pf_kvq(at, st));
            }
            {
                TimedScope ts(c, LLM_K_ATTENTION);
                HIP_TRY(llm::launch_pf_attention(at, st));
            }
            {
                TimedScope ts(c, LLM_K_OPROJ);
                if ((rc = gemm(p.xa, m, c->mat(l, M_O), nullptr, llm::EPI_RESID, p.ha, p.hb, p.xn, gf)))
                    return rc;
            }
            {
                TimedScope ts(c, LLM_K_GATEUP);
                if ((rc = gemm(p.xn, m, c->mat(l, M_GATE), &c->mat(l, M_UP), llm::EPI_SILU, nullptr,
                               nullptr, p.act, nullptr)))
                    return rc;
            }
            {
                TimedScope ts(c, LLM_K_DOWN);
                const bool next = l + 1 < layer_count;
                if ((rc = gemm(p.act, m, c->mat(l, M_DOWN), nullptr, llm::EPI_RESID, p.hb, p.ha,
                               next ? p.xn : nullptr, next ? gn : nullptr)))
                    return rc;
            }
        }
        invalidate_pair(c, 0);
        invalidate_pair(c, 1);
        HIP_TRY(llm::launch_pf_finish(p.hb, p.ha, m, c->H, c->Hp, block, c0 + m == n,
                                      c->norms + (size_t)(2 * c->L) * c->H, c->const_gain,
                                      c->pairs[0], c->pairs[1], st));
    }
    return 0;
}

// The LM-head argmax of rows [row0, row0 + rows) of `pair` enqueued, its
// keys (which are 0 between argmaxes) published to pinned host memory as
// transfer *seq.
int ensure_keys_host(llm_ctx_t* c) {
    if (!c->keys_host &&
        hipHostMalloc((void**)&c->keys_host, 8 * sizeof(unsigned long long),
                      hipHostMallocDefault) != hipSuccess)
        return fail(LLM_E_NOMEM, "hipHostMalloc failed");
    return 0;
}

int enqueue_argmax(llm_ctx_t* c, uint32_t pair, uint32_t row0, uint32_t rows, uint32_t* seq) {
    c->busy = llm_ctx::WORK;
    HIP_TRY(llm::launch_lm_argmax(c->lm.d, c->lm.steps, c->lm_vocab,
                                  c->pairs[pair] + (size_t)row0 * c->Hp, c->Hp, rows,
                                  c->lm.L, c->lm_keys, c->stream));
    *seq = ++c->io_seq;
    HIP_TRY(llm::launch_keys_out(c->lm_keys, c->keys_host, c->io_flag, *seq, c->stream));
    c->n_argmax++;
    return 0;
}

}  // namespace

extern "C" {

int llm_load_lm_head(llm_ctx_t* c, const int16_t* table, uint32_t vocab) {
    if (!c || !table || vocab == 0 || vocab > llm::kArgmaxVocabMax)
        return fail(LLM_E_ARG, "bad LM head arguments");
    if (c->H > 16384) return fail(LLM_E_ARG, "hidden too large for the argmax key");
    HIP_TRY(hipSetDevice(c->device));
    Matrix& m = c->lm;
    const uint32_t n_pad = round_up(vocab, llm::kBlockRows);
    if (!m.d || m.n != vocab) {
        int rc;
        m = Matrix{};
        m.n = vocab;
        m.k = c->H;
        m.n_pad = n_pad;
        m.k_pad = round_up(c->H, llm::kStepCols);
        m.steps = m.k_pad / llm::kStepCols;
        if ((rc = dev_alloc(c, (void**)&m.d, m.elems() * sizeof(int16_t)))) return rc;
        if (!c->lm_keys &&
            (rc = dev_alloc(c, (void**)&c->lm_keys, 8 * sizeof(unsigned long long))))
            return rc;
    }
    const int rc = upload_rows(c, m, 0, vocab, table, 0);
    if (rc) return rc;
    c->lm_vocab = vocab;
    return 0;
}

int llm_lm_head_argmax(llm_ctx_t* c, uint32_t pair, uint32_t row0, uint32_t rows,
                       uint32_t* tokens, int64_t* scores) {
    if (!c || !tokens || pair >= c->pairs.size() || rows == 0 || row0 + rows > 8)
        return fail(LLM_E_ARG, "bad LM head argmax arguments");
    if (!c->lm_vocab) return fail(LLM_E_STATE, "LM head not loaded");
    HIP_TRY(hipSetDevice(c->device));
    if (int rc = ensure_keys_host(c)) return rc;
    uint32_t seq;
    if (int rc = enqueue_argmax(c, pair, row0, rows, &seq)) return rc;
    if (int rc = io_wait(c, seq)) return rc;
    if (int rc = check_waits(c)) return rc;
    for (uint32_t r = 0; r < rows; r++) {
        tokens[r] = key_token(c->keys_host[r]);
        if (scores) scores[r] = key_score(c->keys_host[r]);
    }
    return 0;
}

int llm_generate(llm_ctx_t* c, const int16_t* embedding, uint32_t vocab,
                 const uint32_t* prompt, uint32_t n_prompt, uint32_t block_size,
                 uint32_t layer_count, uint32_t max_new_tokens,
                 uint32_t* out_tokens, llm_generate_stats_t* stats) {
    if (!c || !embedding || !prompt || n_prompt == 0 || block_size == 0 ||
        block_size > 8 || layer_count == 0 || layer_count > c->L ||
        (max_new_tokens && !out_tokens))
        return fail(LLM_E_ARG, "bad generate arguments");
    if (!c->lm_vocab && max_new_tokens) return fail(LLM_E_STATE, "LM head not loaded");
    const uint64_t last_pos = (uint64_t)n_prompt + (max_new_tokens ? max_new_tokens - 1 : 0);
    if (last_pos > c->max_seq)
        return fail(LLM_E_ARG, "sequence exceeds max_seq_len");
    for (uint32_t t = 0; t < n_prompt; t++)
        if (prompt[t] >= vocab) return fail(LLM_E_ARG, "prompt token outside the vocabulary");
    c->busy = llm_ctx::WORK;
    HIP_TRY(hipSetDevice(c->device));
    llm_generate_stats_t local{};
    llm_generate_stats_t& S = stats ? *stats : local;
    S = llm_generate_stats_t{};
    S.prompt_tokens = n_prompt;
    S.generated_tokens = max_new_tokens;
    const auto begin = std::chrono::steady_clock::now();
    // Embedding rows of the whole request in pinned memory (the prompt's
    // now, each sampled token's when it is known): every forward's rows
    // travel by an asynchronous copy, and nothing waits between forwards
    // but the argmax read-back each sampled token needs.
    const size_t need = (size_t)n_prompt + max_new_tokens;
    if (c->stage_rows < need) {
        if (c->stage) (void)hipHostFree(c->stage);
        c->stage = nullptr;
        c->stage_rows = 0;
        if (hipHostMalloc((void**)&c->stage, need * c->H * sizeof(int16_t),
                          hipHostMallocDefault) != hipSuccess)
            return fail(LLM_E_NOMEM, "hipHostMalloc failed");
        c->stage_rows = need;
    }
    if (int rc = ensure_keys_host(c)) return rc;
    if (int rc = gen_events(c, 2 + 2 * (size_t)layer_count + 1 + 8)) return rc;
    const size_t ne = c->gen_events.size();
    hipEvent_t ev_p0 = c->gen_events[ne - 8], ev_p1 = c->gen_events[ne - 7];
    // before a forward's rows' copy, after its last task, after its argmax:
    // two sets, so that a step's times are read behind the next forward
    hipEvent_t* ev_a = &c->gen_events[ne - 6];
    hipEvent_t* ev_b = &c->gen_events[ne - 4];
    hipEvent_t* ev_l = &c->gen_events[ne - 2];
    for (uint32_t t = 0; t < n_prompt; t++)
        std::memcpy(c->stage + (size_t)t * c->H, embedding + (size_t)prompt[t] * c->H,
                    (size_t)c->H * 2);
    const uint64_t h2d0 = c->n_h2d_rows, d2h0 = c->n_d2h_rows, kv0 = c->n_kv_moves,
                   am0 = c->n_argmax;
    const double active0 = c->coarse_active_ms, input0 = c->coarse_input_ms,
                 hostapi0 = c->coarse_host_ms;
    const uint64_t rr0 = c->n_wait_reruns;
    uint32_t last_row = 0;
    int rc;
    // prompt blocks (host/host_qwen_8x64.cpp:9016-9060, :7840-7884), enqueued
    // without waiting; `count` adds them to the request's counters (a re-run
    // after a wait that gave up does not)
    auto run_prompt = [&](bool count) -> int {
        uint32_t uncounted = 0;
        HIP_TRY(hipEventRecord(ev_p0, c->stream));
        const bool layers = prompt_path_ok(c, n_prompt, block_size, layer_count);
        if (layers)
            if (int r = prompt_buffers(c, std::min(n_prompt, kPfMaxRows))) return r;
        if (layers && c->pf.rows) {
            if (int r = run_prompt_layers(c, c->stage, n_prompt, block_size, layer_count)) return r;
            const uint32_t blocks = (uint32_t)cdiv(n_prompt, block_size);
            if (count) {
                S.coarse_task_count += blocks * 2 * layer_count + 1;
                S.prompt_forward_passes = blocks;
                S.output_materializations++;
                S.released_prompt_blocks = blocks - 1;
            }
            last_row = (n_prompt - 1) % block_size;
            HIP_TRY(hipEventRecord(ev_p1, c->stream));
            return 0;
        }
        for (uint32_t b0 = 0; b0 < n_prompt; b0 += block_size) {
            const uint32_t rows = std::min(block_size, n_prompt - b0);
            const bool final_block = b0 + rows == n_prompt;
            if (int r = run_stack(c, c->stage + (size_t)b0 * c->H, rows, b0, layer_count,
                                  final_block, true, count ? &S.coarse_task_count : &uncounted))
                return r;
            if (count) {
                S.prompt_forward_passes++;
                if (final_block) S.output_materializations++;
                else S.released_prompt_blocks++;
            }
            last_row = rows - 1;
        }
        HIP_TRY(hipEventRecord(ev_p1, c->stream));
        return 0;
    };
    // A synchronisation that finds a bounded wait between workgroups given
    // up: what was enqueued since the previous one (`redo`) runs again, once,
    // on launches without such waits, and is synchronised.  K/V rows of the
    // invalid run are rewritten by the re-run from the same inputs.
    uint32_t seq = 0;  // transfer of the last argmax's keys
    auto settle = [&](const std::function<int()>& redo) -> int {
        if (seq) {
            if (int r = io_wait(c, seq)) return r;
        } else {
            HIP_TRY(hipStreamSynchronize(c->stream));
        }
        if (!clear_waits(c)) return 0;
        WaitFreeScope wf(c);
        c->n_wait_reruns++;
        if (int r = redo()) return r;
        SYNC_TRY(c);
        return 0;
    };
    if ((rc = run_prompt(true))) return rc;
    if (max_new_tokens == 0) {
        if ((rc = settle([&] { return run_prompt(false); }))) return rc;
        S.prompt_forward_ms = event_ms(ev_p0, ev_p1);
    }
    // sampled tokens (host/host_qwen_8x64.cpp:9091-9136); times from stream
    // events: a forward from before its rows' copy to after its last task,
    // the LM head from there to its keys' transfer
    auto times = [&](uint32_t step) -> int {
        const uint32_t e = step & 1;
        HIP_TRY(hipEventSynchronize(ev_l[e]));
        if (step == 0) {
            S.prompt_forward_ms = event_ms(ev_p0, ev_p1);
            S.lm_head_ms += event_ms(ev_p1, ev_l[e]);
        } else {
            S.generated_forward_ms += event_ms(ev_a[e], ev_b[e]);
            S.lm_head_ms += event_ms(ev_b[e], ev_l[e]);
        }
        return 0;
    };
    auto forward = [&](uint32_t step, uint32_t* tasks) -> int {  // of the token sampled before it
        const uint32_t t = n_prompt + step - 1;
        HIP_TRY(hipEventRecord(ev_a[step & 1], c->stream));
        if (int r = run_stack(c, c->stage + (size_t)t * c->H, 1, t, layer_count, true, false, tasks))
            return r;
        HIP_TRY(hipEventRecord(ev_b[step & 1], c->stream));
        return 0;
    };
    auto gen0 = std::chrono::steady_clock::now();
    uint32_t token = 0;
    for (uint32_t step = 0; step < max_new_tokens; step++) {
        auto argmax = [&]() -> int {
            if (int r = enqueue_argmax(c, 0, last_row, 1, &seq)) return r;
            HIP_TRY(hipEventRecord(ev_l[step & 1], c->stream));
            return 0;
        };
        if ((rc = argmax())) return rc;
        rc = settle([&]() -> int {
            uint32_t uncounted = 0;
            const int r = step == 0 ? run_prompt(false) : forward(step, &uncounted);
            return r ? r : argmax();
        });
        if (rc) return rc;
        token = key_token(c->keys_host[0]);
        if (step == 0) {
            S.time_to_first_token_ms = ms_since(begin);
            gen0 = std::chrono::steady_clock::now();  // the generated forwards from here
        }
        out_tokens[step] = token;
        if (step + 1 < max_new_tokens) {
            if (token >= vocab) return fail(LLM_E_STATE, "sampled token outside the embedding");
            std::memcpy(c->stage + ((size_t)n_prompt + step) * c->H,
                        embedding + (size_t)token * c->H, (size_t)c->H * 2);
            if ((rc = forward(step + 1, &S.coarse_task_count))) return rc;
            S.generated_forward_passes++;
            S.output_materializations++;
            last_row = 0;
        }
        if ((rc = times(step))) return rc;
    }
    S.generated_wall_ms = max_new_tokens > 1 ? ms_since(gen0) : 0.0;
    S.total_ms = ms_since(begin);
    S.input_migrations = (uint32_t)(c->n_h2d_rows - h2d0);
    S.output_migrations = (uint32_t)(c->n_d2h_rows - d2h0);
    S.kv_migrations = (uint32_t)(c->n_kv_moves - kv0);
    S.argmax_readbacks = (uint32_t)(c->n_argmax - am0);
    S.wait_reruns = (uint32_t)(c->n_wait_reruns - rr0);
    if (c->log_fn) {
        const double mean_ms =
            S.generated_forward_passes ? S.generated_forward_ms / S.generated_forward_passes : 0;
        const double dec = S.generated_forward_ms > 0
                               ? 1000.0 * S.generated_forward_passes / S.generated_forward_ms : 0;
        const double pre = S.prompt_forward_ms > 0 ? 1000.0 * n_prompt / S.prompt_forward_ms : 0;
        emit(c, "QWEN_8X64_E2E_PROFILE prompt_tokens=" + std::to_string(n_prompt) +
                    " generated_tokens=" + std::to_string(max_new_tokens) +
                    " prompt_forward_passes=" + std::to_string(S.prompt_forward_passes) +
                    " generated_forward_passes=" + std::to_string(S.generated_forward_passes) +
                    " prefill_mode=coarse_block prefill_block_size=" +
                    std::to_string(block_size) + " prompt_forward_ms=" +
                    fmt_ms(S.prompt_forward_ms) + " prefill_token_s=" + fmt_ms(pre) +
                    " time_to_first_token_ms=" + fmt_ms(S.time_to_first_token_ms) +
                    " generated_forward_ms=" + fmt_ms(S.generated_forward_ms) +
                    " mean_inter_token_ms=" + fmt_ms(mean_ms) + " decode_token_s=" +
                    fmt_ms(dec) + " lm_head_host_ms=" + fmt_ms(S.lm_head_ms) +
                    " total_host_elapsed_ms=" + fmt_ms(S.total_ms) +
                    // no golden check runs inside the request: the process
                    // time is the inference time and validation is off
                    " total_process_elapsed_ms=" + fmt_ms(S.total_ms) +
                    " post_inference_validation_ms=0 validation_schedule=disabled"
                    " event_timing_domain=hip_stream_event coarse_task_count=" +
                    std::to_string(S.coarse_task_count) + " coarse_kernel_active_ms=" +
                    fmt_ms(c->coarse_active_ms - active0) + " coarse_profiled_sequence_ms=" +
                    fmt_ms(c->coarse_active_ms - active0 + c->coarse_input_ms - input0) +
                    " coarse_host_api_elapsed_ms=" + fmt_ms(c->coarse_host_ms - hostapi0) +
                    " coarse_input_migration_ms=" + fmt_ms(c->coarse_input_ms - input0) +
                    " coarse_status_kernel_ms=0 coarse_status_migration_ms=0"
                    " coarse_output_migration_ms=0"
                    " output_materializations=" + std::to_string(S.output_materializations) +
                    " released_prompt_blocks=" + std::to_string(S.released_prompt_blocks) +
                    " e2e_numeric_golden=0 e2e_numeric_steps=0 e2e_numeric_checked_values=0"
                    " e2e_numeric_max_raw_error=0 e2e_numeric_tolerance=0 e2e_golden_host_ms=0"
                    " input_migrations=" + std::to_string(S.input_migrations) +
                    " output_migrations=" + std::to_string(S.output_migrations) +
                    " kv_migrations=" + std::to_string(S.kv_migrations) +
                    " intermediate_host_copy=0 kv_cache_owner=controller PASS");
    }
    return 0;
}

int llm_set_log(llm_ctx_t* c, llm_log_fn fn, void* user) {
    if (!c) return fail(LLM_E_ARG, "null context");
    c->log_fn = fn;
    c->log_user = user;
    return 0;
}

}  // extern "C"

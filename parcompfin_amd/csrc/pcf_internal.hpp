// pcf_internal.hpp -- host-side internals of libpcf: the context (one HIP
// stream, timing events, resident device buffers), error plumbing and the
// launch-shape helpers shared by the product files.
#pragma once

#include <hip/hip_runtime.h>

#include <cmath>
#include <cstdint>
#include <cstdio>
#include <functional>
#include <mutex>
#include <string>
#include <unordered_map>
#include <vector>

#include "pcf.h"
#include "pcf_device.hpp"

// Grow-only device buffer owned by a context.
struct DevBuf {
    void* ptr = nullptr;
    size_t bytes = 0;
    // Ensures at least n bytes; contents are not preserved.  zero=true clears
    // a newly allocated buffer (once, at allocation).
    hipError_t ensure(size_t n, bool zero = false) {
        if (n <= bytes && ptr) return hipSuccess;
        if (ptr) {
            hipError_t e = hipFree(ptr);
            if (e != hipSuccess) return e;
            ptr = nullptr;
            bytes = 0;
        }
        size_t want = n < 256 ? 256 : n;
        hipError_t e = hipMalloc(&ptr, want);
        if (e != hipSuccess) {
            ptr = nullptr;
            return e;
        }
        bytes = want;
        if (zero) {
            // hipMemset on device memory is asynchronous to the host and runs
            // on the null stream, which the library's non-blocking streams do
            // not wait for: complete it before the buffer is handed out.
            e = hipMemset(ptr, 0, want);
            if (e == hipSuccess) e = hipStreamSynchronize(nullptr);
            if (e != hipSuccess) return e;
        }
        return hipSuccess;
    }
    void release() {
        if (ptr) (void)hipFree(ptr);
        ptr = nullptr;
        bytes = 0;
    }
    template <typename T>
    T* as() const {
        return static_cast<T*>(ptr);
    }
};

// Requests per batched launch; each owns the pcf::kCounterWords arrival
// counters of one grid reduction and kOutPerJob words of results.
constexpr int kMaxBatch = 64;
constexpr int kCounterSlots = kMaxBatch * pcf::kCounterWords;
using pcf::kOutPerJob;
constexpr int kOutDoubles = kMaxBatch * kOutPerJob;
// Bytes of one job record (launch descriptor) staged per batched launch.
constexpr size_t kJobBytes = 512;
// Device-resident basket constants: kMaxBatch slots of 64 KB per context.
constexpr size_t kBasketConstSlot = 64 * 1024;
constexpr int64_t kBasketConstBytes = (int64_t)kBasketConstSlot * kMaxBatch;

// Device-resident basket constants (factor + per-asset terms), LRU slots.
struct BasketCache {
    std::unordered_map<uint64_t, int> where;
    std::vector<uint64_t> key, stamp;
    uint64_t clock = 0;
};

struct pcf_ctx {
    int device = 0;
    hipStream_t stream = nullptr;
    hipEvent_t ev_begin = nullptr, ev_kbeg = nullptr, ev_kend = nullptr, ev_end = nullptr;
    hipEvent_t ev_ready = nullptr;  // hand-off to another stream (no timing)
    std::string last_error;
    std::recursive_mutex mu;
    int cu_count = 0;
    int clock_khz = 0;  // rate of the device clock that kernels stamp
    int64_t total_mem = 0;
    char name[256] = {0};

    DevBuf partials;   // per-block compensated partial sums
    DevBuf counters;   // kCounterSlots uint32 arrival counters, zero at rest
    DevBuf out;        // kOutDoubles final values
    DevBuf normals;    // verification normals copied from the host
    DevBuf logtab;     // binom: glibc log(n), n = 0..N (resident per N)
    int64_t logtab_n = -1;
    DevBuf prefix;     // binom: prefix chain of the descending log sum
    int64_t prefix_n = -1;
    DevBuf logfact;    // binom production: log k! as double-double, k = 0..logfact_n
    int64_t logfact_n = -1;
    DevBuf lsm_store;  // mc_amer path store
    DevBuf lsm_state;  // mc_amer per-path state
    DevBuf lsm_coef;   // mc_amer per-date coefficients / flags
    DevBuf basket_L;   // basket Cholesky factor + per-asset constants
    DevBuf scratch;    // misc (normals dump)
    DevBuf jobs;       // job records of the current batched launch
    DevBuf lattice;    // binomial lattice: u^i, d^k tables + two level rows
    DevBuf lat_ring;   // the one-launch lattice: words its waves exchange (zeroed when allocated)
    uint32_t lat_epoch = 0;               // last tag used in lat_ring
    uint32_t lat_arrived = 0;             // blocks launched on it
    bool lat_in_turn = false;             // blocks by their numbers, not their XCDs'
    double* h_lat = nullptr;              // pinned staging of the tables
    size_t h_lat_bytes = 0;
    uint64_t lattice_key[3] = {0, 0, 0};  // (u, d, N) the tables hold
    void* lattice_ptr = nullptr;          // where they were written
    BasketCache basket_cache;
    double* h_out = nullptr;  // pinned mirror of `out`
    double* h_out_dev = nullptr;  // h_out as kernels address it
    void* h_jobs = nullptr;   // pinned staging of `jobs`
};

// Releases the LSM graphs captured for a context (lsm.hip).
void pcf_lsm_release(pcf_ctx* ctx);

// Error helpers ------------------------------------------------------------
int pcf_fail(pcf_ctx* ctx, int code, const char* fmt, ...);
int pcf_hip_fail(pcf_ctx* ctx, hipError_t e, const char* what);

#define PCF_HIP_CHECK(ctx, expr)                                      \
    do {                                                              \
        hipError_t _e = (expr);                                       \
        if (_e != hipSuccess) return pcf_hip_fail((ctx), _e, #expr);  \
    } while (0)

// Common validation of the reference's scalar arguments.
int pcf_check_common(pcf_ctx* ctx, double S0, double E, double r, double sigma, double T,
                     int64_t N, double payoff_fun);
int pcf_check_opts(pcf_ctx* ctx, const pcf_opts* o);

// Copies `count` FP64 normals to ctx->normals.
int pcf_upload_normals(pcf_ctx* ctx, const pcf_opts* o, int64_t count);

// Waits for an event by polling it from this thread.  A blocking wait sleeps
// in the driver until the completion interrupt and can wake a few hundred
// microseconds after the work ended.
hipError_t pcf_wait_event(hipEvent_t ev);

// Results that kernels write into the pinned buffer (pcf_device.hpp).
//   pcf_arm_results: marks the words of njobs jobs as not yet written; before
//     the launch.
//   pcf_wait_results: waits until words 0..nres-1 and the clock words of every
//     job are there.  s is the stream of the launch, queried now and then so
//     that a failed launch ends the wait; one that ended without its clock
//     words is an error.  *kernel_ms: from the start of the launch's first
//     block to the end of its last, by the device clock.
// A lone call on 2^14 European paths went from 91 us (two copies, five event
// records and a wait whose 10 us sleeps take 60 us) to 12 us.
void pcf_arm_results(pcf_ctx* ctx, int njobs);
int pcf_wait_results(pcf_ctx* ctx, int njobs, int nres, hipStream_t s, double* kernel_ms);

// Launches a grid whose blocks wait for each other (all of them must become
// resident): in order on the device's one stream of such launches, after the
// kernels that other contexts had enqueued.  handover: what the context's
// stream holds goes first.  own_end: the context's kernel-end event is
// recorded after the launch.  *s: the stream it was launched on.
int pcf_launch_persistent(pcf_ctx* ctx, bool handover, bool own_end, hipStream_t* s,
                          const std::function<hipError_t(hipStream_t)>& launch);

// Launches the one-launch lattice, whose waves wait for each other too, on the
// context's stream: after the persistent launches in flight, and after the
// lattices of other contexts unless `capacity` blocks, the most that are
// resident however they are placed, hold theirs and its own.  In turn only a
// persistent launch waits for it, and only if its blocks are not all resident
// yet (word kOutResident of the context's results): each could hold CUs that
// the other's blocks lack.  A wait that cannot be met for another reason gives
// up, and the sweep is made another way.  (Ordered like the persistent
// launches, 300 levels beside 4.4 ms Asian kernels took 4.4 ms a call against
// 0.27, and those kernels, 2^14 American paths and 10^4 chain terms beside 50000
// levels 8.4, 3.6 and 3.6 ms against 5.8, 0.19 and 0.07.)  ctx->ev_end is
// recorded after it.
constexpr int kOutResident = 10;
hipError_t pcf_launch_lattice(pcf_ctx* ctx, int blocks, int capacity,
                              const std::function<hipError_t(hipStream_t)>& launch);
// Before a context's events are destroyed.
void pcf_forget_lattice(pcf_ctx* ctx);

// Waits until no persistent launch of the device is unfinished: the blocks of
// one may still be leaving when its results are there.
void pcf_finish_persistent(int device);

// Ordering around persistent LSM launches, which need all their blocks
// resident at once.  A persistent launch waits for the last kernel every
// other context on its device has enqueued (its kernel-end event), and a
// heavy kernel of any other kind waits for the last persistent launch, so
// neither kind holds CUs the other's blocks are waiting for.
//   pcf_wait_other_contexts: stream s (the persistent stream) waits for the
//     kernel-end event of every other live context on self's device.
//   pcf_after_persistent: called before a request's kernels are enqueued on
//     ctx's stream; when `work` (paths x steps of the launch, paths x assets
//     for a basket, times kPersistentGateFp64 for FP64 arithmetic; HUGE_VAL
//     for the lattices and the per-date LSM form) reaches
//     kPersistentGateWork, the stream waits for the last persistent launch on
//     its device.  2^26 path-steps is about 40 us of the FP32 Asian kernel;
//     its FP64 form takes about 6 times as long.  With `hold`, a heavy launch
//     keeps the device's persistent-launch order locked in *hold; the caller
//     releases it once the kernels' end event (ctx->ev_kend) is recorded, so
//     a persistent launch enqueued from another thread in between cannot miss
//     these kernels (it would wait for that context's previous end event).
constexpr double kPersistentGateWork = 67108864.0;  // 2^26
constexpr double kPersistentGateFp64 = 6.0;
hipError_t pcf_wait_other_contexts(const pcf_ctx* self, hipStream_t s);
hipError_t pcf_after_persistent(pcf_ctx* ctx, double work, std::unique_lock<std::mutex>* hold = nullptr);

// Records the begin event, returns status.  Timing: begin/kbeg/kend/end.
int pcf_timing_begin(pcf_ctx* ctx);
// Device time from pcf_timing_begin to `end`, which is waited for.
int pcf_sequence_ms(pcf_ctx* ctx, hipEvent_t end, double* ms);
// Copies `nout` doubles of results to ctx->h_out, waits, fills timing fields.
int pcf_timing_end(pcf_ctx* ctx, int nout, pcf_result* res);

static inline pcf_opts pcf_opts_or_default(const pcf_opts* o) {
    pcf_opts d;
    pcf_opts_init(&d);
    return o ? *o : d;
}

static inline int pcf_div_up(int64_t a, int64_t b) { return (int)((a + b - 1) / b); }

// Blocks for `items` work items at B threads x ipt items per thread (>= 1).
static inline int pcf_blocks_for(int64_t items, int B, int ipt) {
    const int64_t per = (int64_t)B * (ipt > 0 ? ipt : 1);
    int64_t b = (items + per - 1) / per;
    if (b < 1) b = 1;
    if (b > (1 << 20)) b = 1 << 20;
    return (int)b;
}

// Smallest power-of-two multiple of `ipt` (items per thread) that keeps a
// grid-stride launch over `items` at B threads per block within max_blocks
// blocks.  Beyond a few blocks per CU, extra blocks of a short kernel only
// add dispatch work and arrivals at its final reduction.
static inline int pcf_capped_ipt(int64_t items, int B, int ipt, int64_t max_blocks) {
    while (ipt < 1024 && (items + (int64_t)B * ipt - 1) / ((int64_t)B * ipt) > max_blocks) ipt <<= 1;
    return ipt;
}

// Items per thread of a Monte Carlo launch over `items` work items, of which a
// block takes `per_round` per turn of its loop; item_ps: device time of one
// item with the chip full, in picoseconds.  Modelled time of a shape:
//   rounds of the busiest CU x time of a round x what idle issue slots cost
//   + 3 ns per block (its launch, first loads and closing reduction).
// Measured at B = 256 (basket of 8 assets, 22 10^6 paths): 1, 2, 3, 4, 6, 8
// blocks per CU took 1.51, 1.14, 1.07, 1.04, 1.01, 1.0 times the last; and
// 2033, 3972, 14564 blocks of a 2-asset basket 54.4, 59.2, 91.3 us.  Against
// one item per thread (or 16 blocks per CU): basket 8 x 349525 8.7 -> 6.5 us, x
// 1.4 10^6 18.1 -> 12.7, European 22 10^6 30.2 -> 22.8, Asian 1.4 10^6 x 252
// 247 -> 239 us.
static inline int pcf_items_per_thread(int64_t items, int64_t per_round, int cus, double item_ps) {
    const double c = cus > 0 ? cus : 256;
    const double round_us = item_ps * (double)per_round * c * 1e-6;
    const double idle[9] = {1.51, 1.51, 1.14, 1.07, 1.04, 1.025, 1.01, 1.005, 1.0};
    int best = 1;
    double best_us = HUGE_VAL;
    for (int ipt = 1; ipt < (1 << 20); ipt += ipt < 16 ? 1 : ipt / 8) {
        const double blocks = std::ceil((double)items / ((double)per_round * ipt));
        const double per_cu = std::ceil(blocks / c);
        const double us = per_cu * ipt * round_us * idle[per_cu < 8.0 ? (int)per_cu : 8] + 0.003 * blocks;
        if (us < best_us) {
            best_us = us;
            best = ipt;
        }
        if (blocks <= 0.5 * c) break;  // longer chains on fewer CUs only lose
    }
    return best;
}

// Size class of a request: ceil(log2 N) clamped to [10, 24].
static inline int pcf_size_class(int64_t N) {
    int c = 0;
    while (((int64_t)1 << c) < N && c < 62) ++c;
    return c < 10 ? 10 : (c > 24 ? 24 : c);
}

// Launch shape from the autotuner's table (autotune.cpp); leaves *B / *ipt
// untouched when the (kind, mode, size class) entry was never tuned.
void pcf_tuned_shape(int kind, int mode, int64_t N, int* B, int* ipt);

static inline uint64_t pcf_make_batch_key(int kind, int mode, int variant, int B) {
    return 1ull | ((uint64_t)(kind & 0xff) << 8) | ((uint64_t)(mode & 0xff) << 16) |
           ((uint64_t)(variant & 0xffff) << 24) | ((uint64_t)(B & 0xffff) << 40);
}

static inline pcf_request pcf_make_request(int kind, double S0, double E, double r, double sigma,
                                           double T, int64_t N, double pf, const pcf_opts* o) {
    pcf_request q{};
    q.kind = kind;
    q.S0 = S0;
    q.E = E;
    q.r = r;
    q.sigma = sigma;
    q.T = T;
    q.N = N;
    q.payoff_fun = pf;
    q.assets = 1;
    q.opts = pcf_opts_or_default(o);
    return q;
}

// Per-product batched runners: n requests sharing one batch key, one launch.
// Per-request validation failures land in status[i]; the return value is a
// launch-level failure.  *_batch_key returns 0 and sets *status on invalid input.
uint64_t pcf_eur_batch_key(pcf_ctx* ctx, const pcf_request& q, int* status);
int pcf_eur_run(pcf_ctx* ctx, int n, const pcf_request* const* reqs, pcf_result* res, int* status);
uint64_t pcf_asia_batch_key(pcf_ctx* ctx, const pcf_request& q, int* status);
int pcf_asia_run(pcf_ctx* ctx, int n, const pcf_request* const* reqs, pcf_result* res, int* status);
uint64_t pcf_basket_batch_key(pcf_ctx* ctx, const pcf_request& q, int* status);
int pcf_basket_run(pcf_ctx* ctx, int n, const pcf_request* const* reqs, pcf_result* res, int* status);
// Device bytes an American request holds while in flight: the path store and
// per-path state (grow-only buffers a context keeps between requests) and the
// rest (coefficients, partials, sync words); the footprint is their sum.
struct PcfAmerBytes {
    int64_t store = 0, state = 0, rest = 0;
};
PcfAmerBytes pcf_amer_bytes(int64_t N, int M, int precision, int rng, int ref_exact);
int64_t pcf_amer_footprint(int64_t N, int M, int precision, int rng, int ref_exact);

// opts.fp64_check on a PCF_FP32K Philox request of a Monte Carlo kind: prices
// q again in PCF_FP64 on the same Philox counters and stores |price - FP64
// price| in res->fp64_err (res->fp64_checked = 1).  A no-op otherwise.
int pcf_apply_fp64_check(pcf_ctx* ctx, const pcf_request& q, pcf_result* res);

// glibc pow, never folded by the compiler.  Verification constants follow
// the reference's -O0 build, which calls glibc pow(x, 2.0); compilers fold
// pow(x,2) into x*x, which differs in the last bit for ~0.1% of inputs.
static inline double libm_pow(double x, double y) {
    double (*volatile f)(double, double) = &::pow;
    return f(x, y);
}

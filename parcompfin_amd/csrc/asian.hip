// asian.hip -- fixed-strike arithmetic-average Asian option.
// Hot loop of src/mc_asia.cpp:27-37, per path and step m:
//     I += S (1 + r dt/2 + sigma dB/2);   S *= exp((r - sigma^2/2) dt + sigma dB)
// then payoff(I/M).  (I is the reference's first-order trapezoid of the
// running integral: it includes S_0 and excludes S_M; reproduced as written.)
//
// One path per lane, paths contiguous across lanes; one Philox call feeds 4
// steps.  One kernel serves one request or a batch (see eur.hip: each job
// reduces over exactly the blocks a lone launch of it would use).  FP32 form: S and the exponent in FP32 on the hardware exp2 unit, I
// Kahan-compensated in FP32, per-path payoffs summed in FP64.  The optional
// geometric control averages log S over t_1..t_M on the same paths.
#include "pcf_internal.hpp"

namespace {

struct AsiaArgs {
    double S0, E, pf;
    double a1, a2;          // 1 + r dt/2, sigma sqrt(dt)/2  (I update, standard normal z)
    double mu, vol;         // (r - s^2/2) dt, sigma sqrt(dt)
    double h_c1, h_mu, sigma;  // verification: 1 + r*dt/2, (r - pow(s,2)/2)*dt, sigma
    float mu2f, vol2f;      // FP32; exponent constants x log2(e)
    float awf, bwf;         // FP32: a1 + a2 z = aw + bw e, e the exponent
    double avg32;           // S0 / M, and what rounding aw took from every term
    double invM, sdt;       // 1/M, sqrt(dt)
    int64_t N;
    int32_t M;
    uint64_t seed;
};

enum { kFp32k = 0, kFp64 = 1, kHost = 2, kHostProd = 3 };

// Four steps share one Philox block, one product with S and one compensated
// addition.  With e_j = mu + vol z_j in units of log 2, x_j = e_0 + .. + e_{j-1}
// and w_j = a1 + a2 z_j = aw + bw e_j (a2 / vol is a constant),
//     I += S (w_0 + 2^x_1 w_1 + 2^x_2 w_2 + 2^x_3 w_3),   S *= 2^x_4.
// S takes one exponential and one rounding per 4 steps in place of four of
// each (the hardware exponential's error has a mean, and it grew with M), the
// four terms are rounded three times among themselves, uncompensated, before
// their sum enters the Kahan sum.  (Against a compensated addition per step a
// path's average has the smaller rms error at every M from 1 to 365: 5.3 -> 4.1
// 10^-8 of S0 at 4 steps, 3.4 -> 1.8 10^-7 at 252.)  e_j takes the pair's
// radius times vol, so the normals themselves are never formed.  25 VALU
// instructions per 4 steps against 36 (with the generator, 77 against 88): the
// kernel is bound by their issue, 4.2 10^6 x 252 655 -> 560 us.  What is common to all paths -- S0, the strike, 1 / M and the
// rounding of aw, which is close to 1 -- is applied in FP64 at the path's end.
template <bool CONTROL>
__device__ __forceinline__ void asia_path_f32(const AsiaArgs& a, uint64_t p, double& pay,
                                              double& geo) {
    float S = 1.f, I = 0.f, Ic = 0.f, ls = 0.f, lsum = 0.f;  // S, I: in units of S0
    auto add = [&](float t) {  // Kahan: I += S t
        const float y = fmaf(S, t, -Ic);
        const float u = I + y;
        Ic = (u - I) - y;
        I = u;
    };
    auto control = [&](float e) {
        if (CONTROL) {
            ls += e;
            lsum += ls;
        }
    };
    const int nfull = a.M >> 2;
    for (int b = 0; b < nfull; ++b) {
        const pcf::U4 x = pcf::philox_block(a.seed, PCF_STREAM_ASIA, p, (uint32_t)b);
        float e[4];
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            float R, c, s;
            pcf::box_muller_polar_f32(h ? x.z : x.x, h ? x.w : x.y, R, c, s);
            R *= a.vol2f;
            e[2 * h] = fmaf(R, c, a.mu2f);
            e[2 * h + 1] = fmaf(R, s, a.mu2f);
        }
        float x1 = e[0], t = fmaf(a.bwf, e[0], a.awf);
        control(e[0]);
#pragma unroll
        for (int j = 1; j < 4; ++j) {
            t = fmaf(pcf::exp2_f32(x1), fmaf(a.bwf, e[j], a.awf), t);
            control(e[j]);
            x1 += e[j];
        }
        add(t);
        S *= pcf::exp2_f32(x1);
    }
    const int rem = a.M & 3;
    if (rem) {
        float z[4];
        pcf::normals4<float>(a.seed, PCF_STREAM_ASIA, p, (uint32_t)nfull, z);
        auto step = [&](float zj) {
            const float e = fmaf(a.vol2f, zj, a.mu2f);  // log2 of the step factor
            add(fmaf(a.bwf, e, a.awf));
            S *= pcf::exp2_f32(e);
            control(e);
        };
        step(z[0]);
        if (rem > 1) step(z[1]);
        if (rem > 2) step(z[2]);
    }
    pay = pcf::payoff<double>(a.avg32 * ((double)I - (double)Ic), a.E, a.pf);
    if (CONTROL) geo = pcf::payoff<double>(a.S0 * (double)pcf::exp2_f32(lsum * (float)a.invM), a.E, a.pf);
}

// SMALL: every step's exponent is within pcf::kExpSmall (the host's bound, see
// asia_prepare), so its exponential needs no reduction.
template <bool CONTROL, bool SMALL>
__device__ __forceinline__ void asia_path_f64(const AsiaArgs& a, uint64_t p, double& pay,
                                              double& geo) {
    double S = a.S0, I = 0.0, ls = 0.0, lsum = 0.0;
    auto step = [&](double z) {
        I += S * fma(a.a2, z, a.a1);
        const double e = fma(a.vol, z, a.mu);
        S *= SMALL ? pcf::exp_small(e) : pcf::exp_any(e);
        if (CONTROL) {
            ls += e;
            lsum += ls;
        }
    };
    const int nfull = a.M >> 2;
    for (int b = 0; b < nfull; ++b) {
        double z[4];
        pcf::normals4<double>(a.seed, PCF_STREAM_ASIA, p, (uint32_t)b, z);
        step(z[0]);
        step(z[1]);
        step(z[2]);
        step(z[3]);
    }
    const int rem = a.M & 3;
    if (rem) {
        double z[4];
        pcf::normals4<double>(a.seed, PCF_STREAM_ASIA, p, (uint32_t)nfull, z);
        for (int j = 0; j < rem; ++j) step(z[j]);  // (rolled: three copies of the body made the kernel spill)
    }
    pay = pcf::payoff<double>(I / (double)a.M, a.E, a.pf);
    if (CONTROL) geo = pcf::payoff<double>(a.S0 * exp(lsum / (double)a.M), a.E, a.pf);
}

// The production FP64 step of asia_path_f64 on the reference's draws z = dB/sqrt(dt).
__device__ __forceinline__ double asia_path_prod_host(const AsiaArgs& a, const double* __restrict__ w) {
    double S = a.S0, I = 0.0;
    for (int m = 0; m < a.M; ++m) {
        const double z = w[m] / a.sdt;
        I += S * fma(a.a2, z, a.a1);
        S *= exp(fma(a.vol, z, a.mu));
    }
    return pcf::payoff<double>(I / (double)a.M, a.E, a.pf);
}

// Verification: the reference's expression order, FP64, no contraction.
__device__ __forceinline__ double asia_path_ref(const AsiaArgs& a, const double* __restrict__ z) {
#pragma clang fp contract(off)
    double St = a.S0, I = 0.0;
    for (int m = 0; m < a.M; ++m) {
        const double dBi = z[m];
        I += St * (a.h_c1 + a.sigma * dBi / 2);
        St *= exp(a.h_mu + a.sigma * dBi);
    }
    const double v = a.pf * (I / (double)a.M - a.E);
    return v > 0.0 ? v : 0.0;
}

struct AsiaJob {
    AsiaArgs a;
    const double* hz;
    pcf::CSum* partials;
    unsigned int* counter;
    double* out;
    unsigned int first_block, nblk;
};
static_assert(sizeof(AsiaJob) <= kJobBytes, "job record exceeds its staging slot");

template <int MODE, bool CONTROL, bool SMALL>
__device__ __forceinline__ void asia_body(const AsiaArgs& a, const double* __restrict__ hz,
                                          pcf::CSum* __restrict__ partials,
                                          unsigned int* __restrict__ counter, double* __restrict__ out,
                                          unsigned int blk, unsigned int nblk, pcf::CSum* lds) {
    constexpr int K = CONTROL ? 4 : 2;
    double s = 0.0, s2 = 0.0, g = 0.0, g2 = 0.0;
    const int64_t stride = (int64_t)nblk * blockDim.x;
    for (int64_t p = (int64_t)blk * blockDim.x + threadIdx.x; p < a.N; p += stride) {
        double v, gv = 0.0;
        if constexpr (MODE == kFp32k) {
            asia_path_f32<CONTROL>(a, (uint64_t)p, v, gv);
        } else if constexpr (MODE == kFp64) {
            asia_path_f64<CONTROL, SMALL>(a, (uint64_t)p, v, gv);
        } else if constexpr (MODE == kHostProd) {
            v = asia_path_prod_host(a, hz + p * (int64_t)a.M);
        } else {
            v = asia_path_ref(a, hz + p * (int64_t)a.M);
        }
        s += v;
        s2 += v * v;
        if (CONTROL) {
            g += gv;
            g2 += gv * gv;
        }
    }
    pcf::Acc<K> acc, tot;
    acc.v[0] = {s, 0.0};
    acc.v[1] = {s2, 0.0};
    if (CONTROL) {
        acc.v[2 % K] = {g, 0.0};
        acc.v[3 % K] = {g2, 0.0};
    }
    if (pcf::grid_reduce<K>(acc, partials, counter, lds, tot, blk, nblk) && threadIdx.x == 0)
        pcf::write_moments<K / 2>(tot, a.N, out);
}

template <int MODE, bool CONTROL, bool SMALL>
__global__ __launch_bounds__(1024) void k_asia(const pcf::JobArgs<AsiaJob> args) {
    __shared__ pcf::CSum lds[16 * (CONTROL ? 4 : 2)];
    const AsiaJob J = pcf::job_of(args, blockIdx.x);
    asia_body<MODE, CONTROL, SMALL>(J.a, J.hz, J.partials, J.counter, J.out, blockIdx.x - J.first_block,
                             J.nblk, lds);
}

struct AsiaPrep {
    AsiaArgs a;
    int mode, B, nblk;
    bool control;
    bool small;  // FP64: the steps' exponents are within pcf::kExpSmall
    double disc;
};

int asia_prepare(pcf_ctx* ctx, const pcf_request& q, AsiaPrep& p) {
    const pcf_opts& o = q.opts;
    int st = pcf_check_common(ctx, q.S0, q.E, q.r, q.sigma, q.T, q.N, q.payoff_fun);
    if (st) return st;
    if ((st = pcf_check_opts(ctx, &o))) return st;
    const int M = q.M;
    if (M <= 0) return pcf_fail(ctx, PCF_ERR_INVALID_ARG, "M must be positive (M=%d)", M);
    const double dt = (double)q.T / (double)M;
    const double sdt = std::sqrt(dt);
    const double log2e = 1.4426950408889634;
    AsiaArgs& a = p.a;
    a = AsiaArgs{};
    a.S0 = q.S0;
    a.E = q.E;
    a.pf = q.payoff_fun;
    a.a1 = 1.0 + q.r * dt / 2;
    a.a2 = q.sigma * sdt / 2;
    a.mu = (q.r - 0.5 * q.sigma * q.sigma) * dt;
    a.vol = q.sigma * sdt;
    a.h_c1 = 1 + q.r * dt / 2;
    a.h_mu = (q.r - libm_pow(q.sigma, 2) / 2) * dt;
    a.sigma = q.sigma;
    const double bw = 0.5 / log2e;  // a2 / (vol log2(e))
    a.bwf = (float)bw;
    const double aw = a.a1 - bw * (a.mu * log2e);
    a.awf = (float)aw;
    a.avg32 = q.S0 / (double)M * (a.awf != 0.f ? aw / (double)a.awf : 1.0);
    a.mu2f = (float)(a.mu * log2e);
    a.vol2f = (float)(a.vol * log2e);
    a.invM = 1.0 / (double)M;
    a.sdt = sdt;
    a.N = q.N;
    a.M = M;
    a.seed = o.seed;
    if (o.rng == PCF_RNG_HOST && o.kernel_variant != 0 && o.kernel_variant != 1)
        return pcf_fail(ctx, PCF_ERR_INVALID_ARG, "mc_asia with host normals: kernel_variant 0 (reference "
                        "arithmetic) or 1 (production arithmetic), got %d", o.kernel_variant);
    p.mode = o.rng == PCF_RNG_HOST ? (o.kernel_variant == 1 ? kHostProd : kHost)
                                   : (o.precision == PCF_FP64 ? kFp64 : kFp32k);
    p.control = o.control != 0 && p.mode != kHost && p.mode != kHostProd;
    // |z| <= sqrt(2 * 33 ln 2) = 6.7639 for every Philox normal, so
    // |mu + vol z| <= |mu| + 6.77 vol (false for a NaN).
    p.small = p.mode == kFp64 && std::fabs(a.mu) + 6.77 * a.vol <= pcf::kExpSmall;
    int B = 256;
    // 0.66 ps a path-step (1.7 in FP64)
    int ipt = pcf_items_per_thread(q.N, B, ctx->cu_count, 1.0 + (p.mode == kFp32k ? 0.66 : 1.7) * M);
    pcf_tuned_shape(PCF_KIND_ASIA, p.mode, q.N, &B, &ipt);
    if (o.block_size) B = o.block_size;
    if (o.items_per_thread) ipt = o.items_per_thread;
    p.B = B;
    p.nblk = pcf_blocks_for(q.N, B, ipt);
    p.disc = std::exp(-q.r * q.T);
    return PCF_OK;
}

// Result record of one request from its 8 output doubles (write_moments:
// sum, sum of squares, mean, variance of the payoffs, then of the control).
void asia_result(const AsiaPrep& p, const double* h, int64_t N, int M, int B, int batch, const pcf_result& timing,
                 pcf_result& r) {
    // The reference returns exp(-r*T)*result/(double)N (src/mc_asia.cpp:39).
    r.price = p.disc * h[0] / (double)N;
    r.mean = h[2];
    r.variance = h[3];
    r.std_err = p.disc * std::sqrt(h[3] / (double)N);
    if (p.control) {
        r.control_price = p.disc * h[4] / (double)N;
        r.control_se = p.disc * std::sqrt(h[7] / (double)N);
    }
    r.n_paths = N;
    r.n_steps = M;
    r.kernel_ms = timing.kernel_ms;
    r.total_ms = timing.total_ms;
    // 14 algorithmic flops per path-step: normal 6, I update 2 FMAs (4),
    // S update FMA + exp + mul (4).  No HBM traffic in the Philox forms.
    r.flops = 14.0 * (double)N * (double)M;
    r.bytes = p.mode >= kHost ? 8.0 * (double)N * (double)M : 0.0;
    r.grid_blocks = p.nblk;
    r.block_size = B;
    r.batch_size = batch;
}

// The kernel of a prepared request (every request of a batch has the same).
void launch_asia(const AsiaPrep& p, unsigned int grid, hipStream_t s, const pcf::JobArgs<AsiaJob>& ja) {
    const dim3 g(grid), b((unsigned)p.B);
    if (p.mode == kFp32k) {
        if (p.control) k_asia<kFp32k, true, false><<<g, b, 0, s>>>(ja);
        else k_asia<kFp32k, false, false><<<g, b, 0, s>>>(ja);
    } else if (p.mode == kFp64 && p.small) {
        if (p.control) k_asia<kFp64, true, true><<<g, b, 0, s>>>(ja);
        else k_asia<kFp64, false, true><<<g, b, 0, s>>>(ja);
    } else if (p.mode == kFp64) {
        if (p.control) k_asia<kFp64, true, false><<<g, b, 0, s>>>(ja);
        else k_asia<kFp64, false, false><<<g, b, 0, s>>>(ja);
    } else if (p.mode == kHost) {
        k_asia<kHost, false, false><<<g, b, 0, s>>>(ja);
    } else {
        k_asia<kHostProd, false, false><<<g, b, 0, s>>>(ja);
    }
}

}  // namespace

uint64_t pcf_asia_batch_key(pcf_ctx* ctx, const pcf_request& q, int* status) {
    AsiaPrep p;
    *status = asia_prepare(ctx, q, p);
    if (*status) return 0;
    return pcf_make_batch_key(PCF_KIND_ASIA, p.mode, (p.control ? 1 : 0) + (p.small ? 2 : 0), p.B);
}

int pcf_asia_run(pcf_ctx* ctx, int n, const pcf_request* const* reqs, pcf_result* res, int* status) {
    if (n < 1 || n > kMaxBatch) return pcf_fail(ctx, PCF_ERR_INVALID_ARG, "batch size %d", n);
    PCF_HIP_CHECK(ctx, hipSetDevice(ctx->device));
    AsiaPrep prep[kMaxBatch];
    int live[kMaxBatch], nl = 0;
    for (int i = 0; i < n; ++i) {
        res[i] = pcf_result{};
        status[i] = asia_prepare(ctx, *reqs[i], prep[i]);
        if (status[i] == PCF_OK) live[nl++] = i;
    }
    if (nl == 0) return PCF_OK;
    const int mode = prep[live[0]].mode, B = prep[live[0]].B;
    const bool control = prep[live[0]].control, small = prep[live[0]].small;
    const int K = control ? 4 : 2;
    int64_t nparts = 0, nb = 0, nnorm = 0;
    for (int k = 0; k < nl; ++k) {
        const AsiaPrep& p = prep[live[k]];
        if (p.mode != mode || p.B != B || p.control != control || p.small != small)
            return pcf_fail(ctx, PCF_ERR_INVALID_ARG, "mixed batch keys");
        nparts += (int64_t)p.nblk * K;
        nb += p.nblk;
        if (p.mode >= kHost) nnorm += reqs[live[k]]->N * (int64_t)reqs[live[k]]->M;
    }
    if (nb > (1ll << 30)) return pcf_fail(ctx, PCF_ERR_INVALID_ARG, "batch too large");
    // A lone job on device normals is one launch; anything more is a sequence
    // that is timed by events.
    bool sequence = nl > 1 || nnorm > 0;
    int st = PCF_OK;
    if (sequence && (st = pcf_timing_begin(ctx))) return st;
    PCF_HIP_CHECK(ctx, ctx->partials.ensure((size_t)nparts * sizeof(pcf::CSum)));
    if (nnorm) PCF_HIP_CHECK(ctx, ctx->normals.ensure((size_t)nnorm * sizeof(double)));
    AsiaJob* jobs = (AsiaJob*)ctx->h_jobs;
    int64_t poff = 0, noff = 0;
    unsigned int boff = 0;
    for (int k = 0; k < nl; ++k) {
        const int i = live[k];
        const AsiaPrep& p = prep[i];
        AsiaJob& J = jobs[k];
        J.a = p.a;
        J.hz = nullptr;
        if (p.mode >= kHost) {
            const pcf_opts& o = reqs[i]->opts;
            const int64_t cnt = reqs[i]->N * (int64_t)reqs[i]->M;
            if (!o.host_normals || o.n_host_normals < cnt)
                return pcf_fail(ctx, PCF_ERR_INVALID_ARG, "need %lld host normals", (long long)cnt);
            double* dst = ctx->normals.as<double>() + noff;
            PCF_HIP_CHECK(ctx, hipMemcpyAsync(dst, o.host_normals, (size_t)cnt * sizeof(double),
                                              hipMemcpyHostToDevice, ctx->stream));
            J.hz = dst;
            noff += cnt;
        }
        J.partials = ctx->partials.as<pcf::CSum>() + poff;
        J.counter = ctx->counters.as<unsigned int>() + (size_t)k * pcf::kCounterWords;
        J.out = ctx->h_out_dev + (size_t)kOutPerJob * k;
        J.first_block = boff;
        J.nblk = (unsigned int)p.nblk;
        poff += (int64_t)p.nblk * K;
        boff += (unsigned int)p.nblk;
    }
    if (nl > 1)
        PCF_HIP_CHECK(ctx, hipMemcpyAsync(ctx->jobs.ptr, jobs, sizeof(AsiaJob) * nl, hipMemcpyHostToDevice, ctx->stream));
    const pcf::JobArgs<AsiaJob> ja{jobs[0], ctx->jobs.as<AsiaJob>(), nl};
    pcf_arm_results(ctx, nl);
    double work = 0.0;
    for (int k = 0; k < nl; ++k) work += (double)reqs[live[k]]->N * (double)reqs[live[k]]->M;
    std::unique_lock<std::mutex> order;  // held until the end event is recorded
    PCF_HIP_CHECK(ctx, pcf_after_persistent(ctx, mode == kFp32k ? work : kPersistentGateFp64 * work, &order));
    launch_asia(prep[live[0]], boff, ctx->stream, ja);
    PCF_HIP_CHECK(ctx, hipGetLastError());
    PCF_HIP_CHECK(ctx, hipEventRecord(ctx->ev_kend, ctx->stream));
    if (order.owns_lock()) order.unlock();
    pcf_result timing{};
    if ((st = pcf_wait_results(ctx, nl, control ? 8 : 4, ctx->stream, &timing.kernel_ms))) return st;
    timing.total_ms = timing.kernel_ms;
    if (sequence && (st = pcf_sequence_ms(ctx, ctx->ev_kend, &timing.total_ms))) return st;
    for (int k = 0; k < nl; ++k) {
        const int i = live[k];
        asia_result(prep[i], ctx->h_out + (size_t)kOutPerJob * k, reqs[i]->N, reqs[i]->M, B, nl, timing, res[i]);
    }
    return PCF_OK;
}

// ---- the no-allocation entry point -----------------------------------------
// pcf_mc_asia_noalloc runs the same kernels as pcf_mc_asia with every device
// buffer they need -- the per-block compensated partials, the arrival
// counters and the results -- in one file-scope device array, so a
// call allocates no device memory.  Kernel arguments and host code use the
// array's device address, obtained once per device with hipGetSymbolAddress.
namespace {

constexpr int kNoAllocMaxBlocks = 32768;  // grid blocks of one launch
constexpr size_t kNoAllocPartialsBytes = (size_t)kNoAllocMaxBlocks * 4 * sizeof(pcf::CSum);  // 2 MiB
constexpr size_t kNoAllocCounterOff = kNoAllocPartialsBytes;
constexpr size_t kNoAllocOutOff =
    kNoAllocCounterOff + (pcf::kCounterWords * sizeof(unsigned int) + 255) / 256 * 256;
constexpr size_t kNoAllocBytes = kNoAllocOutOff + 256;

__global__ void k_zero_words(unsigned int* __restrict__ p, int n) {
    for (int i = threadIdx.x; i < n; i += blockDim.x) p[i] = 0u;
}

}  // namespace

// The scratch array (2 MiB + 5 KiB per device, held until the process ends).
static __device__ __align__(256) unsigned char scratch[kNoAllocBytes];

namespace {

// Per device: the array's device address, and a lock that serialises the
// calls using it (each call returns only after its work is complete).
struct ScratchSlot {
    std::mutex mu;
    char* ptr = nullptr;
};
ScratchSlot& scratch_slot(int device) {
    static ScratchSlot slots[64];
    return slots[device & 63];
}

}  // namespace

extern "C" int pcf_mc_asia_noalloc(pcf_ctx* ctx, double S0, double E, double r, double sigma, double T,
                                   int64_t N, int32_t M, double payoff_fun, const pcf_opts* opts,
                                   pcf_result* res) {
    if (!ctx || !res) return PCF_ERR_INVALID_ARG;
    std::lock_guard<std::recursive_mutex> lk(ctx->mu);
    pcf_request q = pcf_make_request(PCF_KIND_ASIA, S0, E, r, sigma, T, N, payoff_fun, opts);
    q.M = M;
    *res = pcf_result{};
    if (q.opts.rng != PCF_RNG_PHILOX)
        return pcf_fail(ctx, PCF_ERR_INVALID_ARG, "pcf_mc_asia_noalloc draws Philox normals (host normals would "
                        "need a device buffer: use pcf_mc_asia)");
    if (q.opts.fp64_check)
        return pcf_fail(ctx, PCF_ERR_INVALID_ARG, "pcf_mc_asia_noalloc does not make the FP64 comparison run");
    if (ctx->device < 0 || ctx->device >= 64) return pcf_fail(ctx, PCF_ERR_NO_DEVICE, "device index");
    AsiaPrep p;
    int st = asia_prepare(ctx, q, p);
    if (st) return st;
    const int K = p.control ? 4 : 2;
    if ((size_t)p.nblk * K * sizeof(pcf::CSum) > kNoAllocPartialsBytes)
        return pcf_fail(ctx, PCF_ERR_INVALID_ARG,
                        "pcf_mc_asia_noalloc holds the partials of at most %zu blocks with %d sums (this launch "
                        "has %d blocks of %d threads): use pcf_mc_asia",
                        kNoAllocPartialsBytes / (K * sizeof(pcf::CSum)), K, p.nblk, p.B);
    PCF_HIP_CHECK(ctx, hipSetDevice(ctx->device));
    ScratchSlot& slot = scratch_slot(ctx->device);
    std::lock_guard<std::mutex> sl(slot.mu);
    if (!slot.ptr) {
        void* dp = nullptr;
        PCF_HIP_CHECK(ctx, hipGetSymbolAddress(&dp, HIP_SYMBOL(scratch)));
        slot.ptr = static_cast<char*>(dp);
    }
    char* const base = slot.ptr;
    unsigned int* const counter = reinterpret_cast<unsigned int*>(base + kNoAllocCounterOff);
    double* const dout = reinterpret_cast<double*>(base + kNoAllocOutOff);
    AsiaJob job{};
    job.a = p.a;
    job.hz = nullptr;
    job.partials = reinterpret_cast<pcf::CSum*>(base);
    job.counter = counter;
    job.out = dout;
    job.first_block = 0;
    job.nblk = (unsigned int)p.nblk;
    if ((st = pcf_timing_begin(ctx))) return st;
    // the arrival counters start at zero (a fill kernel: no memset node)
    k_zero_words<<<1, 256, 0, ctx->stream>>>(counter, pcf::kCounterWords);
    PCF_HIP_CHECK(ctx, hipGetLastError());
    PCF_HIP_CHECK(ctx, hipEventRecord(ctx->ev_kbeg, ctx->stream));
    launch_asia(p, (unsigned int)p.nblk, ctx->stream, pcf::JobArgs<AsiaJob>{job, nullptr, 1});
    PCF_HIP_CHECK(ctx, hipGetLastError());
    PCF_HIP_CHECK(ctx, hipEventRecord(ctx->ev_kend, ctx->stream));
    PCF_HIP_CHECK(ctx, hipEventRecord(ctx->ev_end, ctx->stream));
    PCF_HIP_CHECK(ctx, hipMemcpyAsync(ctx->h_out, dout, kOutPerJob * sizeof(double), hipMemcpyDeviceToHost,
                                      ctx->stream));
    PCF_HIP_CHECK(ctx, hipStreamSynchronize(ctx->stream));
    pcf_result timing{};
    float kms = 0.f, tms = 0.f;
    PCF_HIP_CHECK(ctx, hipEventElapsedTime(&kms, ctx->ev_kbeg, ctx->ev_kend));
    PCF_HIP_CHECK(ctx, hipEventElapsedTime(&tms, ctx->ev_begin, ctx->ev_end));
    timing.kernel_ms = kms;
    timing.total_ms = tms;
    asia_result(p, ctx->h_out, N, M, p.B, 1, timing, *res);
    return PCF_OK;
}

extern "C" int pcf_mc_asia(pcf_ctx* ctx, double S0, double E, double r, double sigma, double T,
                           int64_t N, int32_t M, double payoff_fun, const pcf_opts* opts,
                           pcf_result* res) {
    if (!ctx || !res) return PCF_ERR_INVALID_ARG;
    std::lock_guard<std::recursive_mutex> lk(ctx->mu);
    pcf_request q = pcf_make_request(PCF_KIND_ASIA, S0, E, r, sigma, T, N, payoff_fun, opts);
    q.M = M;
    const pcf_request* qp = &q;
    int status = PCF_OK;
    int st = pcf_asia_run(ctx, 1, &qp, res, &status);
    if (st || status) return st ? st : status;
    return pcf_apply_fp64_check(ctx, q, res);
}

// lattice.hip -- backward induction on the reference's binomial lattice.
// Reference: src/binom_vanilla_eur.cpp:5-39 (European) and
// src/binom_vanilla_amer.cpp:5-40 (American), on the beta tree of
// src/binom_embar.cpp:16-24.
//
// The reference sweeps level n = N-1 .. 0 over nodes i = 0 .. n:
//   European  v[i] = (p v[i+1] + q v[i]) / R
//   American  v[i] = max((p v[i+1] + q v[i]) / R, payoff(S0 u^i d^(n-i), E))
// from the leaves v[i] = max((S0 u^i d^(N-i) - E) pf, 0).  Every node depends
// only on its two children, so any schedule that forms each node from its
// children with the same operations reproduces the reference's bits: FP64,
// no contraction, IEEE division, std::max's "a < b ? b : a", and u^i, d^k
// from tables made on the host with glibc pow (the call the reference makes).
//
// Two schedules.  Up to 98304 levels American and 262144 European (the waves
// that are resident together), and for parameters within the bounds of
// lat_plan, one launch makes the sweep (k_lat_flow).  Beyond those,
// one launch advances K levels (LatTile).  Each wavefront owns
// Wout = 64 R - K output nodes of the last of them and holds the 64 R nodes
// of the first level it needs in registers, R consecutive nodes per lane.
// A level forms every node from itself and its right neighbour; the right
// neighbour of a lane's last node is the next lane's first node, one DPP
// wave shift away.  The span of valid nodes shrinks by one per level, so
// after K levels the wave's first Wout nodes are exact and the waves need no
// barrier or LDS at all.  The K-wide right edge a wave forms is also formed
// by its neighbour, with identical values.  Device data: two level rows of
// N + 1 doubles and the tables u^i, d^k (i, k = 0..N), kept per context for
// the last (u, d, N).
#include <algorithm>
#include <atomic>
#include <cmath>
#include <cstring>
#include <type_traits>
#include <vector>

#include "pcf_internal.hpp"

namespace {

constexpr int kLatThreads = 256;
constexpr int64_t kLatMaxN = (int64_t)1 << 21;

// Tile shape per exercise style: R nodes per lane, K levels per launch, Wout =
// 64 R - K output nodes per wave and launch.  A level costs a wave about R
// node updates in sequence, and a large lattice holds only ~n/Wout waves for
// the 1024 SIMDs, so small tiles run faster per level than they lose to
// redundant edges and extra launches.  Measured over 46 lattices (N = 513 ..
// 10^5) against R = 4, K = 128: American R = 1, K = 32 171.5 -> 104.9 ms in
// total; European R = 2, K = 64 69.3 -> 51.5 ms; bits unchanged.
template <bool AMER>
struct LatTile {
    static constexpr int R = AMER ? 1 : 2;
    static constexpr int K = AMER ? 32 : 64;
    static constexpr int Wout = 64 * R - K;
    static_assert(Wout > 0, "a wave must keep some exact output nodes");
};

struct LatParams {
    double S0, E, pf, p, q, R;
    int64_t N;
};

// std::max(a, b) as the reference calls it.
__device__ __forceinline__ double ref_max(double a, double b) { return (a < b) ? b : a; }

// payoff(St, E, pf) of include/common.h:56-60: max(pf * (St - E), 0).
__device__ __forceinline__ double ref_payoff(double St, double E, double pf) {
#pragma clang fp contract(off)
    return ref_max(pf * (St - E), 0.0);
}

template <bool AMER>
__global__ __launch_bounds__(kLatThreads) void k_lat_leaves(LatParams P, const double* __restrict__ up,
                                                            const double* __restrict__ dn, double* __restrict__ v) {
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i <= P.N;
         i += (int64_t)gridDim.x * blockDim.x) {
#pragma clang fp contract(off)
        const double S = P.S0 * up[i] * dn[P.N - i];
        // European: std::max(((S0*pow(u,i)*pow(d,N-i))-E)*payoff_fun, 0.0)
        // (src/binom_vanilla_eur.cpp:29); American: payoff(...) (src/binom_vanilla_amer.cpp:29).
        v[i] = AMER ? ref_payoff(S, P.E, P.pf) : ref_max((S - P.E) * P.pf, 0.0);
    }
}

// Right neighbour across lanes: lane l receives lane l+1's value (DPP
// wave_shl:1; lane 63 receives 0, which only ever reaches nodes past the
// wave's valid span).  FP64 as two 32-bit halves.
__device__ __forceinline__ double from_next_lane(double v) {
    const uint64_t u = __builtin_bit_cast(uint64_t, v);
    const uint32_t lo = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)(uint32_t)u, 0x130, 0xF, 0xF, false);
    const uint32_t hi = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)(uint32_t)(u >> 32), 0x130, 0xF, 0xF, false);
    return __builtin_bit_cast(double, ((uint64_t)hi << 32) | lo);
}

// Levels n0-1 .. n0-K from level n0 (vin) into vout.  The grid covers the
// n0-K+1 nodes of the last level with waves of LatTile::Wout outputs; the
// host keeps K <= LatTile::K.  Every lane runs every level (no early exit), so the
// cross-lane reads always see active lanes.
template <bool AMER>
__global__ __launch_bounds__(kLatThreads) void k_lat_steps(LatParams P, const double* __restrict__ up,
                                                           const double* __restrict__ dn,
                                                           const double* __restrict__ vin, double* __restrict__ vout,
                                                           int64_t n0, int K) {
    const int lane = threadIdx.x & 63;
    const int64_t wave = ((int64_t)blockIdx.x * blockDim.x + threadIdx.x) >> 6;
    constexpr int kR = LatTile<AMER>::R, kWout = LatTile<AMER>::Wout;
    const int64_t j0 = wave * kWout + (int64_t)lane * kR;  // this lane's first node
    // v: node values; AMER: u = u^j (fixed per node) and d = d^(n-j) for the
    // level n being formed.  d^(n-j) of node j at level n-1 is d^(n-(j+1)) of
    // node j+1 at level n, so d shifts one node left per level (the last node
    // of a lane takes the next lane's first); only lane 63's last node takes a
    // value it does not own, and that node is past the valid span already.
    double v[kR], u[kR], d[kR];
#pragma unroll
    for (int r = 0; r < kR; ++r) {
        const int64_t j = j0 + r;
        v[r] = j <= n0 ? vin[j] : 0.0;
        if constexpr (AMER) {
            u[r] = j <= n0 ? up[j] : 0.0;
            d[r] = j <= n0 - 1 ? dn[n0 - 1 - j] : 0.0;
        }
    }
    for (int s = 1; s <= K; ++s) {
        const int64_t n = n0 - s;
        const double nb = from_next_lane(v[0]);
        double w[kR];
#pragma unroll
        for (int r = 0; r < kR; ++r) {
#pragma clang fp contract(off)
            const double right = r + 1 < kR ? v[r + 1 < kR ? r + 1 : 0] : nb;
            w[r] = (P.p * right + P.q * v[r]) / P.R;
            if constexpr (AMER) {
                const int64_t j = j0 + r;
                if (j <= n) {
                    const double S = P.S0 * u[r] * d[r];
                    w[r] = ref_max(w[r], ref_payoff(S, P.E, P.pf));
                }
            }
        }
#pragma unroll
        for (int r = 0; r < kR; ++r) v[r] = w[r];
        if constexpr (AMER) {
            const double dnext = from_next_lane(d[0]);
#pragma unroll
            for (int r = 0; r + 1 < kR; ++r) d[r] = d[r + 1];
            d[kR - 1] = dnext;
        }
    }
    // The wave's first kWout nodes of level n0-K (and nothing past it).
    const int64_t wend = wave * kWout + kWout;
#pragma unroll
    for (int r = 0; r < kR; ++r) {
        const int64_t j = j0 + r;
        if (j < wend && j <= n0 - K) vout[j] = v[r];
    }
}

// ---- one launch -----------------------------------------------------------
// The launch-per-K-levels schedule above spends most of a level's time between
// launches and in the division: 10^4 levels of an American lattice took 313
// launches of 5.9 us, 32 levels each, for 50 node updates per lane.  Here one
// launch makes the whole sweep.  A wave owns 32 nodes, holds the 32 right of
// them as well, and advances 32 levels on its own as above; then it publishes
// its 32 values and takes the next 32 from the wave on its right.
// Dependencies only point right, so no barrier is needed, and a wave waits
// for its neighbour alone: three of four times through LDS (four waves of
// neighbours share a block, one to a SIMD), else through memory.  (With one
// wave to a block, and every exchange through memory, 10^4 levels took 770 us,
// and 600 with 16 owned nodes and 48 levels to an exchange.)
//
// Exchange.  A value travels as two 64-bit words, each half of its bits beside
// a tag that no earlier exchange used, so a reader polls the words themselves
// and nothing is ever cleared.  Chunk c (of 32 levels) goes to slot
// c mod kLatRing; before a wave overwrites a slot it checks that its reader,
// the wave on its left, has taken the slot's last values (a progress word,
// polled together with the values).
//
// Division.  x / R by a constant: q0 = x y, q = q0 + (x - q0 R) y with y the
// rounded 1 / R.  With exact residuals the corrected quotient is the rounded
// one if q0 is within an ulp of x / R (Markstein), which holds if |1 - y R| <=
// 2^-54; otherwise (about half of the R < 1) a second correction is made.
// Residuals are exact while no product underflows, so a wave looks at its
// values before each 32 levels: with every nonzero one at least LatFlow::lo
// (the host chooses it so that 32 levels of p, q and 1 / R cannot bring it
// below 2^-900) it divides so; with every one below 2^-200 it divides x 2^128
// and lets v_div_fmas scale the last step back, which rounds once, also into
// the subnormals; else it uses the division.  (10^9 random and midpoint
// numerators for each of 24 R, normal and subnormal results: no difference
// from x / R.)
// American put, 10^4 levels: 1871 -> 536 us (54 ns a level), European 1170 ->
// 390; 3000 levels 530 -> 160 us; 98304 23.2 -> 7.4 ms.  What bounds it now is
// the issue of one wave's 12 dependent operations a level (5.5 cycles each
// with one wave to a SIMD) and the exchanges, about 0.4 us per 32 levels.
constexpr int kLatK = 32;     // levels per exchange, and nodes a wave owns
constexpr int kLatWaves = 4;  // waves per block
constexpr int kLatRing = 8;
constexpr int kLatMaxBlocks = 4096;
constexpr size_t kLatWordBytes = (kLatMaxBlocks + 32) * sizeof(unsigned int);  // progress words, error word, arrivals

struct LatFlow {
    LatParams P;
    double y, lo;          // RN(1 / R); smallest nonzero value of the plain division
    const double* up;
    const double* dn;
    unsigned long long* ring;  // [kLatRing][blocks][kLatK][2]: the first waves' values
    unsigned int* prog;        // [blocks]: tag of the last chunk the last wave read
    unsigned int* err;
    unsigned int* arrived;     // blocks of all launches so far
    unsigned int all;          // and what it comes to when this one's are all resident
    double* out;           // price, 1 if a wait gave up, clock words; kOutResident
    unsigned int base;     // tag of chunk c is base + c + 1
    int waves;
    int by_xcd;            // neighbouring blocks on one XCD: kInTurn or kById, or 0
    unsigned int check;    // a wait looks at the clock and the error word once per check + 1 polls
    unsigned long long patience;  // clock ticks after which a wait gives up
};

enum { kInTurn = 1, kById = 2 };
enum { kDivPlain = 0, kDivTiny = 1, kDivIeee = 2 };
template <int CLASS, int STEPS>
__device__ __forceinline__ double lat_divide(double x, double R, double y, double y128) {
#pragma clang fp contract(off)
    if constexpr (CLASS == kDivIeee) return x / R;
    const double t = CLASS == kDivTiny ? x * 0x1p128 : x;
    double q = x * (CLASS == kDivTiny ? y128 : y);
    if constexpr (STEPS == 2) q = fma(fma(-q, R, t), y, q);
    const double r = fma(-q, R, t);
    if constexpr (CLASS == kDivTiny) return __builtin_amdgcn_div_fmas(r, y, q, true);
    return fma(r, y, q);
}

// from_next_lane without the zero it puts into a fresh register: lane 63 reads 0.
__device__ __forceinline__ double next_lane(double v) {
    const uint64_t u = __builtin_bit_cast(uint64_t, v);
    const uint32_t lo = (uint32_t)__builtin_amdgcn_mov_dpp((int)(uint32_t)u, 0x130, 0xF, 0xF, true);
    const uint32_t hi = (uint32_t)__builtin_amdgcn_mov_dpp((int)(uint32_t)(u >> 32), 0x130, 0xF, 0xF, true);
    return __builtin_bit_cast(double, ((uint64_t)hi << 32) | lo);
}

// What a wait stands before it gives up: blocks of this grid may wait for CUs
// that other kernels hold (pcf_launch_lattice).  Waits of a sweep that runs
// are microseconds (the longest sweep takes 28 ms as a whole), and a sweep that
// gave up is made by the other schedule, which needs no block beside another.
// The device clock bounds every wait alike: a poll of LDS takes a tenth of a
// poll of memory.
constexpr double kLatPatienceMs = 20.0;
constexpr unsigned int kLatCheck = 63;

// Testing hook: 1 for waits that give up at their first miss, 2 for blocks in
// the order of their numbers.
std::atomic<int>& lat_debug() {
    static std::atomic<int> bits{0};
    return bits;
}

template <int SCOPE, typename T>
__device__ __forceinline__ T lat_read(const T* p) {
    return __hip_atomic_load(p, __ATOMIC_RELAXED, SCOPE);
}
template <int SCOPE, typename T>
__device__ __forceinline__ void lat_write(T* p, T v) {
    __hip_atomic_store(p, v, __ATOMIC_RELAXED, SCOPE);
}

template <bool AMER, int STEPS>
__global__ __launch_bounds__(64 * kLatWaves) void k_lat_flow(const LatFlow a) {
    constexpr int K = kLatK;
    constexpr int kMem = __HIP_MEMORY_SCOPE_AGENT, kLds = __HIP_MEMORY_SCOPE_WORKGROUP;
    __shared__ double dsw[kLatWaves][64 + K];
    __shared__ unsigned long long exch[kLatRing][kLatWaves][2][K];
    __shared__ unsigned int lprog[kLatWaves];
    const int lane = threadIdx.x & 63;
    const int i = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));  // wave of the block
    // Blocks go to the 8 XCDs in turn.  With few of them, neighbours are put on
    // one XCD (the grid is then a multiple of 8, and the blocks past the last
    // wave leave): 10^4 levels 483 -> 393 us European, 620 -> 536 American; from
    // 157 blocks (20000 levels) on that is slower (American 1.36 -> 1.59 ms).
    // Which XCD the first block goes to depends on what its hardware queue ran
    // before; where the sweep's order wrapped from XCD 7 to 0 on its way, 10^4
    // levels took 580-630 us.  So the XCD's own number orders them.  (Were two
    // blocks of an XCD not 8 apart, one place would be empty and another held
    // twice: the tagged words stay right, the waits for the empty place give up.)
    const int per = (int)gridDim.x / 8;
    const int xcd = a.by_xcd == kById ? (int)__builtin_amdgcn_s_getreg((3 << 11) | 20)  // XCC_ID, bits 0..3
                                      : (int)(blockIdx.x % 8);
    const int blk = a.by_xcd ? xcd * per + (int)(blockIdx.x / 8) : (int)blockIdx.x;
    const int w = blk * kLatWaves + i;
    if (w == 0 && lane == 0) pcf::stamp(a.out + pcf::kOutStart);
    unsigned int arrived = 0;  // (looked at below, when the first loads are waited for)
    if (threadIdx.x == 0) arrived = __hip_atomic_fetch_add(a.arrived, 1u, __ATOMIC_RELAXED, kMem) + 1u;
    // no tag may be found before it is written
    for (int t = threadIdx.x; t < kLatRing * kLatWaves * 2 * K; t += blockDim.x) (&exch[0][0][0][0])[t] = 0;
    if (threadIdx.x < kLatWaves) lprog[threadIdx.x] = a.base;
    __syncthreads();
    if (w >= a.waves) {
        if (arrived == a.all) pcf::stamp(a.out + kOutResident);
        return;
    }
    double* const ds = dsw[i];
    const int N = (int)a.P.N;
    const int j = w * K + lane;
    const double p = a.P.p, q = a.P.q, R = a.P.R, y = a.y, y128 = a.y * 0x1p128;
    // pf (S - E) = (pf S) - (pf E) exactly (pf = +-1), and pf S = (pf S0 u) d.
    const double Epf = a.P.pf * a.P.E;
    double su, v;
    {
#pragma clang fp contract(off)
        su = a.P.pf * (a.P.S0 * a.up[j < N ? j : N]);
        const double leaf = su * a.dn[j < N ? N - j : 0] - Epf;
        v = j <= N ? ref_max(leaf, 0.0) : 0.0;
    }
    if (arrived == a.all) pcf::stamp(a.out + kOutResident);
    const bool last_wave = i == kLatWaves - 1, first_wave = i == 0;
    const int blocks = gridDim.x;
    bool gave_up = false;
    int n0 = N;
    // American: pf S of this lane's node at the K levels of a chunk, which
    // does not depend on the values.  A sweep is a chain of dependent
    // operations with issue slots to spare, so it makes the next chunk's on
    // its way, each in the place of the one it has just used.
    // ds: the next chunk's d^(n0 - 1 - w K - t), t = lane + s at step s, loaded
    // a chunk before that.  (A wave's LDS accesses execute in order.)
    double pfS[AMER ? K : 1];
    double d0 = 0.0, d1 = 0.0;
    auto load_d = [&](int n) {
        const int t0 = n - 1 - w * K - lane, t1 = t0 - 64;
        d0 = a.dn[t0 > 0 ? t0 : 0];
        d1 = a.dn[t1 > 0 ? t1 : 0];
    };
    auto stage_d = [&] {
        __builtin_amdgcn_wave_barrier();
        ds[lane] = d0;
        if (lane < K) ds[64 + lane] = d1;
        __builtin_amdgcn_wave_barrier();
    };
    if constexpr (AMER) {
        load_d(n0);
        stage_d();
#pragma unroll
        for (int s = 0; s < K; ++s) pfS[s] = su * ds[lane + s];
        load_d(n0 - K);
    }
    for (int c = 0;; ++c) {
        const int Kc = n0 < K ? n0 : K;
        if constexpr (AMER) {
            stage_d();
            load_d(n0 - 2 * K);
        }
        if (c > 0) {
            // Values of chunk c - 1 from the right; the reader on the left has
            // taken chunk c - kLatRing, whose slot chunk c will use.
            const unsigned int tag = a.base + (unsigned int)c;
            const unsigned int taken = tag - kLatRing + 1;
            const bool needv = lane >= K && j <= n0;
            const bool needp = lane == 0 && w > 0 && c >= kLatRing;
            const int sl = (c - 1) % kLatRing, src = lane & (K - 1);
            auto await = [&](auto from_mem, auto left_mem) {
                constexpr bool MEM = decltype(from_mem)::value, LEFT_MEM = decltype(left_mem)::value;
                const unsigned long long *rh, *rl;
                if constexpr (MEM) {
                    rh = a.ring + 2 * ((size_t)(sl * blocks + (blk + 1 < blocks ? blk + 1 : blk)) * K + src);
                    rl = rh + 1;
                } else {
                    rh = &exch[sl][i + 1][0][src];
                    rl = &exch[sl][i + 1][1][src];
                }
                const unsigned int* pp;
                if constexpr (LEFT_MEM) pp = a.prog + (blk > 0 ? blk - 1 : 0);
                else pp = &lprog[i - 1];
                unsigned long long since = 0;
                for (unsigned int it = 1;; ++it) {
                    const unsigned long long h = lat_read<MEM ? kMem : kLds>(rh);
                    const unsigned long long l = lat_read<MEM ? kMem : kLds>(rl);
                    const unsigned int g = lat_read<LEFT_MEM ? kMem : kLds>(pp);
                    const bool miss = (needv && ((unsigned int)(h >> 32) != tag || (unsigned int)(l >> 32) != tag)) ||
                                      (needp && (int)(g - taken) < 0);
                    if (needv) v = __builtin_bit_cast(double, (h << 32) | (l & 0xffffffffull));
                    if (!__any(miss)) break;
                    if constexpr (MEM) __builtin_amdgcn_s_sleep(2);
                    if ((it & a.check) == 0) {
                        const unsigned long long now = wall_clock64();
                        if (since == 0) since = now;
                        if (now - since >= a.patience || pcf::fetch_u32(a.err) != 0u) {
                            gave_up = true;
                            break;
                        }
                    }
                }
            };
            using Yes = std::true_type;
            using No = std::false_type;
            if (last_wave) await(Yes{}, No{});
            else if (first_wave) await(No{}, Yes{});
            else await(No{}, No{});
            if (gave_up) {
                if (lane == 0) atomicOr(a.err, 1u);
                break;
            }
            if (lane == 0) {
                if (last_wave) lat_write<kMem>(a.prog + blk, tag);
                else lat_write<kLds>(&lprog[i], tag);
            }
            v = j <= n0 ? v : 0.0;
        }
        const bool plain = !__any(v > 0.0 && v < a.lo);
        const bool tiny = !__any(v >= 0x1p-200);
        auto step = [&](auto cls, int s) {
#pragma clang fp contract(off)
            constexpr int CLASS = decltype(cls)::value;
            const double x = p * next_lane(v) + q * v;
            const double val = lat_divide<CLASS, STEPS>(x, R, y, y128);
            if constexpr (!AMER) {
                v = val;
            } else {
                // max(val, max(pf (S - E), 0)), val >= 0
                const double pay = pfS[s] - Epf;
                v = CLASS == kDivIeee ? ref_max(val, ref_max(pay, 0.0)) : fmax(val, pay);
                pfS[s] = su * ds[lane + s];
            }
        };
        using Plain = std::integral_constant<int, kDivPlain>;
        using Tiny = std::integral_constant<int, kDivTiny>;
        using Ieee = std::integral_constant<int, kDivIeee>;
        if (Kc < K) {  // the last levels
#pragma unroll
            for (int s = 0; s < K; ++s)
                if (s < Kc) step(Ieee{}, s);
        } else if (plain) {
#pragma unroll
            for (int s = 0; s < K; ++s) step(Plain{}, s);
        } else if (tiny) {
#pragma unroll
            for (int s = 0; s < K; ++s) step(Tiny{}, s);
        } else {
#pragma unroll
            for (int s = 0; s < K; ++s) step(Ieee{}, s);
        }
        n0 -= Kc;
        if (n0 == 0) break;
        if (lane < K && j <= n0 && w > 0) {
            const uint64_t b = __builtin_bit_cast(uint64_t, v);
            const unsigned long long t = (unsigned long long)(a.base + (unsigned int)c + 1u) << 32;
            const int sl = c % kLatRing;
            if (first_wave) {
                unsigned long long* const wp = a.ring + 2 * ((size_t)(sl * blocks + blk) * K + lane);
                lat_write<kMem>(wp, t | (b >> 32));
                lat_write<kMem>(wp + 1, t | (b & 0xffffffffull));
            } else {
                lat_write<kLds>(&exch[sl][i][0][lane], t | (b >> 32));
                lat_write<kLds>(&exch[sl][i][1][lane], t | (b & 0xffffffffull));
            }
        }
        // no node of the next K levels' end is this wave's
        if (w * K > n0 - (n0 < K ? n0 : K)) break;
    }
    if (w == 0 && lane == 0) {
        pcf::to_host(a.out, v);
        pcf::to_host(a.out + 1, gave_up || pcf::fetch_u32(a.err) != 0u ? 1.0 : 0.0);
        pcf::stamp(a.out + pcf::kOutEnd);
    }
}

// The one-launch form of a request, or launch == nullptr where it does not
// take it: parameters for which the bounds behind its division do not hold,
// or more waves than can be resident together.
struct LatPlan {
    const void* launch = nullptr;
    int waves = 0, blocks = 0;
    int capacity = 0;  // blocks of any of the four kernels that are resident together
    int by_xcd = 0;
    double lo = 0.0;
};

LatPlan lat_plan(pcf_ctx* ctx, const LatParams& P, double u, double d, bool american) {
    LatPlan pl;
    const double big = 0x1p600, small = 0x1p-700;
    const double un = libm_pow(u, (double)P.N), dN = libm_pow(d, (double)P.N);
    // Prices within [2^-700, 2^600] (E may be 0), probabilities inside (0, 1),
    // nodes that differ: a nonzero payoff is then at least 2^-752, no sum of
    // values overflows, and no value is negative.
    const bool sane = u - d > 1e-10 && P.p > 0.0 && P.q > 0.0 && P.p < 1.0 && P.q < 1.0 && P.R > 0.5 && P.R < 2.0 &&
                      P.S0 > 0.0 && P.S0 * un < big && P.S0 * dN > small && P.S0 < big && P.S0 > small &&
                      std::fabs(P.E) < big && (P.E == 0.0 || std::fabs(P.E) > small);
    if (!sane) return pl;
    pl.waves = P.N > kLatK ? (int)((P.N - kLatK) / kLatK) + 1 : 1;
    pl.blocks = (pl.waves + kLatWaves - 1) / kLatWaves;
    // By the XCDs' numbers where the device is all 8 of them (32 CUs each), until
    // a wait of such a sweep has given up.
    const bool in_turn = ctx->cu_count != 256 || ctx->lat_in_turn || (lat_debug().load(std::memory_order_relaxed) & 2);
    if (pl.blocks > 1 && pl.blocks <= 128) pl.by_xcd = in_turn ? kInTurn : kById;
    if (pl.by_xcd) pl.blocks = (pl.blocks + 7) / 8 * 8;
    // 32 levels scale a value by at least (min(p, q) / R)^32.
    const double m = std::min(P.p, P.q) / P.R * (1.0 - 1e-9);
    pl.lo = 0x1p-900 / std::pow(m, (double)kLatK);
    if (!(pl.lo < 0x1p-755)) return pl;
    const double y = 1.0 / P.R;
    const int steps = std::fabs(std::fma(-y, P.R, 1.0)) <= 0x1p-54 ? 1 : 2;
    const void* const fns[2][2] = {{(const void*)k_lat_flow<false, 1>, (const void*)k_lat_flow<false, 2>},
                                   {(const void*)k_lat_flow<true, 1>, (const void*)k_lat_flow<true, 2>}};
    const void* const fn = fns[american][steps - 1];
    int nb = 0;
    if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&nb, fn, 64 * kLatWaves, 0) != hipSuccess) return pl;
    if (pl.blocks > std::min(kLatMaxBlocks, nb * ctx->cu_count)) return pl;
    for (const auto& f : fns)
        for (const void* g : f) {
            int n = 0;
            if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&n, g, 64 * kLatWaves, 0) != hipSuccess) return pl;
            nb = std::min(nb, n);
        }
    pl.capacity = nb * ctx->cu_count;
    pl.launch = fn;
    return pl;
}

// v_ij[0], returned as is (src/binom_vanilla_eur.cpp:38), and the figures of the sweep.
void lat_result(pcf_result& r, double price, int64_t N, bool american, int launches, int threads) {
    r.price = r.mean = price;
    r.n_paths = 1;
    r.n_steps = N;
    // Node updates: (N+1)(N+2)/2 - 1 over the sweep; 4 flops each European
    // (2 mul, add, div), 9 American (+ 2 mul for S, sub, mul, 2 max).
    const double nodes = 0.5 * (double)(N + 1) * (double)(N + 2) - 1.0;
    r.flops = nodes * (american ? 9.0 : 4.0);
    r.bytes = 0.0;
    r.grid_blocks = launches;
    r.block_size = threads;
    r.batch_size = 1;
}

}  // namespace

extern "C" int pcf_binom_vanilla(pcf_ctx* ctx, double S0, double E, double r, double sigma, double T, int64_t N,
                                 double payoff_fun, int32_t american, const pcf_opts* opts_in, pcf_result* res) {
    if (!ctx || !res) return PCF_ERR_INVALID_ARG;
    std::lock_guard<std::recursive_mutex> lk(ctx->mu);
    pcf_opts o = pcf_opts_or_default(opts_in);
    int st = pcf_check_common(ctx, S0, E, r, sigma, T, N, payoff_fun);
    if (st) return st;
    if ((st = pcf_check_opts(ctx, &o))) return st;
    if (N > kLatMaxN)
        return pcf_fail(ctx, PCF_ERR_INVALID_ARG, "lattice N=%lld exceeds %lld", (long long)N, (long long)kLatMaxN);
    PCF_HIP_CHECK(ctx, hipSetDevice(ctx->device));
    *res = pcf_result{};

    // Tree parameters exactly as src/binom_vanilla_eur.cpp:16-24 (host, glibc).
    const double dt = (double)T / (double)N;
    const double beta = 0.5 * (std::exp(-r * dt) + std::exp((r + libm_pow(sigma, 2)) * dt));
    const double u = beta + std::sqrt(libm_pow(beta, 2) - 1);
    const double d = beta - std::sqrt(libm_pow(beta, 2) - 1);
    const double R = std::exp(r * dt);
    const double p = (R - d) / (u - d);
    const double q = 1 - p;
    const LatParams P{S0, E, payoff_fun, p, q, R, N};

    // Tables u^i, d^k (i, k = 0..N) -- resident for the last (u, d, N).
    const size_t row = (size_t)N + 1;
    uint64_t key[3];
    std::memcpy(&key[0], &u, 8);
    std::memcpy(&key[1], &d, 8);
    key[2] = (uint64_t)N;
    PCF_HIP_CHECK(ctx, ctx->lattice.ensure(4 * row * sizeof(double)));
    double* up = ctx->lattice.as<double>();
    double* dn = up + row;
    double* A = dn + row;
    double* B = A + row;
    bool fresh = std::memcmp(key, ctx->lattice_key, sizeof key) != 0 || ctx->lattice_ptr != (void*)up;
    const size_t tab_bytes = 2 * row * sizeof(double);
    if (fresh) {
        if (ctx->h_lat_bytes < tab_bytes) {
            if (ctx->h_lat) PCF_HIP_CHECK(ctx, hipHostFree(ctx->h_lat));
            ctx->h_lat = nullptr;
            ctx->h_lat_bytes = 0;
            PCF_HIP_CHECK(ctx, hipHostMalloc((void**)&ctx->h_lat, tab_bytes, 0));
            ctx->h_lat_bytes = tab_bytes;
        }
        ctx->lattice_ptr = nullptr;  // until the copy is made
        for (size_t i = 0; i < row; ++i) {
            ctx->h_lat[i] = libm_pow(u, (double)i);        // pow(u,i), src/binom_vanilla_eur.cpp:29
            ctx->h_lat[row + i] = libm_pow(d, (double)i);  // pow(d,N-i)
        }
    }
    // The copy goes before the kernels on their stream; the call returns after
    // them, so the staging is free again by then.
    auto upload = [&](hipStream_t s) -> hipError_t {
        if (!fresh) return hipSuccess;
        const hipError_t e = hipMemcpyAsync(up, ctx->h_lat, tab_bytes, hipMemcpyHostToDevice, s);
        if (e == hipSuccess) {
            std::memcpy(ctx->lattice_key, key, sizeof key);
            ctx->lattice_ptr = (void*)up;
        }
        return e;
    };

    LatPlan plan = lat_plan(ctx, P, u, d, american != 0);
    if (plan.launch) {
        const size_t bytes = kLatWordBytes + 16 * (size_t)kLatRing * plan.blocks * kLatK;
        const uint32_t chunks = (uint32_t)((N + kLatK - 1) / kLatK);
        // tags never repeat while the buffer lives; it starts again from zero
        // when they would
        if (ctx->lat_epoch > 0x7fffffffu - chunks || ctx->lat_ring.bytes < bytes) {
            ctx->lat_ring.release();
            ctx->lat_epoch = 0;
        }
        if (!ctx->lat_ring.ptr) ctx->lat_arrived = 0;
        PCF_HIP_CHECK(ctx, ctx->lat_ring.ensure(bytes, true));
        LatFlow f{};
        f.P = P;
        f.y = 1.0 / R;
        f.lo = plan.lo;
        f.up = up;
        f.dn = dn;
        // The progress words have a place of their own, so that no launch
        // finds an earlier one's values there.
        f.prog = ctx->lat_ring.as<unsigned int>();
        f.err = f.prog + kLatMaxBlocks;
        f.arrived = f.err + 16;
        f.all = ctx->lat_arrived += (uint32_t)plan.blocks;
        f.ring = (unsigned long long*)(ctx->lat_ring.as<char>() + kLatWordBytes);
        f.out = ctx->h_out_dev;
        f.base = ctx->lat_epoch;
        f.waves = plan.waves;
        f.by_xcd = plan.by_xcd;
        const bool impatient = (lat_debug().load(std::memory_order_relaxed) & 1) != 0;
        f.check = impatient ? 0 : kLatCheck;
        f.patience = impatient ? 0 : (unsigned long long)(kLatPatienceMs * ctx->clock_khz);
        ctx->lat_epoch += chunks + 1;
        pcf_arm_results(ctx, 1);
        PCF_HIP_CHECK(ctx, pcf_launch_lattice(ctx, plan.blocks, plan.capacity, [&](hipStream_t s) -> hipError_t {
            if (fresh) {
                hipError_t e = hipEventRecord(ctx->ev_begin, s);
                if (e == hipSuccess) e = upload(s);
                if (e != hipSuccess) return e;
            }
            void* args[] = {&f};
            return hipLaunchKernel(plan.launch, dim3((unsigned)plan.blocks), dim3(64 * kLatWaves), args, 0, s);
        }));
        if ((st = pcf_wait_results(ctx, 1, 2, ctx->stream, &res->kernel_ms))) return st;
        res->total_ms = res->kernel_ms;
        if (fresh && (st = pcf_sequence_ms(ctx, ctx->ev_end, &res->total_ms))) return st;
        if (ctx->h_out[1] == 0.0) {
            lat_result(*res, ctx->h_out[0], N, american != 0, 1, 64 * kLatWaves);
            return PCF_OK;
        }
        // A wait gave up: the sweep is made by the launches below, once the
        // last wave has left and the words (with the error set) are gone.
        ctx->lat_in_turn |= plan.by_xcd == kById && !impatient;
        PCF_HIP_CHECK(ctx, hipStreamSynchronize(ctx->stream));
        ctx->lat_ring.release();
        fresh = false;  // the tables are there
    }
    if ((st = pcf_timing_begin(ctx))) return st;
    PCF_HIP_CHECK(ctx, upload(ctx->stream));

    PCF_HIP_CHECK(ctx, pcf_after_persistent(ctx, HUGE_VAL));
    PCF_HIP_CHECK(ctx, hipEventRecord(ctx->ev_kbeg, ctx->stream));
    const int lgrid = (int)std::min<int64_t>(4096, ((int64_t)row + kLatThreads - 1) / kLatThreads);
    if (american) k_lat_leaves<true><<<lgrid, kLatThreads, 0, ctx->stream>>>(P, up, dn, A);
    else k_lat_leaves<false><<<lgrid, kLatThreads, 0, ctx->stream>>>(P, up, dn, A);
    PCF_HIP_CHECK(ctx, hipGetLastError());
    int launches = 1;
    const int kmax = american ? LatTile<true>::K : LatTile<false>::K;
    const int wout = american ? LatTile<true>::Wout : LatTile<false>::Wout;
    for (int64_t n0 = N; n0 > 0;) {
        const int K = (int)std::min<int64_t>(kmax, n0);
        const int64_t outs = n0 - K + 1;
        const int64_t waves = (outs + wout - 1) / wout;
        const int grid = (int)((waves * 64 + kLatThreads - 1) / kLatThreads);
        if (american) k_lat_steps<true><<<grid, kLatThreads, 0, ctx->stream>>>(P, up, dn, A, B, n0, K);
        else k_lat_steps<false><<<grid, kLatThreads, 0, ctx->stream>>>(P, up, dn, A, B, n0, K);
        PCF_HIP_CHECK(ctx, hipGetLastError());
        std::swap(A, B);
        n0 -= K;
        ++launches;
    }
    PCF_HIP_CHECK(ctx, hipEventRecord(ctx->ev_kend, ctx->stream));
    PCF_HIP_CHECK(ctx, hipMemcpyAsync(ctx->out.ptr, A, sizeof(double), hipMemcpyDeviceToDevice, ctx->stream));
    if ((st = pcf_timing_end(ctx, 1, res))) return st;

    lat_result(*res, ctx->h_out[0], N, american != 0, launches, kLatThreads);
    return PCF_OK;
}

extern "C" void pcf_debug_lattice(int32_t bits) { lat_debug().store(bits, std::memory_order_relaxed); }

// pcf_device.hpp -- device building blocks shared by the gfx950 pricing
// kernels: counter-based Philox4x32-10, Box-Muller normals (FP32 on the
// hardware transcendental unit, FP64 on the functions below), payoff, and
// deterministic compensated FP64 reductions (wavefront shuffles + LDS, then a
// last-arriving-block pass over the per-block partials).
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

namespace pcf {

constexpr int kWave = 64;  // CDNA wavefront width

// ---------------------------------------------------------------------------
// Philox4x32-10 (Salmon et al., SC11).  Multipliers 0xD2511F53/0xCD9E8D57,
// Weyl increments 0x9E3779B9/0xBB67AE85.
struct U4 {
    uint32_t x, y, z, w;
};

// a ^ b ^ c as one gfx950 v_bitop3_b32 (truth table 0x96, the parity of the
// three input bits).  Written as two ^ the compiler issues two v_xor_b32,
// and the Monte Carlo kernels are bound by VALU issue, a third of it Philox.
__device__ __forceinline__ uint32_t xor3(uint32_t a, uint32_t b, uint32_t c) {
    return __builtin_amdgcn_bitop3_b32(a, b, c, 0x96);
}

// Each round needs both halves of two 32x32 products; written as one 64-bit
// product so gfx950 issues a single v_mad_u64_u32 per product (measured
// ~2.4x the throughput of a v_mul_lo_u32 + v_mul_hi_u32 pair).
__device__ __forceinline__ U4 philox4x32_10(U4 c, uint32_t k0, uint32_t k1) {
#pragma unroll
    for (int round = 0; round < 10; ++round) {
        const uint64_t p0 = (uint64_t)0xD2511F53u * c.x;
        const uint64_t p1 = (uint64_t)0xCD9E8D57u * c.z;
        U4 n;
        if (round == 0) {
            // Counter words are often wave-uniform (block, stream): left as
            // plain xors, the compiler keeps this round on the scalar unit.
            n.x = (uint32_t)(p1 >> 32) ^ c.y ^ k0;
            n.z = (uint32_t)(p0 >> 32) ^ c.w ^ k1;
        } else {
            n.x = xor3((uint32_t)(p1 >> 32), c.y, k0);
            n.z = xor3((uint32_t)(p0 >> 32), c.w, k1);
        }
        n.y = (uint32_t)p1;
        n.w = (uint32_t)p0;
        c = n;
        k0 += 0x9E3779B9u;
        k1 += 0xBB67AE85u;
    }
    return c;
}

// Whether a grid-stride loop over n items may count in 32 bits: n plus the
// stride has to be within 2^32, or an item past the last wraps to a small one
// and the loop never ends (2^20 blocks of 1024 threads stride by 2^30).  The
// counter's high path word is then a constant 0, which takes two of the
// generator's 20 products per block and the 64-bit loop arithmetic with it.
__host__ __device__ __forceinline__ bool fits_index32(int64_t n, unsigned int blocks, unsigned int threads) {
    return (uint64_t)n + (uint64_t)blocks * threads <= (uint64_t)1 << 32;
}

// Counter layout: (block of 4 normals, path lo, path hi, stream id).
template <typename Index>
__device__ __forceinline__ U4 philox_block(uint64_t seed, uint32_t stream, Index path,
                                           uint32_t block) {
    U4 c;
    c.x = block;
    c.y = (uint32_t)path;
    c.z = sizeof(Index) == 4 ? 0u : (uint32_t)((uint64_t)path >> 32);
    c.w = stream;
    return philox4x32_10(c, (uint32_t)seed, (uint32_t)(seed >> 32));
}

// ---------------------------------------------------------------------------
// Box-Muller.  Uniform u = (x + 0.5) 2^-32 in (0,1); the pair (u0, u1) gives
// z0 = R cos(2 pi u1), z1 = R sin(2 pi u1), R = sqrt(-2 ln u0).
//
// FP32: v_log_f32 is log2, v_sin_f32 / v_cos_f32 take their argument in
// revolutions (sin(2 pi x)), so one instruction each; u is the FP32 rounding
// of the FP64 uniform.
__device__ __forceinline__ float u01_f32(uint32_t x) {
    return fmaf((float)x, 0x1p-32f, 0x1p-33f);
}

// The pair as its radius and its two directions.
__device__ __forceinline__ void box_muller_polar_f32(uint32_t a, uint32_t b, float& R, float& c, float& s) {
    const float u0 = u01_f32(a);
    const float u1 = u01_f32(b);
    // -2 ln u0 = -2 ln(2) log2(u0)
    R = __builtin_amdgcn_sqrtf(-1.3862943611198906f * __builtin_amdgcn_logf(u0));
    c = __builtin_amdgcn_cosf(u1);
    s = __builtin_amdgcn_sinf(u1);
}
__device__ __forceinline__ void box_muller_f32(uint32_t a, uint32_t b, float& z0, float& z1) {
    float R, c, s;
    box_muller_polar_f32(a, b, R, c, s);
    z0 = R * c;
    z1 = R * s;
}

// ---------------------------------------------------------------------------
// FP64 elementary functions of the Monte Carlo kernels.  Those kernels are
// bound by VALU issue, and the library's log, sqrt, sincos and exp spend much
// of it on cases that cannot arise here (subnormal or huge arguments, a
// reduction modulo pi/2 of any double) and on selecting between them.  These
// take the argument ranges the kernels have; coefficients are Chebyshev
// interpolants computed in 60 digits and rounded to double.  Against 80-bit
// arithmetic on the same counters the normals' largest error is 1.4e-15 (rms
// 1.1e-16); the library's were 3.1e-15 (2.4e-16), mostly from rounding
// 2 pi u1.  500003 paths x 365 steps with the control 729 -> 360 us, 10^8
// European paths 420 -> 300 us.

// p(x) = c[0] + c[1] x + ... by Horner's rule.
template <int N>
__device__ __forceinline__ double horner(const double (&c)[N], double x) {
    double p = c[N - 1];
#pragma unroll
    for (int i = N - 2; i >= 0; --i) p = fma(p, x, c[i]);
    return p;
}

// -2 ln u for u = (x + 0.5) 2^-32, by the reduction and the correction term of
// fdlibm's log with a polynomial of our own.  v = x + 0.5 = m 2^k is exact, m in
// [sqrt(1/2), sqrt(2)); ln m = f - s (f - R), f = m - 1 (exact), s = f / (2 + f),
// R = s^2 P(s^2) (the atanh series), so that the rounding of the correction
// term is small against f; then (k - 32) ln 2 in two parts.
__device__ __forceinline__ double neg2_ln_u(uint32_t x) {
    const double v = (double)x + 0.5;
    const uint64_t b = __builtin_bit_cast(uint64_t, v);
    // exponent of v / sqrt(1/2), and the mantissa scaled into [sqrt(1/2), sqrt(2))
    const uint32_t h = (uint32_t)(b >> 32) + (0x3ff00000u - 0x3fe6a09eu);
    const int k = (int)(h >> 20) - (0x3ff + 32);
    const uint32_t mh = (h & 0x000fffffu) + 0x3fe6a09eu;
    const double m = __builtin_bit_cast(double, ((uint64_t)mh << 32) | (uint32_t)b);
    const double f = m - 1.0, d = m + 1.0;
    double y = __builtin_amdgcn_rcp(d);
    y = fma(fma(-d, y, 1.0), y, y);
    double s = f * y;
    s = fma(fma(-s, d, f), y, s);
    const double z = s * s;
    constexpr double P[7] = {0x1.5555555555558p-1, 0x1.99999999952e2p-2, 0x1.2492492df14dfp-2, 0x1.c71c62e579789p-3,
                             0x1.7462b4ad0d879p-3, 0x1.39fe60271f67fp-3, 0x1.2b584dae87b55p-3};
    const double R = z * horner(P, z);
    const double kd = (double)k;
    // ln m + k ln 2 (its low part first), doubled and negated
    double w = fma(-s, f - R, f);
    w = fma(kd, 0x1.abc9e3b39803fp-56, w);
    return -2.0 * fma(kd, 0x1.62e42fefa39efp-1, w);
}

// sqrt(a) for a positive normal a far from the ends of the exponent range:
// Goldschmidt's iteration from the hardware estimate, then one residual step.
__device__ __forceinline__ double sqrt_mid(double a) {
    const double y = __builtin_amdgcn_rsq(a);
    double g = a * y, h = 0.5 * y;
    const double r = fma(-h, g, 0.5);
    g = fma(g, r, g);
    h = fma(h, r, h);
    return fma(fma(-g, g, a), h, g);
}

// exp(r) for |r| <= ln(2)/2: 1 + r + r^2 Q(r).
__device__ __forceinline__ double exp_small(double r) {
    constexpr double Q[10] = {0x1.0000000000001p-1, 0x1.5555555555556p-3, 0x1.5555555553d68p-5, 0x1.11111111109b5p-7,
                              0x1.6c16c17889ef1p-10, 0x1.a01a01a7c2efep-13, 0x1.a019b9149a41cp-16,
                              0x1.71de0db2f6b19p-19, 0x1.28917c89a43a7p-22, 0x1.af389ecfc4b9cp-26};
    return 1.0 + fma(r * r, horner(Q, r), r);
}
// The largest |r| that exp_small takes.
constexpr double kExpSmall = 0.3465;

// exp(x) for any x: x = k ln 2 + r.  Below -800 the result is 0 (2^-1154
// underflows), above about 709.8 infinity; NaN stays NaN (the comparison is
// false and r is NaN).
__device__ __forceinline__ double exp_any(double x) {
    x = x < -800.0 ? -800.0 : x;
    const double k = fmin(rint(x * 0x1.71547652b82fep+0), 1100.0);
    double r = fma(-k, 0x1.62e42fefa39efp-1, x);
    r = fma(-k, 0x1.abc9e3b39803fp-56, r);
    return ldexp(exp_small(r), (int)k);
}

// The pair (R cos 2 pi u1, R sin 2 pi u1).  u1 modulo 1/2 is t in [-1/4, 1/4),
// exact as w = t 2^33 from the counter's bits, and the half turns left out
// change both signs; the polynomials take w, their coefficients scaled by
// powers of two.
__device__ __forceinline__ void box_muller_f64(uint32_t a, uint32_t b, double& z0, double& z1) {
    const double R = sqrt_mid(neg2_ln_u(a));
    const uint32_t b2 = b << 1;
    const uint32_t flip = (b ^ b2) & 0x80000000u;  // (u1 - t) / (1/2) is odd
    const double w = (double)(int32_t)b2 + 1.0;
    const double y = w * w;
    constexpr double Cs[9] = {0x1.921fb54442d18p-31,   -0x1.4abbce625be52p-94,  0x1.466bc6775aa7dp-159,
                              -0x1.32d2cce627c86p-225, 0x1.5078348551854p-292,  -0x1.e3074dfaf87afp-360,
                              0x1.e8f3675ee37ddp-428,  -0x1.6f7acdb8f6580p-496, 0x1.9d462020fcc78p-565};
    constexpr double Cc[9] = {1.0,
                              -0x1.3bd3cc9be45dbp-62,
                              0x1.03c1f081b5992p-126,
                              -0x1.55d3c7e3bfbf5p-192,
                              0x1.e1f506813a321p-259,
                              -0x1.a6d1efc8c38bep-326,
                              0x1.f9d254582ac30p-394,
                              -0x1.b6957b54dd389p-462,
                              0x1.1678f9078a9b3p-530};
    const uint64_t Rb = __builtin_bit_cast(uint64_t, R) ^ ((uint64_t)flip << 32);
    const double Rs = __builtin_bit_cast(double, Rb);
    z0 = Rs * horner(Cc, y);
    z1 = Rs * (w * horner(Cs, y));
}

template <typename Real>
__device__ __forceinline__ void box_muller(uint32_t a, uint32_t b, Real& z0, Real& z1);
template <>
__device__ __forceinline__ void box_muller<float>(uint32_t a, uint32_t b, float& z0, float& z1) {
    box_muller_f32(a, b, z0, z1);
}
template <>
__device__ __forceinline__ void box_muller<double>(uint32_t a, uint32_t b, double& z0, double& z1) {
    box_muller_f64(a, b, z0, z1);
}

// Four standard normals of (seed, stream, path, block).
template <typename Real, typename Index>
__device__ __forceinline__ void normals4(uint64_t seed, uint32_t stream, Index path,
                                         uint32_t block, Real z[4]) {
    const U4 x = philox_block(seed, stream, path, block);
    box_muller<Real>(x.x, x.y, z[0], z[1]);
    box_muller<Real>(x.z, x.w, z[2], z[3]);
}

// ---------------------------------------------------------------------------
// Fast FP32 exp on the hardware exp2 unit: exp(x) = 2^(x log2 e).  Kernels
// fold log2(e) into their constants and call exp2 directly.
__device__ __forceinline__ float exp2_f32(float x) { return __builtin_amdgcn_exp2f(x); }

template <typename Real>
__device__ __forceinline__ Real payoff(Real S, Real E, Real pf) {
    const Real v = pf * (S - E);
    return v > Real(0) ? v : Real(0);
}

// ---------------------------------------------------------------------------
// Compensated FP64 sums.  value = s + c; TwoSum (Knuth) keeps the rounding
// error of every add in c, so a sum of sums is accurate to ~1 ulp of the
// total independent of the order of the partials.
struct CSum {
    double s, c;
};

__device__ __forceinline__ void csum_add(CSum& a, double v) {
    const double t = a.s + v;
    const double bp = t - a.s;
    const double e = (a.s - (t - bp)) + (v - bp);
    a.s = t;
    a.c += e;
}

__device__ __forceinline__ CSum csum_merge(CSum a, CSum b) {
    const double t = a.s + b.s;
    const double bp = t - a.s;
    const double e = (a.s - (t - bp)) + (b.s - bp);
    CSum r;
    r.s = t;
    r.c = a.c + b.c + e;
    return r;
}

// K compensated sums per thread.
template <int K>
struct Acc {
    CSum v[K];
    __device__ __forceinline__ void zero() {
#pragma unroll
        for (int k = 0; k < K; ++k) v[k].s = v[k].c = 0.0;
    }
};

template <int K>
__device__ __forceinline__ void acc_merge_into(Acc<K>& a, const Acc<K>& b) {
#pragma unroll
    for (int k = 0; k < K; ++k) a.v[k] = csum_merge(a.v[k], b.v[k]);
}

// Lane exchanges without the LDS crossbar (gfx950): DPP within 16-lane rows
// (row_ror:n gives lane l the value of lane (l - n) mod 16; quad_perm 0x4E and
// 0xB1 are xor 2 and xor 1), and v_permlane32_swap / v_permlane16_swap, which
// swap the upper 32 lanes of x with the lower 32 of y (and the odd 16-lane
// rows of x with the even rows of y).  FP64 travels as two 32-bit halves.
template <int CTRL>
__device__ __forceinline__ double dpp_f64(double v) {
    const uint64_t u = __builtin_bit_cast(uint64_t, v);
    const uint32_t lo = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)(uint32_t)u, CTRL, 0xF, 0xF, false);
    const uint32_t hi = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)(uint32_t)(u >> 32), CTRL, 0xF, 0xF, false);
    return __builtin_bit_cast(double, ((uint64_t)hi << 32) | lo);
}
template <bool ROWS16>
__device__ __forceinline__ void permlane_swap_f64(double& x, double& y) {
    const uint64_t ux = __builtin_bit_cast(uint64_t, x), uy = __builtin_bit_cast(uint64_t, y);
    const uint32_t xl = (uint32_t)ux, xh = (uint32_t)(ux >> 32), yl = (uint32_t)uy, yh = (uint32_t)(uy >> 32);
    uint32_t rl0, rl1, rh0, rh1;
    if constexpr (ROWS16) {
        const auto l = __builtin_amdgcn_permlane16_swap(xl, yl, false, false);
        const auto h = __builtin_amdgcn_permlane16_swap(xh, yh, false, false);
        rl0 = l[0]; rl1 = l[1]; rh0 = h[0]; rh1 = h[1];
    } else {
        const auto l = __builtin_amdgcn_permlane32_swap(xl, yl, false, false);
        const auto h = __builtin_amdgcn_permlane32_swap(xh, yh, false, false);
        rl0 = l[0]; rl1 = l[1]; rh0 = h[0]; rh1 = h[1];
    }
    x = __builtin_bit_cast(double, ((uint64_t)rh0 << 32) | rl0);
    y = __builtin_bit_cast(double, ((uint64_t)rh1 << 32) | rl1);
}

// The other lane's CSum of an exchange within a 16-lane row: xor 8, 4, 2 or 1.
template <int XOR>
__device__ __forceinline__ double row_xor(double v) {
    if constexpr (XOR == 8) return dpp_f64<0x128>(v);  // row_ror:8
    if constexpr (XOR == 4) {
        // row_ror:4 for lanes with bit 2 set, row_ror:12 for the others; both
        // run in every lane before the select
        const double r4 = dpp_f64<0x124>(v), r12 = dpp_f64<0x12C>(v);
        return (threadIdx.x & 4) ? r4 : r12;
    }
    if constexpr (XOR == 2) return dpp_f64<0x4E>(v);
    return dpp_f64<0xB1>(v);
}

// Sums of K CSums over the 64 lanes of a wave, a tree of xor exchanges 32, 16,
// 8, 4, 2, 1.  Of a pair of sums, lanes 0..31 keep the first and lanes 32..63
// the second from the first exchange on, so that the other five handle one
// CSum for two: sum 2i ends in lane 0, sum 2i + 1 in lane 32 (the last of an
// odd K in both), in r[i].  No exchange goes through the LDS crossbar: with
// every wave of a full CU reducing at the end of a launch, shuffles took about
// 5 us there, and each block of a longer grid 2.5-5 ns of the whole device's
// time (basket of 8 assets, 2^20 paths: 27.4 -> 17.3 us; European 2^24 24 -> 17).
// A merge of two CSums has the same bits in either order.
template <int K>
__device__ __forceinline__ void wave_reduce(const Acc<K>& a, CSum (&r)[(K + 1) / 2]) {
#pragma unroll
    for (int i = 0; i < (K + 1) / 2; ++i) {
        CSum x = a.v[2 * i], y = a.v[2 * i + 1 < K ? 2 * i + 1 : 2 * i];
        permlane_swap_f64<false>(x.s, y.s);
        permlane_swap_f64<false>(x.c, y.c);
        x = csum_merge(x, y);  // xor 32
        y = x;
        permlane_swap_f64<true>(x.s, y.s);
        permlane_swap_f64<true>(x.c, y.c);
        x = csum_merge(x, y);  // xor 16
        x = csum_merge(x, CSum{row_xor<8>(x.s), row_xor<8>(x.c)});
        x = csum_merge(x, CSum{row_xor<4>(x.s), row_xor<4>(x.c)});
        x = csum_merge(x, CSum{row_xor<2>(x.s), row_xor<2>(x.c)});
        x = csum_merge(x, CSum{row_xor<1>(x.s), row_xor<1>(x.c)});
        r[i] = x;
    }
}

// Block reduction; the result is valid in thread 0.  `lds` holds
// (blockDim/64) * K CSums.  Fixed order => deterministic for a launch shape.
template <int K>
__device__ __forceinline__ Acc<K> block_reduce(const Acc<K>& in, CSum* lds) {
    CSum r[(K + 1) / 2];
    wave_reduce<K>(in, r);
    const int lane = threadIdx.x & (kWave - 1);
    const int wave = threadIdx.x / kWave;
    const int nwaves = (blockDim.x + kWave - 1) / kWave;
    if ((lane & 31) == 0) {
#pragma unroll
        for (int i = 0; i < (K + 1) / 2; ++i) {
            const int k = 2 * i + (lane >> 5);
            if (k < K) lds[wave * K + k] = r[i];
        }
    }
    __syncthreads();
    Acc<K> a;
    a.zero();
    if (threadIdx.x == 0) {
#pragma unroll
        for (int k = 0; k < K; ++k) a.v[k] = lds[k];
        for (int w = 1; w < nwaves; ++w) {
#pragma unroll
            for (int k = 0; k < K; ++k) a.v[k] = csum_merge(a.v[k], lds[w * K + k]);
        }
    }
    return a;
}

// Cross-block data (partials, counters, flags) is published with coherent
// agent-scope atomic stores, which write through the per-XCD L2, and read
// with coherent atomic loads.  Ordering a block's published values before its
// arrival only needs those stores to be complete (vmcnt 0), so no agent-scope
// fence -- i.e. no whole-L2 write-back or invalidate -- is needed anywhere.
__device__ __forceinline__ void publish(double* p, double v) {
    __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ double fetch(const double* p) {
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ void publish_u32(unsigned int* p, unsigned int v) {
    __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ unsigned int fetch_u32(const unsigned int* p) {
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ unsigned long long fetch_u64(const unsigned long long* p) {
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
// Wait until every memory operation this wave issued is complete.
__device__ __forceinline__ void stores_complete() { __builtin_amdgcn_s_waitcnt(0); }

// Arrival counting of grid_reduce.  Device-scope atomics on one address run
// one after another, so a single arrival counter costs nblk such atomics in
// sequence at the end of a launch whose blocks finish together.  Block b
// counts on group counter b mod kArriveGroups instead; the last block of each
// group then counts on a top counter, whose last arrival is the last block
// overall.  Each counter has its own 128-byte line; one reduction uses
// kCounterWords uint32 of counter space.
constexpr int kArriveGroups = 32;
constexpr int kCounterLine = 32;  // uint32 per 128-byte line
constexpr int kCounterWords = (kArriveGroups + 1) * kCounterLine;

// Per-block partial write + "last block finishes" grid reduction.
//   partials: nblk * K CSums;  counter: kCounterWords uint32, zero at launch and left
//   zero on exit.  Returns true in the (single) block that performed the
//   final pass, whose thread 0 then holds the totals in `tot`.
//   blk / nblk: this block's index and the block count of the reduction (the
//   launch grid for a single request; the request's share of a batched grid).
template <int K>
__device__ __forceinline__ bool grid_reduce(Acc<K> a, CSum* __restrict__ partials,
                                            unsigned int* __restrict__ counter, CSum* lds,
                                            Acc<K>& tot, unsigned int blk, unsigned int nblk) {
    __shared__ bool is_last;
    a = block_reduce<K>(a, lds);
    if (threadIdx.x == 0) {
#pragma unroll
        for (int k = 0; k < K; ++k) {
            publish(&partials[(size_t)blk * K + k].s, a.v[k].s);
            publish(&partials[(size_t)blk * K + k].c, a.v[k].c);
        }
        stores_complete();
        // Group g holds blocks g, g + 32, ...: ceil((nblk - g) / 32) of them
        // (blk < nblk, so g < nblk and the group is not empty).
        const unsigned int g = blk % kArriveGroups;
        const unsigned int ng = (nblk - g + kArriveGroups - 1) / kArriveGroups;
        const unsigned int groups = nblk < (unsigned)kArriveGroups ? nblk : (unsigned)kArriveGroups;
        bool last = false;
        if (atomicAdd(&counter[g * kCounterLine], 1u) == ng - 1)
            last = atomicAdd(&counter[kArriveGroups * kCounterLine], 1u) == groups - 1;
        is_last = last;
    }
    __syncthreads();
    if (!is_last) return false;
    // Thread t folds partials t, t+B, t+2B, ... in order, then a block reduce.
    // The loads of U consecutive partials are issued before their merges, so
    // they are in flight together; the merge order is unchanged.
    constexpr int U = K <= 2 ? 4 : K <= 4 ? 2 : 1;
    Acc<K> r;
    r.zero();
    unsigned int b = threadIdx.x;
    for (; b + (U - 1) * blockDim.x < nblk; b += U * blockDim.x) {
        CSum p[U][K];
#pragma unroll
        for (int u = 0; u < U; ++u)
#pragma unroll
            for (int k = 0; k < K; ++k) {
                p[u][k].s = fetch(&partials[(size_t)(b + u * blockDim.x) * K + k].s);
                p[u][k].c = fetch(&partials[(size_t)(b + u * blockDim.x) * K + k].c);
            }
#pragma unroll
        for (int u = 0; u < U; ++u)
#pragma unroll
            for (int k = 0; k < K; ++k) r.v[k] = csum_merge(r.v[k], p[u][k]);
    }
    for (; b < nblk; b += blockDim.x) {
#pragma unroll
        for (int k = 0; k < K; ++k) {
            CSum p;
            p.s = fetch(&partials[(size_t)b * K + k].s);
            p.c = fetch(&partials[(size_t)b * K + k].c);
            r.v[k] = csum_merge(r.v[k], p);
        }
    }
    __syncthreads();  // lds reuse
    r = block_reduce<K>(r, lds);
    // Every block has counted (the top counter is complete): clear the
    // counters for the next launch.
    for (unsigned int c = threadIdx.x; c <= (unsigned)kArriveGroups; c += blockDim.x)
        publish_u32(&counter[c * kCounterLine], 0u);
    if (threadIdx.x == 0) tot = r;
    return true;
}

// Results go straight to the host: `out` is the context's pinned buffer (or a
// device copy of its layout), kOutPerJob words per job: up to 8 results, the
// device clock when the launch's first block started (job 0 only) and when the
// job's last block ended.  The host waits for the words themselves (it marks
// them as unwritten before the launch), so a pricing needs no copy back, no
// event and no blocking wait: launch, a few microseconds, result.
constexpr int kOutPerJob = 16;
constexpr int kOutStart = 8, kOutEnd = 9;
__device__ __forceinline__ void to_host(double* p, double v) {
    __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
}
// The constant-rate device clock (s_memrealtime), as bits.
__device__ __forceinline__ void stamp(double* p) {
    to_host(p, __builtin_bit_cast(double, (uint64_t)wall_clock64()));
}

// Final FP64 moments of NP (sum, sum of squares) pairs: out[4k..4k+3] =
// sum, sum of squares, mean, sample variance; and the job's end.
template <int NP>
__device__ __forceinline__ void write_moments(const Acc<2 * NP>& tot, int64_t N, double* out) {
    const double n = (double)N;
#pragma unroll
    for (int k = 0; k < NP; ++k) {
        const double sum = tot.v[2 * k].s + tot.v[2 * k].c;
        const double sq = tot.v[2 * k + 1].s + tot.v[2 * k + 1].c;
        const double mean = sum / n;
        to_host(out + 4 * k + 0, sum);
        to_host(out + 4 * k + 1, sq);
        to_host(out + 4 * k + 2, mean);
        to_host(out + 4 * k + 3, N > 1 ? (sq - sum * mean) / (n - 1.0) : 0.0);
    }
    stamp(out + kOutEnd);
}

// Batched launches: job j owns blocks [first_block, first_block + nblk) of the
// grid.  Returns the job of block b (jobs sorted by first_block; b is
// block-uniform, so the search runs on scalar loads).
template <typename Job>
__device__ __forceinline__ int find_job(const Job* __restrict__ jobs, int njobs, unsigned int b) {
    int lo = 0, hi = njobs - 1;
    while (lo < hi) {
        const int mid = (lo + hi + 1) >> 1;
        if (jobs[mid].first_block <= b) lo = mid;
        else hi = mid - 1;
    }
    return lo;
}

// What a launch of one or more jobs is given.  A lone job travels in the
// kernel arguments, so that it needs no copy before its launch; a batch's
// table is in device memory.
template <typename Job>
struct JobArgs {
    Job one;
    const Job* table;
    int njobs;
};
// The job of block b; the first block of the launch notes the time.
template <typename Job>
__device__ __forceinline__ Job job_of(const JobArgs<Job>& a, unsigned int b) {
    Job J;
    if (a.njobs == 1) J = a.one;
    else J = a.table[find_job(a.table, a.njobs, b)];
    if (b == 0 && threadIdx.x == 0) stamp(J.out + kOutStart);
    return J;
}

}  // namespace pcf

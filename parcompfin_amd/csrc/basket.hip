// basket.hip -- arithmetic basket on d correlated GBM assets, one terminal step.
// Reference: src/mc_eur_multi.cpp:26-33 with mvnorm (include/mvn.h:42-82):
//     B = L Z (L = Cholesky factor of the correlation matrix, Z ~ N(0, I))
//     basket_n = sum_a w_a S0_a exp((r - s_a^2/2) T + s_a sqrt(T) B_a)
// (the reference has one scalar sigma, S0, weights 1/d, equicorrelation rho,
// and omits sqrt(T): ref_exact=1 reproduces that; all configs have T = 1).
//
// Kernels:
//  * k_basket_one<Real>: factors whose columns are constant below the diagonal,
//    which is what one correlation for every pair gives (the reference's only
//    form).  Then B_i = P_i + L_ii z_i with P_{i+1} = P_i + l_i z_i: 2 d FMAs
//    in place of d (d + 1) / 2, in the same order, so the same bits as below.
//  * k_basket_fma<Real, DMAX, MODE, FULL>: one path per lane; d normals in
//    registers, B = L z with scalar-broadcast L, per-asset exp and the weighted
//    sum fused; FP32/Kahan, FP64 and host-normal verification forms.
//  * k_basket_mfma<Real, NB, FULL>: 13 assets and more.  One wavefront prices
//    16 paths per tile: the exponents X^T (16 NB assets x 16 paths) = c0 +
//    (c1 L) Z^T, with L zero padded to blocks of 16 and each row scaled by c1
//    (x log2 e in FP32), on v_mfma_f32_16x16x4f32 or v_mfma_f64_16x16x4f64,
//    skipping the factor's zero upper-right blocks, the accumulation starting
//    from c0.  Each lane generates exactly the normals it feeds, so Z and X
//    never touch memory; the epilogue (exponential, weights, basket sum) runs
//    on the accumulator registers, the four lane groups combined by lane
//    exchange.
#include <cmath>
#include <atomic>
#include <cstring>
#include <map>
#include <memory>
#include <mutex>
#include <vector>

#include "pcf_internal.hpp"

namespace {

constexpr int kMaxAssets = 64;
// A general factor goes to the MFMA kernel from 13 assets: its work is that of
// the next multiple of 16, the FMA kernel's grows with d^2 and past 32 its
// normals leave the registers (2^20 paths, FP32 / FP64, MFMA against FMA: d =
// 12 22.5 / 56.7 against 23.3 / 58.2 us, 15 22.5 / 56.7 against 29.6 / 76.1, 17
// 39.1 / 99 against 39.0 / 118, 33 66 / 163 against 471 / 1141).
constexpr int kMfmaFrom = 13;
// Threads per block of both basket kernels; their LDS reduction buffers are
// sized for it and the host refuses larger blocks.
constexpr int kBasketThreads = 256;
enum { kFp32k = 0, kFp64 = 1, kHost = 2 };

struct BasketArgs {
    double E, pf;
    float Ef, pff;
    int64_t N;
    int32_t d;
    int32_t full;  // the factor is not lower triangular (eigen fallback)
    uint64_t seed;
};

// Device constants, one buffer: FP64 block then FP32 block.
//   FP64: L[d*d] (row-major), c0[d] = (r - s^2/2)T, c1[d] = s sqrt(T) (or s),
//         ws[d] = w S0
//   FP32: Lf[d*d] (the FMA kernel's factor), c0f[64], c1f[64] (x log2 e),
//         wsf[64].
// (The MFMA kernel forms its operands from L and c1 in FP64.)
// And for k_basket_one, in both types, per 4 assets (the last 4 padded): l[4], L_ii[4], c0[4], c1[4], ws[4].
struct BasketLayout {
    size_t off_one64, off_one32, off_L64, off_c064, off_c164, off_ws64, off_Lf, off_c0f, off_c1f, off_wsf, bytes;
    static BasketLayout make(int d) {
        BasketLayout l;
        size_t o = 0;
        l.off_L64 = o; o += sizeof(double) * d * d;
        l.off_c064 = o; o += sizeof(double) * d;
        l.off_c164 = o; o += sizeof(double) * d;
        l.off_ws64 = o; o += sizeof(double) * d;
        l.off_Lf = o; o += sizeof(float) * d * d;
        l.off_c0f = o; o += sizeof(float) * kMaxAssets;
        l.off_c1f = o; o += sizeof(float) * kMaxAssets;
        l.off_wsf = o; o += sizeof(float) * kMaxAssets;
        o = (o + 63) / 64 * 64;
        l.off_one64 = o; o += sizeof(double) * 20 * ((d + 3) / 4);
        l.off_one32 = o; o += sizeof(float) * 20 * ((d + 3) / 4);
        l.bytes = o;
        return l;
    }
};

struct BasketJob {
    BasketArgs a;
    const void* Lm;   // FMA: d x d factor (Real); MFMA: the FP64 factor; prefix form: its constants
    const void* c0;
    const void* c1;
    const void* ws;
    const double* hz;
    pcf::CSum* partials;
    unsigned int* counter;
    double* out;
    unsigned int first_block, nblk;
};
static_assert(sizeof(BasketJob) <= kJobBytes, "job record exceeds its staging slot");

// The factor and the per-asset constants are read-only and the same for every
// lane, so the FMA kernel reads them through the constant address space: the
// compiler then issues scalar loads whose results feed the FMAs as SGPR
// operands.  Through generic pointers every asset's row was a flat vector load
// followed by a wait on the vector memory counter inside the path loop.
template <typename T>
using cptr = const __attribute__((address_space(4))) T*;

template <typename Real, int DMAX, int MODE, bool FULL>
__device__ __forceinline__ void basket_fma_body(const BasketArgs& a, cptr<Real> Lm, cptr<Real> c0,
                                                cptr<Real> c1, cptr<Real> ws,
                                                const double* __restrict__ hz,
                                                pcf::CSum* __restrict__ partials,
                                                unsigned int* __restrict__ counter,
                                                double* __restrict__ out, unsigned int blk,
                                                unsigned int nblk, pcf::CSum* lds) {
    const int d = a.d;
    double s = 0.0, s2 = 0.0;
    const int64_t stride = (int64_t)nblk * blockDim.x;
    for (int64_t p = (int64_t)blk * blockDim.x + threadIdx.x; p < a.N; p += stride) {
        Real z[DMAX];
        if (MODE == kHost) {
#pragma unroll
            for (int k = 0; k < DMAX; ++k) {
                if (k < d) z[k] = (Real)hz[p * d + k];
                else z[k] = Real(0);
            }
        } else {
#pragma unroll
            for (int b = 0; b < DMAX / 4; ++b) {
                if (4 * b < d) {
                    Real t[4];
                    pcf::normals4<Real>(a.seed, PCF_STREAM_BASKET, (uint64_t)p, (uint32_t)b, t);
#pragma unroll
                    for (int q = 0; q < 4; ++q) z[4 * b + q] = t[q];
                } else {
#pragma unroll
                    for (int q = 0; q < 4; ++q) z[4 * b + q] = Real(0);
                }
            }
        }
        Real basket = 0;
#pragma unroll
        for (int i = 0; i < DMAX; ++i) {
            if (i < d) {
                Real B = 0;
                if (MODE == kHost) {
#pragma clang fp contract(off)
#pragma unroll
                    for (int k = 0; k < DMAX; ++k)
                        if ((FULL ? true : k <= i) && k < d) B += Lm[i * d + k] * z[k];
                    // (w S0) * exp((r - pow(s,2)/2) T + s B)  (src/mc_eur_multi.cpp:30)
                    basket += ws[i] * exp(c0[i] + c1[i] * B);
                } else {
#pragma unroll
                    for (int k = 0; k < DMAX; ++k)
                        if ((FULL ? true : k <= i) && k < d) B = fma(Lm[i * d + k], z[k], B);
                    if constexpr (sizeof(Real) == 4)
                        basket = fmaf(ws[i], pcf::exp2_f32(fmaf(c1[i], B, c0[i])), basket);
                    else
                        basket = fma(ws[i], pcf::exp_any(fma(c1[i], B, c0[i])), basket);
                }
            }
        }
        Real v = pcf::payoff<Real>(basket, (Real)a.E, (Real)a.pf);
        const double dv = (double)v;
        s += dv;
        s2 += dv * dv;
    }
    pcf::Acc<2> acc, tot;
    acc.v[0] = {s, 0.0};
    acc.v[1] = {s2, 0.0};
    if (pcf::grid_reduce<2>(acc, partials, counter, lds, tot, blk, nblk) && threadIdx.x == 0)
        pcf::write_moments<1>(tot, a.N, out);
}

template <typename Real, int DMAX, int MODE, bool FULL>
__global__ __launch_bounds__(kBasketThreads) void k_basket_fma(const pcf::JobArgs<BasketJob> args) {
    __shared__ pcf::CSum lds[(kBasketThreads / pcf::kWave) * 2];
    const BasketJob J = pcf::job_of(args, blockIdx.x);
    basket_fma_body<Real, DMAX, MODE, FULL>(J.a, (cptr<Real>)J.Lm, (cptr<Real>)J.c0, (cptr<Real>)J.c1,
                                            (cptr<Real>)J.ws, J.hz, J.partials, J.counter, J.out,
                                            blockIdx.x - J.first_block, J.nblk, lds);
}

// One path per lane; a Philox block feeds 4 assets, and nothing of an earlier
// block is kept but the prefix P, so any d runs with the registers of 4 assets.
// Index: uint32_t where every path number fits, which leaves the counter's
// high word a constant 0.
template <typename Real, typename Index>
__device__ __forceinline__ void basket_one_paths(const BasketArgs& a, cptr<Real> k, unsigned int blk,
                                                 unsigned int nblk, double& s, double& s2) {
    const int nb = a.d >> 2, rem = a.d & 3;
    const Index N = (Index)a.N, stride = (Index)nblk * blockDim.x;
    for (Index p = (Index)blk * blockDim.x + threadIdx.x; p < N; p += stride) {
        Real P = 0, basket = 0;
        auto asset = [&](cptr<Real> c, int i, Real z) {
            const Real B = fma(c[4 + i], z, P);
            P = fma(c[i], z, P);
            if constexpr (sizeof(Real) == 4)
                basket = fmaf(c[16 + i], pcf::exp2_f32(fmaf(c[12 + i], B, c[8 + i])), basket);
            else
                basket = fma(c[16 + i], pcf::exp_any(fma(c[12 + i], B, c[8 + i])), basket);
        };
        for (int b = 0; b < nb; ++b) {
            Real z[4];
            pcf::normals4<Real>(a.seed, PCF_STREAM_BASKET, p, (uint32_t)b, z);
#pragma unroll
            for (int i = 0; i < 4; ++i) asset(k + 20 * b, i, z[i]);
        }
        if (rem) {  // the same for every lane: branches, no work for padding
            Real z[4];
            const pcf::U4 x = pcf::philox_block(a.seed, PCF_STREAM_BASKET, p, (uint32_t)nb);
            const cptr<Real> c = k + 20 * nb;
            pcf::box_muller<Real>(x.x, x.y, z[0], z[1]);
            asset(c, 0, z[0]);
            if (rem > 1) asset(c, 1, z[1]);
            if (rem > 2) {
                pcf::box_muller<Real>(x.z, x.w, z[2], z[3]);
                asset(c, 2, z[2]);
            }
        }
        const double dv = (double)pcf::payoff<Real>(basket, (Real)a.E, (Real)a.pf);
        s += dv;
        s2 += dv * dv;
    }
}

template <typename Real>
__global__ __launch_bounds__(kBasketThreads) void k_basket_one(const pcf::JobArgs<BasketJob> args) {
    __shared__ pcf::CSum lds[(kBasketThreads / pcf::kWave) * 2];
    const BasketJob J = pcf::job_of(args, blockIdx.x);
    const unsigned int blk = blockIdx.x - J.first_block;
    double s = 0.0, s2 = 0.0;
    if (pcf::fits_index32(J.a.N, J.nblk, blockDim.x))
        basket_one_paths<Real, uint32_t>(J.a, (cptr<Real>)J.Lm, blk, J.nblk, s, s2);
    else
        basket_one_paths<Real, int64_t>(J.a, (cptr<Real>)J.Lm, blk, J.nblk, s, s2);
    pcf::Acc<2> acc, tot;
    acc.v[0] = {s, 0.0};
    acc.v[1] = {s2, 0.0};
    if (pcf::grid_reduce<2>(acc, J.partials, J.counter, lds, tot, blk, J.nblk) && threadIdx.x == 0)
        pcf::write_moments<1>(tot, J.a.N, J.out);
}

typedef float v4f __attribute__((ext_vector_type(4)));
typedef double v4d __attribute__((ext_vector_type(4)));
template <typename Real>
struct Mfma16;
template <>
struct Mfma16<float> {
    using V = v4f;
    static __device__ __forceinline__ V mac(float a, float b, V c) {
        return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
    }
    static __device__ __forceinline__ int row(int g, int r) { return 4 * g + r; }
};
template <>
struct Mfma16<double> {
    using V = v4d;
    static __device__ __forceinline__ V mac(double a, double b, V c) {
        return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
    }
    static __device__ __forceinline__ int row(int g, int r) { return g + 4 * r; }
};
// Blocks of 16 x 16 of the factor, row block a, column block k.
template <int NB, bool FULL>
struct FactorBlocks {
    static constexpr int count = FULL ? NB * NB : NB * (NB + 1) / 2;
    static __device__ constexpr int at(int a, int k) { return FULL ? a * NB + k : a * (a + 1) / 2 + k; }
};

// The 16x16x4 forms (A: 16 rows x 4 k, lane l supplies row l%16, k l/16; B: 4 k
// x 16 columns, lane l supplies k l/16, column l%16; D: lane l holds 4 rows of
// column l%16, rows 4(l/16)+r in FP32 and l/16+4r in FP64).  Rows are assets
// in blocks of 16, columns the tile's paths.  Step q of column block k sums
// over 16k + 4g + q for the four lane groups g = l/16: lane (g, j) feeds the 4
// normals of Philox block 4k + g of path j, a whole block, in order.  A
// Cholesky factor is lower triangular, so row block a needs only k <= a.
// The factor's operands are in LDS in the order the lanes read them (no bank
// conflicts).  Where all of them, c0 and ws fit in registers beside the rest
// (FP32 up to 32 assets) they stay there; otherwise they are read again for
// each tile: at 64 assets in FP64 that is 20 KB, 160 cycles of a CU's LDS
// against about 1300 of arithmetic, and 112 registers less, so four waves fit
// a SIMD instead of two.
template <typename Real, int NB, bool FULL, typename Index>
__device__ __forceinline__ void basket_mfma_paths(const BasketArgs& a, const Real* A, const Real* c0, const Real* ws,
                                                  unsigned int blk, unsigned int nblk, double& s, double& s2) {
    using Mm = Mfma16<Real>;
    using Fb = FactorBlocks<NB, FULL>;
    constexpr bool kStream = sizeof(Real) == 8 || NB > 2;
    const int lane = threadIdx.x & 63;
    const int j = lane & 15;  // path column of the tile; also the A-operand row
    const int g = lane >> 4;  // k group fed by this lane
    const Index N = (Index)a.N, ntiles = (N + 15) >> 4;
    const Index wave = (Index)(((uint64_t)blk * blockDim.x + threadIdx.x) >> 6);
    const Index nwaves = (Index)(((uint64_t)nblk * blockDim.x) >> 6);
    for (Index t = wave; t < ntiles; t += nwaves) {
        const Index p = (t << 4) + j;
        int at = lane, row0 = Mm::row(g, 0);
        if constexpr (kStream) asm volatile("" : "+v"(at), "+v"(row0));  // not loop invariants, so not held in registers
        typename Mm::V acc[NB];
#pragma unroll
        for (int b = 0; b < NB; ++b)
#pragma unroll
            for (int r = 0; r < 4; ++r) acc[b][r] = c0[16 * b + row0 + Mm::row(0, r)];
#pragma unroll(kStream ? 1 : NB)
        for (int k = 0; k < NB; ++k) {
            Real z[4];
            pcf::normals4<Real>(a.seed, PCF_STREAM_BASKET, p, (uint32_t)(4 * k + g), z);
#pragma unroll
            for (int b = 0; b < NB; ++b)
                if (FULL || b >= k)
#pragma unroll
                    for (int q = 0; q < 4; ++q)
                        acc[b] = Mm::mac(A[(4 * Fb::at(b, k) + q) * 64 + at], z[q], acc[b]);
        }
        Real part = 0;
#pragma unroll
        for (int b = 0; b < NB; ++b)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                // (in FP64 register r holds 4 consecutive assets, past the last: skipped)
                if (sizeof(Real) == 8 && 16 * b + 4 * r >= a.d) break;
                const Real w = ws[16 * b + row0 + Mm::row(0, r)];
                if constexpr (sizeof(Real) == 4) part = fmaf(w, pcf::exp2_f32(acc[b][r]), part);
                else part = fma(w, pcf::exp_any(acc[b][r]), part);
            }
        // the assets of path j sit in the four lane groups
        if constexpr (sizeof(Real) == 4) {
            const uint32_t u = __builtin_bit_cast(uint32_t, part);
            const auto x = __builtin_amdgcn_permlane16_swap(u, u, false, false);
            part = __builtin_bit_cast(float, (uint32_t)x[0]) + __builtin_bit_cast(float, (uint32_t)x[1]);
            const uint32_t v = __builtin_bit_cast(uint32_t, part);
            const auto y = __builtin_amdgcn_permlane32_swap(v, v, false, false);
            part = __builtin_bit_cast(float, (uint32_t)y[0]) + __builtin_bit_cast(float, (uint32_t)y[1]);
        } else {
            double x = part, y = part;
            pcf::permlane_swap_f64<true>(x, y);
            x += y;
            y = x;
            pcf::permlane_swap_f64<false>(x, y);
            part = x + y;
        }
        if (g == 0 && p < N) {
            const double dv = (double)pcf::payoff<Real>(part, (Real)a.E, (Real)a.pf);
            s += dv;
            s2 += dv * dv;
        }
    }
}

// What bounds it: the normals and exponentials (a path's contraction is under a
// fifth of the FP32 vector work at 64 assets).  2^20 paths against the FMA
// kernel: FP32 d = 33 471 -> 66 us, 64 1030 -> 100; FP64 d = 16 79 -> 57, 32 261
// -> 114, 64 3130 -> 254.  The error against 64-bit prices is the FMA kernel's
// (FP32 9e-8 to 2.5e-7, FP64 below 1e-15).
// At least four waves per SIMD: operands and accumulators then stay in VGPRs.
template <typename Real, int NB, bool FULL>
__global__ __launch_bounds__(kBasketThreads) __attribute__((amdgpu_waves_per_eu(4)))
void k_basket_mfma(const pcf::JobArgs<BasketJob> args) {
    using Fb = FactorBlocks<NB, FULL>;
    __shared__ pcf::CSum lds[(kBasketThreads / pcf::kWave) * 2];
    __shared__ Real A[Fb::count * 256], c0[16 * NB], ws[16 * NB];
    const BasketJob J = pcf::job_of(args, blockIdx.x);
    const int d = J.a.d;
    const double* __restrict__ L = (const double*)J.Lm;
    const double* __restrict__ c1 = (const double*)J.c1;
    const double unit = sizeof(Real) == 4 ? 1.4426950408889634 : 1.0;  // exponents to base 2 in FP32
    for (int b = 0; b < NB; ++b)
        for (int k = 0; k < (FULL ? NB : b + 1); ++k)
            for (int e = threadIdx.x; e < 256; e += blockDim.x) {
                const int row = 16 * b + (e & 15), col = 16 * k + 4 * ((e >> 4) & 3) + (e >> 6);
                A[256 * Fb::at(b, k) + e] =
                    row < d && col < d ? (Real)(L[(size_t)row * d + col] * (c1[row] * unit)) : Real(0);
            }
    for (int i = threadIdx.x; i < 16 * NB; i += blockDim.x) {
        c0[i] = i < d ? ((const Real*)J.c0)[i] : Real(0);
        ws[i] = i < d ? ((const Real*)J.ws)[i] : Real(0);
    }
    __syncthreads();
    double s = 0.0, s2 = 0.0;
    const unsigned int blk = blockIdx.x - J.first_block;
    if (pcf::fits_index32(J.a.N, J.nblk, blockDim.x))
        basket_mfma_paths<Real, NB, FULL, uint32_t>(J.a, A, c0, ws, blk, J.nblk, s, s2);
    else
        basket_mfma_paths<Real, NB, FULL, int64_t>(J.a, A, c0, ws, blk, J.nblk, s, s2);
    pcf::Acc<2> acc, tot;
    acc.v[0] = {s, 0.0};
    acc.v[1] = {s2, 0.0};
    if (pcf::grid_reduce<2>(acc, J.partials, J.counter, lds, tot, blk, J.nblk) && threadIdx.x == 0)
        pcf::write_moments<1>(tot, J.a.N, J.out);
}

// ---- host linear algebra (FP64) ---------------------------------------------
// Lower Cholesky factor, textbook column order; false if not positive definite.
bool cholesky(int d, const std::vector<double>& C, std::vector<double>& L) {
    L.assign((size_t)d * d, 0.0);
    for (int j = 0; j < d; ++j) {
        double s = C[j * d + j];
        for (int k = 0; k < j; ++k) s -= L[j * d + k] * L[j * d + k];
        if (!(s > 0)) return false;
        const double ljj = std::sqrt(s);
        L[j * d + j] = ljj;
        for (int i = j + 1; i < d; ++i) {
            double t = C[i * d + j];
            for (int k = 0; k < j; ++k) t -= L[i * d + k] * L[j * d + k];
            L[i * d + j] = t / ljj;
        }
    }
    return true;
}

// Symmetric eigen-decomposition by cyclic Jacobi rotations; the factor
// V sqrt(Lambda) used by mvnorm when the Cholesky factorisation fails
// (include/mvn.h:73-76).  Returns false if an eigenvalue is clearly negative.
bool eigen_factor(int d, const std::vector<double>& C, std::vector<double>& F) {
    std::vector<double> A = C, V((size_t)d * d, 0.0);
    for (int i = 0; i < d; ++i) V[i * d + i] = 1.0;
    for (int sweep = 0; sweep < 100; ++sweep) {
        double off = 0.0;
        for (int p = 0; p < d; ++p)
            for (int q = p + 1; q < d; ++q) off += A[p * d + q] * A[p * d + q];
        if (off < 1e-30) break;
        for (int p = 0; p < d; ++p)
            for (int q = p + 1; q < d; ++q) {
                const double apq = A[p * d + q];
                if (std::fabs(apq) < 1e-300) continue;
                const double theta = (A[q * d + q] - A[p * d + p]) / (2.0 * apq);
                const double t = (theta >= 0 ? 1.0 : -1.0) / (std::fabs(theta) + std::sqrt(theta * theta + 1.0));
                const double c = 1.0 / std::sqrt(t * t + 1.0), sn = t * c;
                for (int k = 0; k < d; ++k) {
                    const double akp = A[k * d + p], akq = A[k * d + q];
                    A[k * d + p] = c * akp - sn * akq;
                    A[k * d + q] = sn * akp + c * akq;
                }
                for (int k = 0; k < d; ++k) {
                    const double apk = A[p * d + k], aqk = A[q * d + k];
                    A[p * d + k] = c * apk - sn * aqk;
                    A[q * d + k] = sn * apk + c * aqk;
                }
                for (int k = 0; k < d; ++k) {
                    const double vkp = V[k * d + p], vkq = V[k * d + q];
                    V[k * d + p] = c * vkp - sn * vkq;
                    V[k * d + q] = sn * vkp + c * vkq;
                }
            }
    }
    F.assign((size_t)d * d, 0.0);
    for (int k = 0; k < d; ++k) {
        double lam = A[k * d + k];
        if (lam < -1e-10) return false;
        lam = lam > 0 ? std::sqrt(lam) : 0.0;
        for (int i = 0; i < d; ++i) F[i * d + k] = V[i * d + k] * lam;
    }
    return true;
}

// ---- host: factor cache, preparation, batched launch ------------------------

// Process-wide cache of factorised baskets (Cholesky or eigen factor plus the
// per-asset constants), found by a hash of everything they depend on; an
// entry keeps that full key and is used only when it equals the request's
// (a hash collision is a miss).  id is unique per entry and never reused, so
// the contexts' device slots are keyed by it.
struct BasketConsts {
    std::vector<char> blob;
    std::vector<double> key;
    uint64_t id = 0;
    BasketLayout lay;
    bool full;
    bool one;  // columns constant below the diagonal
};

std::atomic<uint64_t>& consts_next_id() {
    static std::atomic<uint64_t> n{1};
    return n;
}
std::atomic<uint64_t>& consts_hash_mask() {
    static std::atomic<uint64_t> m{~0ull};
    return m;
}

uint64_t fnv(uint64_t h, const void* p, size_t n) {
    const unsigned char* c = (const unsigned char*)p;
    for (size_t i = 0; i < n; ++i) {
        h ^= c[i];
        h *= 1099511628211ull;
    }
    return h;
}

std::mutex& consts_mu() {
    static std::mutex m;
    return m;
}
std::map<uint64_t, std::shared_ptr<BasketConsts>>& consts_cache() {
    static std::map<uint64_t, std::shared_ptr<BasketConsts>> c;
    return c;
}

struct BasketPrep {
    BasketArgs a;
    int mode, B, nblk, dmax;
    bool mfma, full, one;
    int nb;  // blocks of 16 assets (MFMA)
    uint64_t key;  // the constants' entry id (device slots are keyed by it)
    std::shared_ptr<BasketConsts> consts;
    double disc;
};

int basket_prepare(pcf_ctx* ctx, const pcf_request& q, BasketPrep& p) {
    const pcf_opts& o = q.opts;
    int st = pcf_check_common(ctx, q.S0, q.E, q.r, q.sigma, q.T, q.N, q.payoff_fun);
    if (st) return st;
    if ((st = pcf_check_opts(ctx, &o))) return st;
    const int d = q.assets;
    if (d < 1 || d > kMaxAssets)
        return pcf_fail(ctx, PCF_ERR_INVALID_ARG, "assets must be in [1, %d] (got %d)", kMaxAssets, d);
    const pcf_basket_ext* ext = q.basket;
    // Key of the constants: d, rho, r, T, sqrt(T) convention, scalar sigma/S0
    // and every extension array (absent arrays marked by a NaN-free flag).
    const int refx = o.ref_exact ? 1 : 0;
    const double* arrs[4] = {ext ? ext->sigma : nullptr, ext ? ext->S0 : nullptr,
                             ext ? ext->weights : nullptr, ext ? ext->corr : nullptr};
    std::vector<double> key = {(double)d, q.rho, q.r, q.T, q.sigma, q.S0, (double)refx};
    for (int k = 0; k < 4; ++k) {
        key.push_back(arrs[k] ? 1.0 : 0.0);
        if (arrs[k]) key.insert(key.end(), arrs[k], arrs[k] + (k == 3 ? (size_t)d * d : (size_t)d));
    }
    const uint64_t h = fnv(1469598103934665603ull, key.data(), key.size() * sizeof(double)) &
                       consts_hash_mask().load(std::memory_order_relaxed);
    std::shared_ptr<BasketConsts> c;
    {
        std::lock_guard<std::mutex> lk(consts_mu());
        auto it = consts_cache().find(h);
        // bitwise comparison of the full key: a hash collision is a miss
        if (it != consts_cache().end() && it->second->key.size() == key.size() &&
            std::memcmp(it->second->key.data(), key.data(), key.size() * sizeof(double)) == 0)
            c = it->second;
    }
    if (!c) {
        // Correlation matrix: ext->corr or equicorrelation rho (include/mvn.h:55-60).
        std::vector<double> C((size_t)d * d);
        for (int i = 0; i < d; ++i)
            for (int k = 0; k < d; ++k) {
                const double v = (ext && ext->corr) ? ext->corr[i * d + k] : (i != k ? q.rho : 1.0);
                if (!std::isfinite(v)) return pcf_fail(ctx, PCF_ERR_INVALID_ARG, "non-finite correlation");
                C[(size_t)i * d + k] = v;
            }
        for (int i = 0; i < d; ++i)
            for (int k = 0; k < i; ++k)
                if (std::fabs(C[i * d + k] - C[k * d + i]) > 1e-12)
                    return pcf_fail(ctx, PCF_ERR_INVALID_ARG, "correlation matrix is not symmetric");
        std::vector<double> L;
        bool full = false;
        if (!cholesky(d, C, L)) {
            if (!eigen_factor(d, C, L))
                return pcf_fail(ctx, PCF_ERR_INVALID_ARG, "correlation matrix is not positive semi-definite");
            full = true;
        }
        c = std::make_shared<BasketConsts>();
        c->full = full;
        c->one = !full;
        for (int k = 0; k < d && c->one; ++k)
            for (int i = k + 2; i < d; ++i) c->one = c->one && L[(size_t)i * d + k] == L[(size_t)(k + 1) * d + k];
        c->key = key;
        c->id = consts_next_id().fetch_add(1);
        c->lay = BasketLayout::make(d);
        c->blob.assign(c->lay.bytes, 0);
        char* hb = c->blob.data();
        const BasketLayout& lay = c->lay;
        double* L64 = (double*)(hb + lay.off_L64);
        double* c064 = (double*)(hb + lay.off_c064);
        double* c164 = (double*)(hb + lay.off_c164);
        double* ws64 = (double*)(hb + lay.off_ws64);
        float* Lf = (float*)(hb + lay.off_Lf);
        float* c0f = (float*)(hb + lay.off_c0f);
        float* c1f = (float*)(hb + lay.off_c1f);
        float* wsf = (float*)(hb + lay.off_wsf);
        const double log2e = 1.4426950408889634;
        const double sqT = refx ? 1.0 : std::sqrt(q.T);
        const double w_i = 1.0 / (double)d;
        for (int i = 0; i < d * d; ++i) {
            L64[i] = L[i];
            Lf[i] = (float)L[i];
        }
        for (int i = 0; i < d; ++i) {
            const double sg = (ext && ext->sigma) ? ext->sigma[i] : q.sigma;
            const double s0 = (ext && ext->S0) ? ext->S0[i] : q.S0;
            const double wt = (ext && ext->weights) ? ext->weights[i] : w_i;
            if (!(sg >= 0) || !std::isfinite(sg) || !std::isfinite(s0) || !std::isfinite(wt))
                return pcf_fail(ctx, PCF_ERR_INVALID_ARG, "bad per-asset parameter at %d", i);
            // (w_i*S0)*exp((r-pow(sigma,2)/2)*T + sigma*B)  (src/mc_eur_multi.cpp:30)
            c064[i] = (q.r - libm_pow(sg, 2) / 2) * q.T;
            c164[i] = sg * sqT;
            ws64[i] = wt * s0;
            c0f[i] = (float)(c064[i] * log2e);
            c1f[i] = (float)(c164[i] * log2e);
            wsf[i] = (float)ws64[i];
        }
        if (c->one) {
            double* k64 = (double*)(hb + lay.off_one64);
            float* k32 = (float*)(hb + lay.off_one32);
            for (int i = 0; i < d; ++i) {
                const int at = 20 * (i / 4) + i % 4;
                const double below = i + 1 < d ? L[(size_t)(i + 1) * d + i] : 0.0;
                const double v64[5] = {below, L[(size_t)i * d + i], c064[i], c164[i], ws64[i]};
                const float v32[5] = {(float)below, (float)L[(size_t)i * d + i], c0f[i], c1f[i], wsf[i]};
                for (int t = 0; t < 5; ++t) {
                    k64[at + 4 * t] = v64[t];
                    k32[at + 4 * t] = v32[t];
                }
            }
        }
        std::lock_guard<std::mutex> lk(consts_mu());
        if (consts_cache().size() > 1024) consts_cache().clear();
        consts_cache()[h] = c;
    }
    p.consts = c;
    p.key = c->id;
    p.full = c->full;
    p.mode = o.rng == PCF_RNG_HOST ? kHost : (o.precision == PCF_FP64 ? kFp64 : kFp32k);
    if (o.kernel_variant == 2 && !(p.mode == kFp32k && d >= 16 && d <= 32))
        return pcf_fail(ctx, PCF_ERR_INVALID_ARG, "kernel_variant 2 (MFMA basket kernel) is taken for FP32/Philox and 16 <= assets <= 32");
    p.one = c->one && p.mode != kHost && o.kernel_variant == 0;
    p.mfma = !p.one && p.mode != kHost && d >= kMfmaFrom && o.kernel_variant != 1;
    p.nb = p.mfma ? (d + 15) / 16 : 0;
    p.dmax = p.one || p.mfma ? 0 : d <= 4 ? 4 : d <= 8 ? 8 : d <= 16 ? 16 : d <= 32 ? 32 : 64;
    BasketArgs& a = p.a;
    a = BasketArgs{};
    a.E = q.E;
    a.pf = q.payoff_fun;
    a.Ef = (float)q.E;
    a.pff = (float)q.payoff_fun;
    a.N = q.N;
    a.d = d;
    a.full = p.full ? 1 : 0;
    a.seed = o.seed;
    // Built-in shape: the MFMA kernel's items are 16-path tiles, one wavefront
    // per tile at a time.  Picoseconds a path, measured: prefix form 1.3 + 0.53 d
    // (FP64 1 + 2 d), MFMA 0.9 per padded asset (FP64 3.5), general about 1.5 +
    // 0.6 d + 0.03 d^2 (FP64 1 + 2 d + 0.1 d^2).
    const int64_t ntiles = (q.N + 15) / 16;
    const double dd = d;
    const bool f32 = p.mode == kFp32k;
    const double ps = p.mfma ? 16 * (f32 ? 0.9 : 3.5) * (16 * p.nb)
                      : p.one ? (f32 ? 1.3 + 0.53 * dd : 1.0 + 2.0 * dd)
                              : (f32 ? 1.5 + 0.6 * dd + 0.03 * dd * dd : 1.0 + 2.0 * dd + 0.1 * dd * dd);
    int B = 256;
    int ipt = p.mfma ? pcf_items_per_thread(ntiles, B / 64, ctx->cu_count, ps)
                     : pcf_items_per_thread(q.N, B, ctx->cu_count, ps);
    // Tuned shapes: the prefix form and the general kernel have their own; the
    // MFMA entry is measured with two blocks of 16 assets and holds for those.
    const int tuned = p.one ? 6 + p.mode : !p.mfma ? 2 * p.mode : p.nb == 2 ? 2 * p.mode + 1 : -1;
    pcf_tuned_shape(PCF_KIND_BASKET, tuned, q.N, &B, &ipt);
    if (o.block_size) B = o.block_size;
    if (o.items_per_thread) ipt = o.items_per_thread;
    if (B > kBasketThreads)
        return pcf_fail(ctx, PCF_ERR_INVALID_ARG, "mc_eur_multi takes at most %d threads per block (block_size %d)",
                        kBasketThreads, B);
    p.B = B;
    p.nblk = p.mfma ? pcf_blocks_for(ntiles, B / 64, ipt) : pcf_blocks_for(q.N, B, ipt);
    p.disc = std::exp(-q.r * q.T);
    return PCF_OK;
}

// Device-resident constants: fixed-size slots in ctx->basket_L, LRU by stamp.
constexpr size_t kConstSlot = kBasketConstSlot;
constexpr int kConstSlots = kMaxBatch;

// *sequence: set, and its begin recorded, when this copies constants to the device.
int resident_consts(pcf_ctx* ctx, const BasketPrep& p, uint64_t batch_stamp, char** dev, bool* sequence) {
    auto& bc = ctx->basket_cache;
    if (bc.key.empty()) {
        bc.key.assign(kConstSlots, 0);
        bc.stamp.assign(kConstSlots, 0);
        PCF_HIP_CHECK(ctx, ctx->basket_L.ensure(kConstSlot * kConstSlots));
    }
    auto it = bc.where.find(p.key);
    int slot;
    if (it != bc.where.end()) {
        slot = it->second;
    } else {
        slot = -1;
        for (int s = 0; s < kConstSlots; ++s)
            if (bc.stamp[s] < batch_stamp && (slot < 0 || bc.stamp[s] < bc.stamp[slot])) slot = s;
        if (slot < 0) return pcf_fail(ctx, PCF_ERR_INVALID_ARG, "too many distinct baskets in one batch");
        if (bc.key[slot]) bc.where.erase(bc.key[slot]);
        bc.key[slot] = p.key;
        bc.where[p.key] = slot;
        if (p.consts->blob.size() > kConstSlot) return pcf_fail(ctx, PCF_ERR_INVALID_ARG, "basket too large");
        if (!*sequence) {
            const int st = pcf_timing_begin(ctx);
            if (st) return st;
            *sequence = true;
        }
        PCF_HIP_CHECK(ctx, hipMemcpyAsync(ctx->basket_L.as<char>() + kConstSlot * slot, p.consts->blob.data(),
                                          p.consts->blob.size(), hipMemcpyHostToDevice, ctx->stream));
    }
    bc.stamp[slot] = ++bc.clock;
    *dev = ctx->basket_L.as<char>() + kConstSlot * slot;
    return PCF_OK;
}

template <typename Real, int NB>
void launch_mfma_n(pcf_ctx* ctx, unsigned int grid, int B, const pcf::JobArgs<BasketJob>& ja, bool full) {
    if (full) k_basket_mfma<Real, NB, true><<<grid, B, 0, ctx->stream>>>(ja);
    else k_basket_mfma<Real, NB, false><<<grid, B, 0, ctx->stream>>>(ja);
}

template <typename Real>
void launch_mfma(pcf_ctx* ctx, unsigned int grid, int B, const pcf::JobArgs<BasketJob>& ja, bool full, int nb) {
    if (nb == 1) launch_mfma_n<Real, 1>(ctx, grid, B, ja, full);
    else if (nb == 2) launch_mfma_n<Real, 2>(ctx, grid, B, ja, full);
    else if (nb == 3) launch_mfma_n<Real, 3>(ctx, grid, B, ja, full);
    else launch_mfma_n<Real, 4>(ctx, grid, B, ja, full);
}

template <typename Real, int DMAX, int MODE>
void launch_fma(pcf_ctx* ctx, unsigned int grid, int B, const pcf::JobArgs<BasketJob>& ja, bool full) {
    if (full) k_basket_fma<Real, DMAX, MODE, true><<<grid, B, 0, ctx->stream>>>(ja);
    else k_basket_fma<Real, DMAX, MODE, false><<<grid, B, 0, ctx->stream>>>(ja);
}

template <typename Real, int MODE>
void launch_fma_d(pcf_ctx* ctx, unsigned int grid, int B, const pcf::JobArgs<BasketJob>& ja, bool full, int dmax) {
    if (dmax == 4) launch_fma<Real, 4, MODE>(ctx, grid, B, ja, full);
    else if (dmax == 8) launch_fma<Real, 8, MODE>(ctx, grid, B, ja, full);
    else if (dmax == 16) launch_fma<Real, 16, MODE>(ctx, grid, B, ja, full);
    else if (dmax == 32) launch_fma<Real, 32, MODE>(ctx, grid, B, ja, full);
    else launch_fma<Real, 64, MODE>(ctx, grid, B, ja, full);
}

}  // namespace

uint64_t pcf_basket_batch_key(pcf_ctx* ctx, const pcf_request& q, int* status) {
    BasketPrep p;
    *status = basket_prepare(ctx, q, p);
    if (*status) return 0;
    const int variant = p.mfma ? 200 + 2 * p.nb + (p.full ? 1 : 0) : p.one ? 2 : (2 + (p.full ? 1 : 0) + 2 * p.dmax);
    return pcf_make_batch_key(PCF_KIND_BASKET, p.mode, variant, p.B);
}

int pcf_basket_run(pcf_ctx* ctx, int n, const pcf_request* const* reqs, pcf_result* res, int* status) {
    if (n < 1 || n > kMaxBatch) return pcf_fail(ctx, PCF_ERR_INVALID_ARG, "batch size %d", n);
    PCF_HIP_CHECK(ctx, hipSetDevice(ctx->device));
    static thread_local BasketPrep prep[kMaxBatch];
    int live[kMaxBatch], nl = 0;
    for (int i = 0; i < n; ++i) {
        res[i] = pcf_result{};
        status[i] = basket_prepare(ctx, *reqs[i], prep[i]);
        if (status[i] == PCF_OK) live[nl++] = i;
    }
    if (nl == 0) return PCF_OK;
    const BasketPrep& p0 = prep[live[0]];
    int64_t nparts = 0, nb = 0, nnorm = 0;
    for (int k = 0; k < nl; ++k) {
        const BasketPrep& p = prep[live[k]];
        if (p.mode != p0.mode || p.B != p0.B || p.mfma != p0.mfma || p.one != p0.one || p.nb != p0.nb || p.dmax != p0.dmax ||
            p.full != p0.full)
            return pcf_fail(ctx, PCF_ERR_INVALID_ARG, "mixed batch keys");
        nparts += (int64_t)p.nblk * 2;
        nb += p.nblk;
        if (p.mode == kHost) nnorm += reqs[live[k]]->N * (int64_t)reqs[live[k]]->assets;
    }
    if (nb > (1ll << 30)) return pcf_fail(ctx, PCF_ERR_INVALID_ARG, "batch too large");
    // A lone job on device normals is one launch; anything more is a sequence
    // that is timed by events.
    bool sequence = nl > 1 || nnorm > 0;
    int st = PCF_OK;
    if (sequence && (st = pcf_timing_begin(ctx))) return st;
    PCF_HIP_CHECK(ctx, ctx->partials.ensure((size_t)nparts * sizeof(pcf::CSum)));
    if (nnorm) PCF_HIP_CHECK(ctx, ctx->normals.ensure((size_t)nnorm * sizeof(double)));
    BasketJob* jobs = (BasketJob*)ctx->h_jobs;
    const uint64_t batch_stamp = ctx->basket_cache.clock + 1;
    int64_t poff = 0, noff = 0;
    unsigned int boff = 0;
    for (int k = 0; k < nl; ++k) {
        const int i = live[k];
        const BasketPrep& p = prep[i];
        char* dev = nullptr;
        if ((st = resident_consts(ctx, p, batch_stamp, &dev, &sequence))) return st;
        const BasketLayout& lay = p.consts->lay;
        const bool f64 = p.mode != kFp32k;
        BasketJob& J = jobs[k];
        J.a = p.a;
        J.Lm = dev + (p.one ? (f64 ? lay.off_one64 : lay.off_one32) : f64 || p.mfma ? lay.off_L64 : lay.off_Lf);
        J.c0 = dev + (f64 ? lay.off_c064 : lay.off_c0f);
        J.c1 = dev + (f64 || p.mfma ? lay.off_c164 : lay.off_c1f);
        J.ws = dev + (f64 ? lay.off_ws64 : lay.off_wsf);
        J.hz = nullptr;
        if (p.mode == kHost) {
            const pcf_opts& o = reqs[i]->opts;
            const int64_t cnt = reqs[i]->N * (int64_t)reqs[i]->assets;
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
        poff += (int64_t)p.nblk * 2;
        boff += (unsigned int)p.nblk;
    }
    if (nl > 1)
        PCF_HIP_CHECK(ctx, hipMemcpyAsync(ctx->jobs.ptr, jobs, sizeof(BasketJob) * nl, hipMemcpyHostToDevice, ctx->stream));
    const pcf::JobArgs<BasketJob> ja{jobs[0], ctx->jobs.as<BasketJob>(), nl};
    pcf_arm_results(ctx, nl);
    double work = 0.0;
    for (int k = 0; k < nl; ++k) work += (double)reqs[live[k]]->N * (double)reqs[live[k]]->assets;
    std::unique_lock<std::mutex> order;  // held until the end event is recorded
    PCF_HIP_CHECK(ctx, pcf_after_persistent(ctx, p0.mode == kFp32k ? work : kPersistentGateFp64 * work, &order));
    if (p0.one && p0.mode == kFp32k)
        k_basket_one<float><<<boff, p0.B, 0, ctx->stream>>>(ja);
    else if (p0.one)
        k_basket_one<double><<<boff, p0.B, 0, ctx->stream>>>(ja);
    else if (p0.mfma)
        p0.mode == kFp32k ? launch_mfma<float>(ctx, boff, p0.B, ja, p0.full, p0.nb)
                          : launch_mfma<double>(ctx, boff, p0.B, ja, p0.full, p0.nb);
    else if (p0.mode == kFp32k)
        launch_fma_d<float, kFp32k>(ctx, boff, p0.B, ja, p0.full, p0.dmax);
    else if (p0.mode == kFp64)
        launch_fma_d<double, kFp64>(ctx, boff, p0.B, ja, p0.full, p0.dmax);
    else
        launch_fma_d<double, kHost>(ctx, boff, p0.B, ja, p0.full, p0.dmax);
    PCF_HIP_CHECK(ctx, hipGetLastError());
    PCF_HIP_CHECK(ctx, hipEventRecord(ctx->ev_kend, ctx->stream));
    if (order.owns_lock()) order.unlock();
    pcf_result timing{};
    if ((st = pcf_wait_results(ctx, nl, 4, ctx->stream, &timing.kernel_ms))) return st;
    timing.total_ms = timing.kernel_ms;
    if (sequence && (st = pcf_sequence_ms(ctx, ctx->ev_kend, &timing.total_ms))) return st;
    for (int k = 0; k < nl; ++k) {
        const int i = live[k];
        const BasketPrep& p = prep[i];
        const double* h = ctx->h_out + (size_t)kOutPerJob * k;
        const int64_t N = reqs[i]->N;
        const double d = reqs[i]->assets;
        pcf_result& r = res[i];
        // The reference returns (exp(-r*T)*result)/(double)N (src/mc_eur_multi.cpp:34).
        r.price = (p.disc * h[0]) / (double)N;
        r.mean = h[2];
        r.variance = h[3];
        r.std_err = p.disc * std::sqrt(h[3] / (double)N);
        r.n_paths = N;
        r.n_steps = 1;
        r.kernel_ms = timing.kernel_ms;
        r.total_ms = timing.total_ms;
        // d^2 + 12 d + 3 algorithmic flops per path: normals 6d, triangular
        // Z L^T d(d+1), per asset FMA + exp + FMA 5d, payoff 3 (the
        // algorithm's count, whichever kernel runs; the prefix form does 15 d + 3).
        r.flops = (d * d + 12.0 * d + 3.0) * (double)N;
        r.bytes = p.mode == kHost ? 8.0 * d * (double)N : 0.0;
        r.grid_blocks = p.nblk;
        r.block_size = p.B;
        r.batch_size = nl;
        r.lsm_fallback = p.full ? 1 : 0;
    }
    for (int k = 0; k < nl; ++k) prep[live[k]].consts.reset();
    return PCF_OK;
}

extern "C" int pcf_mc_eur_multi(pcf_ctx* ctx, double S0, double E, double r, double sigma,
                                double T, int64_t N, double payoff_fun, int32_t assets, double rho,
                                const pcf_basket_ext* ext, const pcf_opts* opts, pcf_result* res) {
    if (!ctx || !res) return PCF_ERR_INVALID_ARG;
    std::lock_guard<std::recursive_mutex> lk(ctx->mu);
    pcf_request q = pcf_make_request(PCF_KIND_BASKET, S0, E, r, sigma, T, N, payoff_fun, opts);
    q.assets = assets;
    q.rho = rho;
    q.basket = ext;
    const pcf_request* qp = &q;
    int status = PCF_OK;
    int st = pcf_basket_run(ctx, 1, &qp, res, &status);
    if (st || status) return st ? st : status;
    return pcf_apply_fp64_check(ctx, q, res);
}

extern "C" void pcf_debug_basket_hash_mask(uint64_t mask) {
    consts_hash_mask().store(mask, std::memory_order_relaxed);
}

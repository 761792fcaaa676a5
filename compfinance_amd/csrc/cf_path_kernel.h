// HIP path kernels for gfx950 (MI355X): Sobol -> inverse normal -> model
// step -> product, one path per lane, forward (pricing) and forward +
// hand-written adjoint (risk).
//
// Reference semantics followed: sobol.h:55-151, gaussians.h:47-87,
// interp.h:26-63, mcMdlDupire.h:238-280, mcMdlBS.h:321-350,
// mcPrd.h:113-125, :235-288, :374-399; the adjoint reproduces the derivative
// conventions of the reference tape (AADExpr.h:115-253, :364-598).
//
// Block organisation
//   * a persistent grid; wave w of the grid takes Sobol blocks q = w, w + W, ...
//     of 64 consecutive Sobol indices n = 64q + lane (path p = n - 1);
//   * Gray code splits as gray(64q + r) = gray6(r) ^ (q & 1) << 5 ^ gray(q) << 6,
//     so the point of lane r in dimension d is  LO[d][r] ^ HI_q[d]:  LO is a
//     per-block LDS table built once, HI_q a per-wave LDS row built per block
//     of paths;
//   * local-vol table, interval table, knot search table and timeline sample
//     map in LDS (the LEAN layout of long timelines and large grids reads the
//     local-vol and knot search tables from global memory through L1 instead);
//     the FP32 inverse-normal table through L1 or in LDS (GINV);
//   * FP64 draws four steps at a time, the inverse normal's tail form
//     evaluated once per wave for the lanes that need it (a per-wave LDS row
//     of 64 doubles, 32 in the LEAN layout);
//   * mrg32k3a instead of Sobol: one generator per lane in registers, jumped
//     to its path's block of numbers and stepped back in the reverse sweeps;
//   * payoffs reduced per wave with DPP cross-lane moves into per-wave LDS
//     accumulators, then per block, then across blocks in fixed order by the
//     last block or a separate kernel (fused_reduction);
//   * adjoint: path states checkpointed in a per-wave HBM slot (reused by the
//     wave for each block of paths) with the knot bracket of each state in a
//     byte, reverse sweep over the Euler steps,
//     local-vol adjoints accumulated with LDS atomics on a per-block
//     (step x spot) grid.
// This header holds the device helpers and the path kernel template; each
// cf_kern_inst.hip build instantiates one (precision, adjoint, source of
// normals: Sobol or mrg32k3a) family.
#pragma once

#include <hip/hip_runtime.h>

#include <type_traits>

#include "cf_internal.h"

namespace cfk {

// ------------------------------------------------------------------ helpers

// One DPP move of an FP64 value (both halves, the same lane pattern); lanes
// the pattern does not write, or whose source lies outside the row, read 0.
template <int CTRL, int ROW_MASK>
__device__ __forceinline__ double dpp_f64(double v)
{
    const unsigned long long u = __builtin_bit_cast(unsigned long long, v);
    const int lo = __builtin_amdgcn_update_dpp(0, int(u & 0xffffffffu), CTRL, ROW_MASK, 0xf, true);
    const int hi = __builtin_amdgcn_update_dpp(0, int(u >> 32), CTRL, ROW_MASK, 0xf, true);
    return __builtin_bit_cast(double, (static_cast<unsigned long long>(unsigned(hi)) << 32) | unsigned(lo));
}

// The wave's sum lands in this lane.
constexpr int kSumLane = kWave - 1;

// FP64 sum over the wave by data-parallel primitives in registers (no LDS):
// prefix sums of 2, 4, 8 and 16 lanes within each row of 16 (row_shr), then
// row 0's sum into row 1 and row 2's into row 3 (row_bcast:15), then rows
// 0-1 into rows 2-3 (row_bcast:31).  The total is valid in lane kSumLane
// only; the order of the additions is fixed, so the sum is reproducible.
__device__ __forceinline__ double wave_sum(double v)
{
    v += dpp_f64<0x111, 0xf>(v);   // row_shr:1
    v += dpp_f64<0x112, 0xf>(v);   // row_shr:2
    v += dpp_f64<0x114, 0xf>(v);   // row_shr:4
    v += dpp_f64<0x118, 0xf>(v);   // row_shr:8
    v += dpp_f64<0x142, 0xa>(v);   // row_bcast:15 into rows 1 and 3
    v += dpp_f64<0x143, 0xc>(v);   // row_bcast:31 into rows 2 and 3
    return v;
}

__device__ __forceinline__ void wave_sync_lds()
{
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// Read-only global data read with wave-uniform indices: a pointer into the
// constant address space, which the compiler reads with scalar loads through
// the scalar cache into scalar registers.
template <typename T>
using CPtr = const __attribute__((address_space(4))) T*;
template <typename T>
__device__ __forceinline__ CPtr<T> cptr(const void* p)
{
    return (CPtr<T>)(p);
}

// Maximum and minimum in one instruction (the builtins first quiet their
// operands, one more instruction each); a NaN gives the other operand.
__device__ __forceinline__ double max_f64(double a, double b)
{
    double r;
    asm("v_max_f64 %0, %1, %2" : "=v"(r) : "v"(a), "v"(b));
    return r;
}
__device__ __forceinline__ double min_f64(double a, double b)
{
    double r;
    asm("v_min_f64 %0, %1, %2" : "=v"(r) : "v"(a), "v"(b));
    return r;
}
// a b + c with c a constant in a scalar register pair, in one instruction (the
// compiler keeps a polynomial's constants in vector registers where scalar
// ones run short and copies each before a two-address multiply-add)
__device__ __forceinline__ double fma_s(double a, double b, double c)
{
    double r;
    asm("v_fma_f64 %0, %1, %2, %3" : "=v"(r) : "v"(a), "v"(b), "s"(c));
    return r;
}

// a / b in FP64 from the hardware reciprocal (relative error e below 2^-22):
// one third-order step r (1 + e + e^2), whose error e^3 is far under an ulp,
// and a residual correction of the quotient (within an ulp of the IEEE
// quotient, which it equals but for rare last-bit cases).  Seven
// instructions; two Newton steps take eight and the compiler's IEEE division
// twelve.
__device__ __forceinline__ double fast_div(double a, double b)
{
    double r = __builtin_amdgcn_rcp(b);
    const double e = fma(-b, r, 1.0);
    r = fma(r, fma(e, e, e), r);
    const double q = a * r;
    return fma(fma(-b, q, a), r, q);
}

// Beasley-Springer-Moro inverse normal (gaussians.h:47-87), FP64, same
// branches and constants as the reference: the central rational form of
// x = p - 1/2 for |x| < 0.42 (an odd function of x), else the tail polynomial
// in log(-log(v)) of v = min(p, 1 - p).  The tail is read from a table of
// polynomials of degree 11 on the quarters of the binades of v
// (moro_tail_f64.inc, written by gen_moro_tail_f64.py in extended precision):
// within 2.0 half-ulps of the exact tail (0.48 on average) over the Sobol
// words, where two logarithms and the polynomial in double round to 4.1
// (0.75), for 18 instructions and six 16-byte reads instead of 95
// instructions.
alignas(16) static __constant__ double kMoroTailF64[kMoroTailRows * kMoroTailCoefs] = {
#include "moro_tail_f64.inc"
};
__device__ __forceinline__ double moro_central(double x)
{
    const double r = x * x;
    return fast_div(x * (((-25.44106049637 * r + 41.39119773534) * r + -18.61500062529) * r + 2.50662823884),
                    (((3.13082909833 * r + -21.06224101826) * r + 23.08336743743) * r + -8.47351093090) * r + 1.0);
}
// the row's polynomial from its coefficients c, and the distance to its midpoint
__device__ __forceinline__ double moro_tail_row(double v, const double* row)
{
    const uint32_t hi = uint32_t(__builtin_bit_cast(uint64_t, v) >> 32);
    const double mid = __builtin_bit_cast(double, uint64_t((hi & 0xfffc0000u) | 0x20000u) << 32);
    const double d = v - mid;   // exact
    const double2* c = reinterpret_cast<const double2*>(row);
    double r = fma(c[5].y, d, c[5].x);
#pragma unroll
    for (int k = 4; k >= 0; --k) r = fma(fma(r, d, c[k].y), d, c[k].x);
    return r;
}
// (a mass outside the table, which only an idle lane's word 0 gives, takes an
// end row)
__device__ __forceinline__ int moro_row(double v)
{
    return min(max(int(uint32_t(__builtin_bit_cast(uint64_t, v) >> 32) >> 18) - kMoroTailBias, 0), kMoroTailRows - 1);
}
__device__ __forceinline__ double moro_tail(double v)
{
    return moro_tail_row(v, kMoroTailF64 + moro_row(v) * kMoroTailCoefs);
}
__device__ __forceinline__ double inv_normal_p(double p)
{
    const double x = p - 0.5;
    double z = moro_central(x);
    if (!(fabs(x) < 0.42)) z = __builtin_copysign(moro_tail(min_f64(p, 1.0 - p)), x);
    return z;
}

// of the Sobol uniform u = ONEOVER2POW32 * xi (sobol.h:26, :110-116)
__device__ __forceinline__ double inv_normal(uint32_t xi, const double*)
{
    return inv_normal_p(2.3283064365387E-10 * double(xi));
}

// FP32 form: v = min(u, 1 - u) is formed exactly in the integer domain as
// xs = 2^32 v in [1, 2^31]; the IEEE bits of float(xs) give the table row
// (exponent and top three mantissa bits: one eighth of a binade of v) and
// t in [-1, 1) (the low 20 mantissa bits).  Each row is a cubic in t fitted
// to the same Moro function in FP64 (inv_normal_f32.inc, written by
// gen_inv_normal_f32.py).  No logarithm, no branch: one 16-byte table read
// and three FMAs.  Differences to the FP64 Moro values are below 5e-7 (the FP32
// rounding of the result in the far tail).
// `tabm` is the table's address less 1016 rows (kInvNormalRowBias): row r of
// the table is at tabm + 4 (r + 1016), so the row address is formed from the
// float's bits by one mask and one add.
constexpr int kInvNormalRowBias = 127 << 3;
__device__ __forceinline__ float inv_normal(uint32_t xi, const float* tabm)
{
    // 2^32 min(u, 1 - u) is |xi| as signed integers (xi < 0 exactly when
    // u >= 1/2, and 2^31 maps to itself): one conversion gives its float, with
    // the sign of 1/2 - u in the sign bit.  xi = 0 would give row -1016: the
    // kernel never passes it (only Sobol index 0 has a zero word, and its lane
    // reads 2^31 instead)
    const uint32_t bits = __float_as_uint(float(int(xi)));
    // row (bits >> 20) - 1016 in [0, kInvNormalRows - 1], 16 bytes a row
    const float4 c = *reinterpret_cast<const float4*>(tabm + ((bits >> 18) & 0x1ffcu));
    // the row's argument m / 2^19 - 1 of the float's last 20 bits m, exactly:
    // as the mantissa of a float in [4, 4.5)
    const float t = fmaf(__uint_as_float((bits & 0xfffffu) | 0x40800000u), 4.0f, -17.0f);
    const float p = fmaf(fmaf(fmaf(c.w, t, c.z), t, c.y), t, c.x);
    return __uint_as_float(__float_as_uint(p) ^ (bits & 0x80000000u));   // -p for u >= 1/2
}

// Four FP64 normals of this lane's uniforms, with Moro's tail evaluated once
// per wave.  About 16% of draws need the tail, so a wave of 64 lanes almost
// always has one that does and, draw by draw, every lane would run it.  Here
// every lane runs the central form of its four draws; the tail masses of the
// wave, counted by ballots, go to `row` (this wave's ROW doubles of LDS) by
// their rank, each lane evaluates at most one, and the owners read their
// values back (in rounds of ROW when more draws need the tail: 41 on
// average, more than 64 once in 20,000 groups).  The values equal
// inv_normal_p's, draw by draw.  LTAB: `tab` holds the table's rows from
// kMoroLdsRow on in LDS (through L1 the reads would wait for the checkpoint
// stores issued before them: one counter orders loads and stores); a wave with
// a mass below them, 12% of the groups, reads the whole table through L1.
template <int ROW, bool LTAB>
__device__ __forceinline__ void inv_normal4_p(const double p[4], double z[4], double* row, const double* tab, int lane)
{
    static_assert(ROW >= 1 && ROW <= kWave, "a row of at most one double per lane");
    bool tail[4];
    int pos[4];    // rank of this lane's draw among the wave's tail draws
    int total = 0;
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        const double x = p[k] - 0.5;
        tail[k] = !(fabs(x) < 0.42);
        z[k] = moro_central(x);
        const uint64_t m = __builtin_amdgcn_ballot_w64(tail[k]);
        pos[k] = int(__builtin_amdgcn_mbcnt_hi(uint32_t(m >> 32), __builtin_amdgcn_mbcnt_lo(uint32_t(m), uint32_t(total))));
        total += __builtin_popcountll(m);
    }
    for (int r0 = 0; r0 < total; r0 += ROW) {
#pragma unroll
        for (int k = 0; k < 4; ++k)
            if (bool(tail[k] & (uint32_t(pos[k] - r0) < uint32_t(ROW)))) row[pos[k] - r0] = min_f64(p[k], 1.0 - p[k]);
        wave_sync_lds();
        if (lane < ROW && lane < total - r0) {
            const double v = row[lane];
            if constexpr (LTAB) {
                const int r = moro_row(v);
                if (__builtin_amdgcn_ballot_w64(r < kMoroLdsRow) == 0)
                    row[lane] = moro_tail_row(v, tab + (r - kMoroLdsRow) * kMoroTailCoefs);
                else
                    row[lane] = moro_tail_row(v, kMoroTailF64 + r * kMoroTailCoefs);
            } else {
                row[lane] = moro_tail(v);
            }
        }
        wave_sync_lds();
#pragma unroll
        for (int k = 0; k < 4; ++k)
            if (bool(tail[k] & (uint32_t(pos[k] - r0) < uint32_t(ROW))))
                z[k] = __builtin_copysign(row[pos[k] - r0], p[k] - 0.5);
        wave_sync_lds();
    }
}

// Of Sobol words (sobol.h:26, :110-116)
template <int ROW, bool LTAB>
__device__ __forceinline__ void inv_normal4_f64(const uint32_t w[4], double z[4], double* row, const double* tab, int lane)
{
    double p[4];
#pragma unroll
    for (int k = 0; k < 4; ++k) p[k] = 2.3283064365387E-10 * double(w[k]);
    inv_normal4_p<ROW, LTAB>(p, z, row, tab, lane);
}

// FP32 inverse-normal table: [rows][4 monomial coefficients]
static __constant__ float kInvNormalF32[kInvNormalRows * 4] = {
#include "inv_normal_f32.inc"
};

// ------------------------------------------------------------------ mrg32k3a

// L'Ecuyer's combined multiple recursive generator as the reference runs it
// (mrg32k3a.h:41-86), one generator per lane in registers:
//   x_n = a12 x_{n-2} - a13 x_{n-3}  mod m1,   y_n = a21 y_{n-1} - a23 y_{n-3}  mod m2,
// uniform (x_n - y_n) / (m1 + 1) folded into (0, 1).  Both moduli are
// 2^32 - c with small c, so a product r < 2^64 reduces by folds
// r -> (r >> 32) c + (r mod 2^32) (one 32 x 32 + 64 multiply-add each) and a
// last conditional subtraction.  Both recursions are invertible (a13, a23
// are units modulo the primes m1, m2), so the generator also steps back.
namespace mrg {
constexpr uint32_t kM1 = 4294967087u, kM2 = 4294944443u;
constexpr uint32_t kC1 = 209u, kC2 = 22853u;            // 2^32 - m
constexpr uint32_t kA12 = 1403580u, kA13 = 810728u;
constexpr uint32_t kA21 = 527612u, kA23 = 1370589u;
constexpr uint64_t pow_mod(uint64_t a, uint64_t e, uint64_t m)
{
    uint64_t r = 1;
    for (a %= m; e; e >>= 1, a = a * a % m)
        if (e & 1) r = r * a % m;
    return r;
}
constexpr uint32_t kInv13 = uint32_t(pow_mod(kA13, kM1 - 2, kM1));   // a13^-1 mod m1 (Fermat)
constexpr uint32_t kInv23 = uint32_t(pow_mod(kA23, kM2 - 2, kM2));   // a23^-1 mod m2
static_assert(uint64_t(kInv13) * kA13 % kM1 == 1 && uint64_t(kInv23) * kA23 % kM2 == 1, "inverses");

// r mod (2^32 - C) for any r < 2^64 (C < 2^15): the three folds leave
// r < 2^32 + C < 2 (2^32 - C)
template <uint32_t C>
__device__ __forceinline__ uint32_t reduce(uint64_t r)
{
    constexpr uint32_t M = uint32_t(0u - C);
#pragma unroll
    for (int k = 0; k < 3; ++k) r = uint64_t(uint32_t(r >> 32)) * C + uint32_t(r);
    return uint32_t(r >= M ? r - M : r);
}

// v = A v mod M, A a 3 x 3 matrix of residues (row-major), v residues
template <uint32_t C>
__device__ __forceinline__ void mat_vec(const uint64_t* __restrict__ A, uint32_t v[3])
{
    uint32_t r[3];
#pragma unroll
    for (int j = 0; j < 3; ++j) {
        uint32_t acc = 0;
#pragma unroll
        for (int l = 0; l < 3; ++l) acc = reduce<C>(uint64_t(uint32_t(A[3 * j + l])) * v[l] + acc);
        r[j] = acc;
    }
    v[0] = r[0];
    v[1] = r[1];
    v[2] = r[2];
}

// One lane's generator.  x[0], y[0] are the pos-th numbers of the lane's
// block (x[1], x[2] the two before); number pos feeds draw pos - 1.
struct Lane {
    uint32_t x[3], y[3];
    uint32_t x0[3], y0[3];   // the block's start state (pos 0)
    int pos;
    bool neg;                // odd path: the antithetic (negated) normals of its pair

    // Path p of a call (absolute index) draws from block p >> 1 of `dim`
    // numbers, negated for odd p (mrg32k3a.h:147-180); its start state is the
    // seed state advanced by (p >> 1) dim numbers through the jump matrices
    // A^(dim 2^j) of the set bits j (mrg32k3a.h:187-381; jump: 2 x 9 per j,
    // x then y).  Seeds are residues.
    __device__ __forceinline__ void start(const uint64_t* __restrict__ jump, uint32_t s1, uint32_t s2, int64_t p)
    {
        uint32_t xs[3] = {s1, s1, s1}, ys[3] = {s2, s2, s2};
        const uint64_t k = uint64_t(p) >> 1;
        for (int j = 0; j < 32 && (k >> j); ++j) {   // p < 2^32 (checked on the host)
            if ((k >> j) & 1) {
                mat_vec<kC1>(jump + size_t(18 * j), xs);
                mat_vec<kC2>(jump + size_t(18 * j + 9), ys);
            }
        }
#pragma unroll
        for (int l = 0; l < 3; ++l) {
            x[l] = x0[l] = xs[l];
            y[l] = y0[l] = ys[l];
        }
        pos = 0;
        neg = (p & 1) != 0;
    }
    __device__ __forceinline__ void forward()
    {
        // a12 x1 + a13 (m1 - x2) = x_n mod m1: both terms below 2^53
        const uint32_t xn = reduce<kC1>(uint64_t(kA12) * x[1] + uint64_t(kA13) * (kM1 - x[2]));
        const uint32_t yn = reduce<kC2>(uint64_t(kA21) * y[0] + uint64_t(kA23) * (kM2 - y[2]));
        x[2] = x[1]; x[1] = x[0]; x[0] = xn;
        y[2] = y[1]; y[1] = y[0]; y[0] = yn;
        ++pos;
    }
    __device__ __forceinline__ void back()
    {
        // x_{n-3} = (a12 x_{n-2} - x_n) / a13,  y_{n-3} = (a21 y_{n-1} - y_n) / a23
        const uint32_t dx = reduce<kC1>(uint64_t(kA12) * x[2] + (kM1 - x[0]));
        const uint32_t dy = reduce<kC2>(uint64_t(kA21) * y[1] + (kM2 - y[0]));
        const uint32_t xp = reduce<kC1>(uint64_t(dx) * kInv13);
        const uint32_t yp = reduce<kC2>(uint64_t(dy) * kInv23);
        x[0] = x[1]; x[1] = x[2]; x[2] = xp;
        y[0] = y[1]; y[1] = y[2]; y[2] = yp;
        --pos;
    }
    // Draw i is number i + 1 of the block, reached from the current position
    // by stepping forward or back, or forward from the start when that is
    // shorter.
    __device__ __forceinline__ void seek(int i)
    {
        const int t = i + 1;
        if (t < pos - t) {
#pragma unroll
            for (int l = 0; l < 3; ++l) { x[l] = x0[l]; y[l] = y0[l]; }
            pos = 0;
        }
        while (pos < t) forward();
        while (pos > t) back();
    }
    // FP64: the reference's uniform (mrg32k3a.h:84-86) and inverse normal
    // (gaussians.h:47-87)
    __device__ __forceinline__ double uniform(int i)
    {
        seek(i);
        // d / (m1 + 1), the division by its reciprocal and one residual step
        const double diff = double(x[0]) - double(y[0]);
        const double d = x[0] > y[0] ? diff : diff + 4294967087.0;
        const double q = d * (1.0 / 4294967088.0);
        return fma(fma(-q, 4294967088.0, d), 1.0 / 4294967088.0, q);
    }
    __device__ __forceinline__ double normal(int i)
    {
        const double z = inv_normal_p(uniform(i));
        return neg ? -z : z;
    }
    // FP32: the uniform d / (m1 + 1), d in [1, m1], as a word of 32 bits,
    // w = d + floor(208 d / 2^32) in [1, 2^32 - 2] (within one unit of
    // 2^32 u), for the FP32 inverse normal of Sobol words
    __device__ __forceinline__ float normal_f32(int i, const float* tabm)
    {
        seek(i);
        const uint32_t d = x[0] > y[0] ? x[0] - y[0] : x[0] - y[0] + kM1;
        const uint32_t w = d + uint32_t((uint64_t(d) * 208u) >> 32);
        const float z = inv_normal(w, tabm);
        return neg ? -z : z;
    }
};
}   // namespace mrg

// e^d - 1 over d, without its leading 1: the Taylor series of degree N - 1
// from d / 2 on, by Horner's rule; N = 8 for |d| <= 0.05 (truncation of e^d below
// 6e-18), N = 13 for |d| <= 0.3466 (4e-18).
template <int N>
__device__ __forceinline__ double exp_series(double d)
{
    constexpr double c[14] = {1.0, 1.0, 1.0 / 2.0, 1.0 / 6.0, 1.0 / 24.0, 1.0 / 120.0, 1.0 / 720.0, 1.0 / 5040.0,
                              1.0 / 40320.0, 1.0 / 362880.0, 1.0 / 3628800.0, 1.0 / 39916800.0, 1.0 / 479001600.0,
                              1.0 / 6227020800.0};
    double q = fma(d, c[N], c[N - 1]);
#pragma unroll
    for (int k = N - 2; k >= 3; --k) q = fma_s(q, d, c[k]);
    return fma(q, d, 0.5);
}
// exp in FP64 by Cody and Waite's reduction: x = n ln(2) + d,
// 2^n (1 + d (1 + d series)), the last step rounded once: within 0.85 ulp, 0.257
// on average, over 2^21 arguments of -30 to 14, as the library function (0.85,
// 0.258); 1 + (d + d^2 series) is within 0.96 (0.267).  x beyond +-800 saturates
// to 0 or infinity, and a NaN stays one (v_max_f64 would drop it: under -800 the
// high word is replaced instead, by that of -800; above 800 only n is bounded, d
// overflows).  22 instructions, no table (a load would wait for the checkpoint
// stores issued before it), against the library's 35.
__device__ __forceinline__ double exp_f64(double x)
{
    const uint64_t bits = __builtin_bit_cast(uint64_t, x);
    const uint32_t hi = x < -800.0 ? 0xc0890000u : uint32_t(bits >> 32);
    x = __builtin_bit_cast(double, uint64_t(hi) << 32 | uint32_t(bits));
    const double n = __builtin_rint(min_f64(x, 800.0) * 1.4426950408889634);
    // ln(2) in two parts, the first of 33 bits: n times it is exact
    double d = fma(n, -6.93147180369123816490e-01, x);
    d = fma(n, -1.90821492927058770002e-10, d);
    const double s = fma(d, exp_series<13>(d), 1.0);
    return __builtin_amdgcn_ldexp(fma(d, s, 1.0), int(n));
}

// e^x as a sum hi + lo good to some 2^-60, for constants formed once per block:
// x = n ln(2) / 8 + d, 2^(n / 8) from a table as a sum.
static __constant__ double kExpEighths[16] = {   // 2^(j / 8), hi and lo
    1.00000000000000000e+00, 0.00000000000000000e+00,
    1.09050773266525769e+00, -3.04678207981247115e-17,
    1.18920711500272103e+00, 3.98201523146564611e-17,
    1.29683955465100964e+00, 2.53825027948883150e-17,
    1.41421356237309515e+00, -9.66729331345291345e-17,
    1.54221082540794074e+00, 7.94983480969762086e-17,
    1.68179283050742900e+00, 8.19901002058149652e-17,
    1.83400808640934243e+00, 3.28310722424562720e-17,
};
struct ExpScale {
    double hi, lo;
};
__device__ __forceinline__ ExpScale exp_pair(double x)
{
    const double n = __builtin_rint(x * 11.541560327111707);   // 8 / ln(2)
    // ln(2) / 8 in two parts, the first of 29 bits: n times it is exact
    double d = fma(n, -8.66433973424136638641e-02, x);
    d = fma(n, -2.27579499813018278006e-10, d);
    const int k = int(n);
    const double2 t = reinterpret_cast<const double2*>(kExpEighths)[k & 7];
    const double r = fma(d * d, exp_series<8>(d), d);
    const double s = fma(t.x, r, t.y), hi = t.x + s;
    return {__builtin_amdgcn_ldexp(hi, k >> 3), __builtin_amdgcn_ldexp((t.x - hi) + s, k >> 3)};
}

// Spot from the path state: FP64 state is log(S) (reference), FP32 state is
// log(S / S0), which keeps more significant bits in single precision.
__device__ __forceinline__ double state_spot(double x, double) { return exp_f64(x); }
__device__ __forceinline__ float state_spot(float x, double s0) { return float(s0) * __expf(x); }

__device__ __forceinline__ double rexp(double x) { return exp_f64(x); }
__device__ __forceinline__ float rexp(float x) { return __expf(x); }

// Local vol at state x on one timeline row (interp.h:26-63): upper_bound on
// the knots, linear in between, flat outside.  Returns the two grid nodes
// touched and their weights for the adjoint.
template <typename R>
struct Bracket {
    R vol;
    R slope;      // d vol / d x
    int j;        // padded column of the left node (the row's columns j, j + 1)
    R wa, wb;     // adjoint weights of nodes j and j + 1
};

// Interval c = knot_count(x), the number of knots <= x, found by the
// caller (the reverse sweep reloads it from the forward's).  The interval
// tables make the flat extrapolation an ordinary interval: for c = 0 and
// c = m the padded row repeats the end value and the inverse width is 0, so
// t = 0, vol = the end value, slope = 0; inside, t = (x - k[c-1]) / (k[c] -
// k[c-1]) and vol = y[c-1] + (y[c] - y[c-1]) t.  No clamps, no selects.
// kxi: [m + 1] (interval start, inverse width) pairs, one aligned read;
// row: [m + 2].
template <typename R>
__device__ __forceinline__ Bracket<R> local_vol_at(const R* kxi, const R* row, R x, int c)
{
    const R y1 = row[c], y2 = row[c + 1];
    const R ih = kxi[2 * c + 1];
    const R t = (x - kxi[2 * c]) * ih;
    const R dy = y2 - y1;
    Bracket<R> b;
    b.j = c;
    b.vol = y1 + dy * t;
    b.slope = dy * ih;
    b.wa = R(1) - t;
    b.wb = t;
    return b;
}

__device__ __forceinline__ double recip_mul(double a, double b) { return fast_div(a, b); }
__device__ __forceinline__ float recip_mul(float a, float b) { return a * __builtin_amdgcn_rcpf(b); }

// Log-Euler step of the Dupire state (mcMdlDupire.h:271); one definition for
// the forward sweep and the recompute variant's re-simulation, so both give
// the same states.
template <typename R>
__device__ __forceinline__ R euler_step(R x, R vol, R g)
{
    return x + vol * (R(-0.5) * vol + g);
}

// ------------------------------------------------------------------ Sobol

// Sobol points of a block of 64 indices n = 64 q + r (sobol.h:55-151):
// gray(64q + r) = gray6(r) ^ (q & 1) << 5 ^ gray(q) << 6, so the word of lane r
// in dimension d is LO[d][r] ^ HI_q[d].  The path kernels and the points
// kernel share these functions.

// LO staged in LDS by a block, in one of four layouts: rows (the 64 lanes'
// low words of each dimension, [d][lane]), quads (the same words interleaved
// by groups of four dimensions, [d / 4][lane][d % 4], for kernels that read a
// lane's four consecutive dimensions in one 16-byte word; a lane reading one
// word at a time would stride 16 bytes and conflict on the LDS banks), LEAN
// (only direction numbers 0..5: the low word is formed in registers from the
// lane's masks), or split: gray6 is linear over the bits of the lane, so its
// word is the XOR of one of eight words for lane % 8 and one of eight for
// lane / 8, a quarter of the rows' size; interleaved by four dimensions,
// [d / 4][16][d % 4], read four at a time (lanes with the same octet read the
// same address, without conflicts).
enum SobolLoLayout { kLoRows = 0, kLoLean = 1, kLoQuads = 2, kLoSplit = 3 };

// All six direction numbers of a word are loaded, of four words at a time, and
// the ones that are not its own masked out: a branch around each load would
// wait for them one by one (2^15 paths x 156 steps, pricing: FP32 46 -> 39 us,
// FP64 89 -> 75).
template <int LO>
__device__ __forceinline__ void sobol_stage_lo(uint32_t* lo_tab, const uint32_t* dirs, int n, int tid, int nthr)
{
    if constexpr (LO == kLoLean) {
        for (int e = tid; e < n * 8; e += nthr) {
            const int d = e >> 3, k = e & 7;
            lo_tab[e] = k < 6 ? dirs[k * kSobolDims + d] : 0u;
        }
    } else {
        // word e: rows dimension e >> 6, lane e & 63; quads dimension
        // 4 (e >> 8) + (e & 3), lane (e >> 2) & 63; split dimension
        // 4 (e >> 6) + (e & 3), entry (e >> 2) & 15 (lane % 8, then 8 + lane / 8)
        const int total = sobol_dims4(n) * (LO == kLoSplit ? 16 : kWave);
        auto stage = [&](auto batch) {
            constexpr int kBatch = decltype(batch)::value;
            for (int e0 = tid; e0 < total; e0 += kBatch * nthr) {
                uint32_t v[kBatch][6], g[kBatch];
                int dim[kBatch];
#pragma unroll
                for (int b = 0; b < kBatch; ++b) {
                    const int e = e0 + b * nthr;
                    const int o = (e >> 2) & 15;
                    const int r = LO == kLoSplit ? (o < 8 ? o : (o - 8) << 3) : LO == kLoQuads ? (e >> 2) & 63 : e & 63;
                    dim[b] = LO == kLoSplit ? ((e >> 6) << 2) + (e & 3) : LO == kLoQuads ? ((e >> 8) << 2) + (e & 3) : e >> 6;
                    g[b] = uint32_t(r ^ (r >> 1));
                    const uint32_t d = uint32_t(min(dim[b], n - 1));
#pragma unroll
                    for (int k = 0; k < 6; ++k) v[b][k] = (dirs + k * kSobolDims)[d];
                }
#pragma unroll
                for (int b = 0; b < kBatch; ++b) {
                    uint32_t x = 0;
#pragma unroll
                    for (int k = 0; k < 6; ++k) x ^= v[b][k] & uint32_t(-int((g[b] >> k) & 1u));
                    if (dim[b] < n) lo_tab[e0 + b * nthr] = x;
                }
            }
        };
        // (a few steps, at most one word a thread: 18 loads less each; 5 steps
        // on 2^10 paths, FP32 risk 20.6 -> 19.9 us)
        if (total <= nthr) stage(std::integral_constant<int, 1>{});
        else stage(std::integral_constant<int, 4>{});
    }
}

// `bytes` of a 16-byte aligned table into LDS, both padded to whole words of
// four bytes.
__device__ __forceinline__ void stage_table(void* lds, const void* table, size_t bytes, int tid, int nthr)
{
    const int n16 = int(bytes >> 4), n4 = int(bytes >> 2);
    const uint4* g = static_cast<const uint4*>(table);
    uint4* l = static_cast<uint4*>(lds);
    for (int e0 = tid; e0 < n16; e0 += 4 * nthr) {
        uint4 v[4];
#pragma unroll
        for (int b = 0; b < 4; ++b) v[b] = g[min(e0 + b * nthr, n16 - 1)];
#pragma unroll
        for (int b = 0; b < 4; ++b)
            if (e0 + b * nthr < n16) l[e0 + b * nthr] = v[b];
    }
    for (int e = 4 * n16 + tid; e < n4; e += nthr)
        static_cast<uint32_t*>(lds)[e] = static_cast<const uint32_t*>(table)[e];
}

// LEAN: masks of the bits of gray6(lane), selecting direction numbers 0..5
struct SobolLaneMasks {
    uint32_t m[6];
};
__device__ __forceinline__ SobolLaneMasks sobol_lane_masks(int lane)
{
    SobolLaneMasks lm;
    const uint32_t g6 = uint32_t(lane ^ (lane >> 1));
#pragma unroll
    for (int k = 0; k < 6; ++k) lm.m[k] = ((g6 >> k) & 1u) ? 0xffffffffu : 0u;
    return lm;
}

// low word of dimension i for this lane
template <int LO>
__device__ __forceinline__ uint32_t sobol_low_word(const uint32_t* lo_tab, const SobolLaneMasks& lm, int lane, int i)
{
    if constexpr (LO == kLoLean) {
        const uint32_t* v = lo_tab + i * 8;
        return (lm.m[0] & v[0]) ^ (lm.m[1] & v[1]) ^ (lm.m[2] & v[2]) ^ (lm.m[3] & v[3]) ^ (lm.m[4] & v[4]) ^
               (lm.m[5] & v[5]);
    } else if constexpr (LO == kLoQuads) {
        return lo_tab[sobol_lo_el(i, lane)];
    } else if constexpr (LO == kLoSplit) {
        const uint32_t* v = lo_tab + ((i >> 2) << 6) + (i & 3);
        return v[(lane & 7) << 2] ^ v[(8 + (lane >> 3)) << 2];
    } else {
        return lo_tab[i * kWave + lane];
    }
}

// Quads and split layouts: this lane's words of dimensions i .. i + 3 (i a
// multiple of four, below the padded dimension count), one 16-byte read of LO
// (two of the split one) and one of the lane's high row (16-byte aligned rows)
template <int LO = kLoQuads>
__device__ __forceinline__ void sobol_words4(const uint32_t* lo_tab, const uint32_t* hl, int lane, int i, uint32_t* w)
{
    const uint4 hw = *reinterpret_cast<const uint4*>(hl + i);
    uint4 lw;
    if constexpr (LO == kLoSplit) {
        const uint4* v = reinterpret_cast<const uint4*>(lo_tab) + ((i >> 2) << 4);
        const uint4 a = v[lane & 7], b = v[8 + (lane >> 3)];
        lw = make_uint4(a.x ^ b.x, a.y ^ b.y, a.z ^ b.z, a.w ^ b.w);
    } else {
        lw = *reinterpret_cast<const uint4*>(lo_tab + sobol_lo_el(i, lane));
    }
    w[0] = lw.x ^ hw.x;
    w[1] = lw.y ^ hw.y;
    w[2] = lw.z ^ hw.z;
    w[3] = lw.w ^ hw.w;
}

// HI_qb of the n dimensions into a wave's LDS row, formed by the wave's lanes.
// AHEAD: sixteen direction numbers loaded together and masked, for the Dupire
// adjoint kernels, whose few waves wait for them (2^20 paths x 156 steps, risk:
// FP32 0.354 -> 0.346 ms, FP64 0.654 -> 0.650); the others, with up to twice
// the waves, take only the ones they need (FP64 pricing 0.239 against 0.251 ms).
template <bool AHEAD>
__device__ __forceinline__ void sobol_fill_hi(uint32_t* row, const uint32_t* dirs, int n, int64_t qb, int lane)
{
    const uint32_t gq = uint32_t(qb ^ (qb >> 1));
    if constexpr (AHEAD) {
        // the direction numbers of the row, by the bits of g
        uint32_t g = gq << 6 | uint32_t(qb & 1) << 5;
        for (int d = lane; d < n; d += kWave) {
            // (opaque: the bits' masks and the addresses are formed here, not
            // kept in registers over the whole kernel)
            uint32_t at = uint32_t(d);
            asm volatile("" : "+s"(g), "+v"(at));
            uint32_t x = 0;
            auto rows = [&](auto first, auto count) {
                constexpr int B = decltype(first)::value, N = decltype(count)::value;
                uint32_t v[N];
#pragma unroll
                for (int k = 0; k < N; ++k) v[k] = (dirs + (B + k) * kSobolDims)[at];
#pragma unroll
                for (int k = 0; k < N; ++k) x ^= v[k] & uint32_t(-int((g >> (B + k)) & 1u));
            };
            rows(std::integral_constant<int, 5>{}, std::integral_constant<int, 16>{});
            if (g >> 21) rows(std::integral_constant<int, 21>{}, std::integral_constant<int, 11>{});
            row[d] = x;
        }
    } else {
        for (int d = lane; d < n; d += kWave) {
            uint32_t x = (qb & 1) ? dirs[5 * kSobolDims + d] : 0u;
            uint32_t b = gq;
            while (b) {
                const int j = __builtin_ctz(b);
                x ^= dirs[(j + 6) * kSobolDims + d];
                b &= b - 1u;
            }
            row[d] = x;
        }
    }
}

// One lane's share of a wave's block of 64 Sobol indices: its high-word row,
// Sobol index, whether it holds a path of [nlo, nhi] and which.
struct SobolLane {
    const uint32_t* hl;
    int64_t sidx;
    bool active;
    int64_t pidx;
};

// Fills the wave's high rows for block q (and, for the first block when the
// last block is merged into its idle low lanes, the tail row of block q1) and
// selects this lane's.  Sobol index 0 (lane 0 of block 0, never a path) has
// every word 0, outside the FP32 inverse normal's domain; without a merge the
// tail row is free, so that lane reads words of 2^31 from it instead (its low
// words are 0) and its draws stay inside the table.  fill: the rows are
// formed (false when the words are not used).
template <bool AHEAD = false>
__device__ __forceinline__ SobolLane sobol_block(uint32_t* hi, uint32_t* hi_tail, const uint32_t* dirs, int n,
                                                 int64_t q, int64_t q0, int64_t q1, int64_t nlo, int64_t nhi,
                                                 bool merge, int lane, bool fill)
{
    const bool tail_wave = merge && q == q0;
    if (fill) {
        sobol_fill_hi<AHEAD>(hi, dirs, n, q, lane);
        if (tail_wave) sobol_fill_hi<AHEAD>(hi_tail, dirs, n, q1, lane);
        if (!merge && q == 0)
            for (int d = lane; d < n; d += kWave) hi_tail[d] = 0x80000000u;
        wave_sync_lds();
    }
    // lanes 0..(nhi mod 64) of the first block take the last block's paths
    const bool tail = tail_wave && lane <= int(nhi & (kWave - 1));
    SobolLane sl;
    sl.sidx = (tail ? q1 : q) * kWave + lane;
    sl.hl = (tail || sl.sidx == 0) ? hi_tail : hi;
    sl.active = sl.sidx >= nlo && sl.sidx <= nhi;
    sl.pidx = sl.sidx - nlo;
    return sl;
}

// ------------------------------------------------------------------ products

// Per-lane product state carried along the path.
template <typename R>
struct ProductState {
    R alive;        // barrier: product of smoothing factors (before a breach)
    R pnz;          // barrier: after an exactly-zero smoothing factor, the product of the non-zero ones
    int nzero;      // barrier: number of exactly-zero factors
    bool dead;      // barrier: breached (alive forced to 0, no derivative)
    R euro;         // barrier: vanilla payoff at maturity
    R fin_f;        // barrier: final forward
    R fin_num;      // barrier: final numeraire
    R aggp;         // running aggregate of payoffs emitted at samples
};

// ------------------------------------------------------------------ kernel

// The kernel of one call, run by block bid of the call's nblk blocks (the
// whole grid, or the call's share of a packed launch).
template <typename R, int MODEL, int PRD, int ADJ, bool LEAN, bool MRG, bool ITEM>
__device__ __forceinline__ void path_body(const LaunchParams& P, const int bid, const int nblk)
{
    extern __shared__ __align__(16) unsigned char smem[];
    constexpr bool DUP = MODEL == MODEL_DUPIRE;
    constexpr bool AD = ADJ != ADJ_NONE;
    constexpr bool RECOMP = ADJ == ADJ_RECOMPUTE;
    constexpr int kSeg = sizeof(R) == 4 ? kSegF32 : kSegF64;   // recompute segment
    constexpr bool EUS = PRD == PRD_EUROPEANS;
    const int waves = blockDim.x >> 6;
    const int n = P.n_steps, m = P.n_spots, ns = P.n_samples, npay = P.n_pay;
    const int mp = lv_cols(m);   // padded local-vol row
    const int stride = out_stride(npay);
    constexpr bool BOOK = PRD == PRD_BOOK;
    constexpr bool SPLIT = split_layout(int(sizeof(R)), DUP, AD, LEAN);
    constexpr bool BSR = bs_row_layout(DUP, PRD, LEAN);
    const SmemLayout L = smem_layout(n, m, ns, npay, waves, int(sizeof(R)), DUP, EUS, AD, LEAN, P.n_buckets,
                                     P.ivbar_copies, SPLIT, BSR);

    uint32_t* lo_tab = reinterpret_cast<uint32_t*>(smem + L.lo);
    uint32_t* hi_all = reinterpret_cast<uint32_t*>(smem + L.hi);
    int* step_sample = reinterpret_cast<int*>(smem + L.step_sample);
    R* kxi = reinterpret_cast<R*>(smem + L.knots);   // interval (start, inverse width) pairs
    BucketOne<R>* bucket = reinterpret_cast<BucketOne<R>*>(smem + L.bucket);
    R* iv_lds = reinterpret_cast<R*>(smem + L.iv);
    R* drift = reinterpret_cast<R*>(smem + L.drift);
    R* stdv = reinterpret_cast<R*>(smem + L.stdv);
    constexpr int kBsReals = bs_row_reals(AD);
    R* bsr = reinterpret_cast<R*>(smem + L.bs);      // BSR: [n][kBsReals]
    double* s_ff = reinterpret_cast<double*>(smem + L.samples);
    double* s_disc = s_ff + ns;
    double* s_num = s_disc + ns;
    int* pay_first = reinterpret_cast<int*>(smem + L.pay_first);
    double* pay_strike = reinterpret_cast<double*>(smem + L.pay_strike);
    double* acc = reinterpret_cast<double*>(smem + L.acc);
    constexpr int TR = tail_row(LEAN);
    double* tails = reinterpret_cast<double*>(smem + L.tails);   // FP64: [waves][TR]
    double* ivbar = reinterpret_cast<double*>(smem + L.ivbar);
    R* invn = reinterpret_cast<R*>(smem + L.invn);   // FP32 inverse-normal table

    const int tid = threadIdx.x, nthr = blockDim.x;
    // The inverse-normal table (FP32) and the knot search table are read from
    // global memory through the L1 cache, not LDS, by the LEAN kernels.  The
    // FP32 recompute kernels and the FP32 Dupire kernels but the book's, bound
    // by the LDS pipe, read the inverse-normal table through L1, the widest of
    // a step's LDS reads and the one with the most bank conflicts.  (Pricing
    // 2^19 paths x 156 steps 0.131 -> 0.116 ms, C3 risk 0.587 -> 0.576 ms; with
    // the knot search table as well the vector memory path saturates instead.)
    constexpr bool GINV = LEAN || (sizeof(R) == 4 && (RECOMP || (DUP && !BOOK)));

    // Sobol LO layout: the FP32 Dupire kernels other than the book and the FP32
    // Black-Scholes barrier read four dimensions at once (quads), FP64 ones too (split); the others one at a
    // time (rows)
    constexpr bool QUADS = sizeof(R) == 4 && ((DUP && !BOOK && !LEAN) || BSR) && !MRG;
    constexpr int LOL = LEAN ? kLoLean : SPLIT ? kLoSplit : (QUADS ? kLoQuads : kLoRows);
    // ---- stage the block's tables in LDS
    if constexpr (!MRG) sobol_stage_lo<LOL>(lo_tab, P.dirs, n, tid, nthr);
    double* mtab = reinterpret_cast<double*>(smem + L.mtab);   // SPLIT: tail table rows from kMoroLdsRow on
    if constexpr (SPLIT)
        stage_table(mtab, kMoroTailF64 + kMoroLdsRow * kMoroTailCoefs, kMoroLdsBytes, tid, nthr);
    for (int e = tid; e <= n; e += nthr) step_sample[e] = P.step_sample[e];
    if constexpr (sizeof(R) == 4 && !GINV)
        for (int e = tid; e < kInvNormalRows * 4; e += nthr) invn[e] = kInvNormalF32[e];
    if constexpr (DUP) {
        const R* gk = static_cast<const R*>(P.knots);
        const R* gi = static_cast<const R*>(P.inv_dx);
        const R* gv = static_cast<const R*>(P.iv);
        for (int e = tid; e <= m; e += nthr) { kxi[2 * e] = gk[e]; kxi[2 * e + 1] = gi[e]; }
        if constexpr (!LEAN)
            for (int e = tid; e < P.n_buckets; e += nthr) {
                const BucketEntry<R>& b = static_cast<const BucketEntry<R>*>(P.bucket)[e];
                bucket[e].k0 = b.k0;
                bucket[e].lo = b.lo;
            }
        if constexpr (!LEAN)
            stage_table(iv_lds, gv, size_t(n) * size_t(mp) * sizeof(R), tid, nthr);
    } else {
        const R* gd = static_cast<const R*>(P.drift);
        const R* gs = static_cast<const R*>(P.stdv);
        if constexpr (BSR) {
            const double* dt = P.bs_aux + 3 * ns;
            for (int e = tid; e < n; e += nthr) {
                const int s = P.step_sample[e + 1];
                bsr[e * kBsReals] = gd[e];
                bsr[e * kBsReals + 1] = gs[e];
                bsr[e * kBsReals + 2] = s >= 0 ? R(P.ff[s]) : R(NAN);
                if constexpr (AD) {
                    const R dti = R(dt[e]), vol = R(P.bs_vol);
                    bsr[e * kBsReals + 4] = P.spot_measure ? vol * dti : -vol * dti;
                    bsr[e * kBsReals + 5] = R(sqrt(dt[e]));
                    bsr[e * kBsReals + 6] = dti;
                }
            }
        } else {
            for (int e = tid; e < n; e += nthr) { drift[e] = gd[e]; stdv[e] = gs[e]; }
        }
        for (int e = tid; e < ns; e += nthr) { s_ff[e] = P.ff[e]; s_disc[e] = P.disc[e]; s_num[e] = P.num[e]; }
    }
    if constexpr (EUS) {
        for (int e = tid; e <= ns; e += nthr) pay_first[e] = P.pay_first[e];
        for (int e = tid; e < npay; e += nthr) pay_strike[e] = P.pay_strike[e];
    }
    for (int e = tid; e < waves * stride; e += nthr) acc[e] = 0.0;
    if constexpr (AD && DUP)
        for (int e = tid; e < P.ivbar_copies * ivbar_copy_stride(n, m); e += nthr) ivbar[e] = 0.0;
    __syncthreads();

    // the wave index is uniform: block-level offsets derived from it stay in
    // scalar registers
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
    // local-vol table: LDS (FULL) or global memory (LEAN)
    const R* iv;
    if constexpr (LEAN) iv = static_cast<const R*>(P.iv); else iv = iv_lds;
    const SobolLaneMasks lmask = sobol_lane_masks(lane);
    auto low_word = [&](int i) -> uint32_t { return sobol_low_word<LOL>(lo_tab, lmask, lane, i); };
    uint32_t* hi = hi_all + wave * sobol_hi_stride(n);
    double* accw = acc + wave * stride;
    const int64_t nlo = P.first_path + 1, nhi = P.first_path + P.n_path;   // Sobol indices
    const int64_t q0 = nlo >> 6, q1 = nhi >> 6;
    // the last block's paths ride in the first block's idle low lanes when
    // they fit there (e.g. 2^k paths from path 0: Sobol indices 1..2^k), so no
    // wave makes an extra pass for them; those lanes read their high words
    // from the block's tail row
    const bool merge = P.merge_tail != 0;
    const int64_t qe = merge ? q1 - 1 : q1;
    uint32_t* hi_tail = reinterpret_cast<uint32_t*>(smem + L.hi_tail);
    const int slot = bid * waves + wave;
    // checkpoint slot of the wave: [n][64] states (Dupire) or normals
    // (Black-Scholes); recompute variant: [ceil(n / kSeg)][64] Dupire states
    const int ck_rows = ckpt_rows(n, DUP, RECOMP, int(sizeof(R)));
    // bracket bytes after the states: the knot count of x_i at each step
    constexpr bool CKB = DUP && ADJ == ADJ_CHECKPOINT;
    // (the Dupire checkpoint slot starts with kCkptGuardRows guard rows);
    // a wave's slot, or with ck_mode 1 and 2 the slot of each block of 64
    // Sobol indices (set per block below)
    // (only the ITEM checkpoint kernels read ck_mode)
    const int ck_mode = ITEM && ADJ == ADJ_CHECKPOINT ? P.ck_mode : 0;
    // PK: the swept paths of up to ck_slots blocks share a reverse sweep (see
    // there); ck is the slot of the block in work.  FP64 (2^20 paths x 156
    // steps, one path in ten swept: 0.80 -> 0.67 ms).  FP32 sweeps each block by
    // itself: its sweeps take less than the checkpoints of four slots, which
    // leave the last-level cache, cost (0.38 against 0.41 ms).
    constexpr bool PK = CKB && !ITEM && sizeof(R) == 8 && (PRD == PRD_BARRIER || PRD == PRD_EUROPEAN);
    const int ck_slots = PK ? P.ck_slots : 1;
    R* const ck0 = AD ? static_cast<R*>(P.ckpt) +
                            (size_t(slot) * ck_slots * ck_rows + (CKB ? kCkptGuardRows : 0)) * kWave : nullptr;
    R* ck = ck0;
    // (the FULL layout is only chosen for grids of at most kMaxStoredKnots knots)
    const bool ck_lo = CKB && (!LEAN || m <= kMaxStoredKnots);
    // States and bracket bytes interleaved by groups of four steps (a lane's
    // four in one 16-byte, in FP64 32-byte, word and one 4-byte word), except
    // those of the FP64 book, whose steps run one by one: gathering four costs
    // it more than the wider access saves (55 payoffs, 250,007 paths 0.84
    // against 0.79 ms; an Asian alone, 2^19 paths of 52 steps 0.33 against 0.28).
    // FP32 pads the steps to whole groups; FP64 keeps the steps from n4 on,
    // up to three, in rows.
    constexpr bool IL = CKB && !(BOOK && sizeof(R) == 8);
    const int nck = ckpt_steps(n, int(sizeof(R)));
    const int n4 = n & ~3;
    uint8_t* const ckl0 = CKB ? reinterpret_cast<uint8_t*>(ck + size_t(nck) * kWave) : nullptr;
    uint8_t* ckl = ckl0;
    // element of step i of this lane in the states (and bracket bytes)
    auto ck_el = [&](int i) -> int {
        return IL && (sizeof(R) == 4 || i < n4) ? ((i >> 2) << 8) + (lane << 2) + (i & 3) : i * kWave + lane;
    };
    constexpr int kStateRows = BOOK ? 8 + 2 * kMaxBookBarriers + 2 * kMaxBookGroups : 12;
    static_assert(kStateRows == (BOOK ? 8 + 2 * kMaxBookBarriers + 2 * kMaxBookGroups : 8 + 2 + 2),
                  "state rows as state_rows() counts them");
    KnotSearch<R> ks;
    ks.knots = kxi + 2;     // the knots themselves: interval starts from interval 1
    ks.stride = 2;
    ks.table = static_cast<const BucketEntry<R>*>(P.bucket);
    ks.m = m;
    ks.fix = P.bucket_fix;
    ks.invh = R(P.bucket_invh);
    ks.c0 = R(P.bucket_c0);
    ks.top = R(P.n_buckets - 1);
    ks.itop = P.n_buckets - 1;
    // number of knots <= x.  FP32: the entry's address straight from the
    // bucket's bits
    const uint32_t bucket_at = bucket_base(L.bucket);
    auto knot_count = [&](R x) -> int {
        if constexpr (LEAN) {
            return count_le<true>(ks, x);
        } else if constexpr (sizeof(R) == 4) {
            const uint32_t off = bucket_offset(x, ks.invh, ks.c0, ks.top, bucket_at);
            return count_le_one(*reinterpret_cast<const BucketOne<R>*>(smem + off), x);
        } else {
            return count_le_one(bucket[bucket_index(x, ks.invh, ks.c0, ks.top, ks.itop)], x);
        }
    };
    const double s0 = P.spot;
    const int last = ns - 1;

    // The spot of a barrier sample before the last.  FP64: where the smoothing
    // zone is narrow in log-spot (half-width at most kNarrowZone), it is
    // e^z_c e^(x - z_c) about the zone's centre z_c, with no reduction: 12
    // instructions.  States under the zone are taken at its edge, where
    // nothing changes; above it the polynomial increases, so a spot over the
    // zone stays over it.  (A zone that reaches down to 0 has no lower edge in
    // log-spot and is not narrow.)
    constexpr bool NZONE = DUP && PRD == PRD_BARRIER && sizeof(R) == 8;
    R z_c = R(0), z_lo = R(0);
    ExpScale z_e{0.0, 0.0};
    bool narrow = false;
    if constexpr (NZONE) {
        const R xu = log(R(P.bar_smooth)), xl = R(P.bar_xlo);
        narrow = __builtin_amdgcn_readfirstlane(int(R(0.5) * (xu - xl) <= R(kNarrowZone))) != 0;
        if (narrow) {
            z_c = R(0.5) * (xu + xl);
            z_e = exp_pair(z_c);
            z_lo = xl - z_c;
        }
    }

    // this lane's local-vol adjoint grid: odd lanes use the second copy, which
    // halves the lanes contending for one address in an atomic
    double* ivbl = ivbar + ((P.ivbar_copies > 1 && (lane & 1)) ? ivbar_copy_stride(n, m) : 0);
    // per-lane parameter adjoints, summed over the lane's paths
    double padj[kMaxParamAdj] = {0.0, 0.0, 0.0, 0.0};

    // Book tables and aggregation weights: wave-uniform values, read from
    // global memory through the scalar cache (constant address space) into
    // scalar registers, not staged in LDS
    const unsigned char* bkb = static_cast<const unsigned char*>(P.book);
    CPtr<double> bk_van_strike = cptr<double>(bkb + P.bk.van_strike);
    CPtr<int> bk_van_col = cptr<int>(bkb + P.bk.van_col);
    // per sample: barriers observing (bits 0-15) and maturing (16-31),
    // schedules fixing (bits 0-3) and ending (4-7), and the sample's vanillas
    // [van_lo, van_hi)
    struct alignas(16) SampleRow {
        uint32_t bars, grps;
        int van_lo, van_hi;
    };
    // (grps also: kBookAllBars, every barrier observes and none matures;
    // kBookPlain, nothing else happens either).  Dupire: one row per timeline
    // point (an empty row where it is no sample), so that a step's row is read
    // by its own index, ahead of the step; Black-Scholes: one per sample.
    CPtr<SampleRow> bk_rows_c = cptr<SampleRow>(DUP ? static_cast<const void*>(P.pay_first) : bkb + P.bk.masks);
    auto bk_rows = [&](int s) -> SampleRow {
        SampleRow r;
        r.bars = bk_rows_c[s].bars;
        r.grps = bk_rows_c[s].grps;
        r.van_lo = bk_rows_c[s].van_lo;
        r.van_hi = bk_rows_c[s].van_hi;
        return r;
    };
    // barriers by fours, in the kernel's precision, past the last one at
    // +infinity: the lower ends of their zones, B + w, 1 / 2w, and the lowest
    // of the lower ends
    struct alignas(16) BarFour {
        R lo[4], up[4], i2s[4], lo_min[4];
    };
    CPtr<BarFour> bk_four_c =
        cptr<BarFour>(bkb + (sizeof(R) == 4 ? P.bk.bar_par_f + P.bk.n_bar * 16 : P.bk.bar_par + P.bk.n_bar * 32));
    CPtr<int> bk_grp_first = cptr<int>(bkb + P.bk.grp_first);
    CPtr<double> bk_as_strike = cptr<double>(bkb + P.bk.as_strike);
    CPtr<int> bk_as_col = cptr<int>(bkb + P.bk.as_col);
    CPtr<int> bk_as_put = cptr<int>(bkb + P.bk.as_put);
    CPtr<int> bk_bar_col = cptr<int>(bkb + P.bk.bar_col);
    CPtr<int> bk_bar_put = cptr<int>(bkb + P.bk.bar_put);
    // fixing weights in the kernel's precision
    CPtr<R> bk_ginv = cptr<R>(bkb + (sizeof(R) == 4 ? P.bk.grp_inv_f : P.bk.grp_inv));
    // barrier b's (strike, B + w, B - w, 1 / 2w) in the kernel's precision
    struct alignas(16) BarPar {
        R k, up, lo, i2s;
    };
    CPtr<BarPar> bk_par_c = cptr<BarPar>(bkb + (sizeof(R) == 4 ? P.bk.bar_par_f : P.bk.bar_par));
    auto bar_par = [&](int b) -> BarPar {
        BarPar r;
        r.k = bk_par_c[b].k;
        r.up = bk_par_c[b].up;
        r.lo = bk_par_c[b].lo;
        r.i2s = bk_par_c[b].i2s;
        return r;
    };
    CPtr<double> wts = cptr<double>(P.weights);
    // Barrier smoothing factors (B + w - F) / 2w: FP64 tracks exactly-zero
    // factors (F = B + w) as the tape does.  FP32 keeps B + w - F at least
    // tiny_d instead, so a factor is never 0 and the product of the others,
    // the tape's derivative at a zero factor, stays the product over the
    // factor; the price moves by at most 1e-30 of the payoff there.
    constexpr bool ZT = sizeof(R) == 8;
    const R tiny_d = ZT ? R(0) : max(R(P.two_smooth) * R(1e-30), R(1e-37));
    constexpr int NBAR = BOOK ? kMaxBookBarriers : 1, NGRP = BOOK ? kMaxBookGroups : 1;
    // Book barrier state in one real per barrier:
    //   sign bit set  breached (survival 0, no derivative)
    //   v in [0, 1]   the product of the smoothing factors (the survival factor)
    // A smoothing factor is (B + w - F) / 2w clamped to [0, 1], so an update is
    // a product for every lane, in the zone, under it or breached.  An
    // exactly-zero factor (FP64) is left out of the product and marked in the
    // path's bit mask zmask, beside the state, whose range stays free for any
    // weight: the survival factor is 0, and v is the product of the others,
    // which the derivative takes at that factor; a second one makes v 0 too, as
    // two have no derivative.  FP32 keeps every factor at least 1e-30 (as the
    // single barrier keeps B + w - F above a floor) and marks none.
    // v after an observation at distance t = B + w - F, 1 / 2w = i2s
    auto bar_update = [&](R v, R t, R i2s) -> R {
        if constexpr (sizeof(R) == 4) {
            const R f = __builtin_amdgcn_fmed3f(t * i2s, 1e-30f, 1.0f);
            return __uint_as_float(__float_as_uint(v * f) | (__float_as_uint(t) & 0x80000000u));
        } else {
            double f;
            asm("v_mul_f64 %0, %1, %2 clamp" : "=v"(f) : "v"(t), "s"(i2s));
            const uint64_t sign = __builtin_bit_cast(uint64_t, t) & (uint64_t(1) << 63);
            return __builtin_bit_cast(double, __builtin_bit_cast(uint64_t, v * f) | sign);
        }
    };
    const R bk_xlo = BOOK && DUP ? R(P.bar_xlo) : R(0);   // every zone is above this state
    // Black-Scholes: and above this forward, one test a sample where the fours
    // load and test four (5 steps, a book of 2 barriers, 2^22 FP32 paths: risk
    // 208 -> 198 us)
    const R bk_lo = BOOK && !DUP ? R(P.bar_xlo) : R(0);

    // PK: swept paths waiting for a full wave, in lanes 0 .. pk_n - 1 of pk_src
    // (lane of the block, slot << 6, count of zero factors << 28, breached
    // << 30), from pk_used slots up to the one before pk_slot
    uint32_t pk_src = 0;
    int pk_n = 0, pk_used = 0, pk_slot = 0;

    for (int64_t q = q0 + int64_t(bid) * waves + wave; q <= qe; q += int64_t(nblk) * waves) {
        // ---- high Sobol words of this block of 64 indices (and of the
        // merged last block); this lane's row, index and path
        const SobolLane sl = sobol_block<AD && DUP && !BOOK>(hi, hi_tail, P.dirs, n, q, q0, q1, nlo, nhi, merge, lane, !MRG);
        const uint32_t* hl = sl.hl;
        const bool active = sl.active;
        const int64_t pidx = sl.pidx;
        // itemized risk: the checkpoint slot and the end state of this block of 64 paths
        R* stq = nullptr;
        if (ck_mode != 0) {
            const size_t sb = size_t(q - q0);
            ck = static_cast<R*>(P.ckpt) + (sb * ck_rows + (CKB ? kCkptGuardRows : 0)) * kWave;
            if constexpr (CKB) ckl = reinterpret_cast<uint8_t*>(ck + size_t(nck) * kWave);
            stq = static_cast<R*>(P.state) + sb * kStateRows * kWave + lane;
        }
        // normal of step i: from the Sobol point, or from this lane's
        // mrg32k3a generator (idle lanes run the call's first path)
        mrg::Lane gen;
        if constexpr (MRG) gen.start(P.mrg_jump, P.mrg_seed1, P.mrg_seed2, P.first_path + (active ? pidx : 0));
        // the inverse-normal table (LDS, or for LEAN the constant array
        // itself) less kInvNormalRowBias rows (FP32)
        const R* invn_tab;
        if constexpr (GINV && sizeof(R) == 4) invn_tab = reinterpret_cast<const R*>(kInvNormalF32);
        else invn_tab = invn;
        if constexpr (sizeof(R) == 4) invn_tab -= 4 * kInvNormalRowBias;
        auto draw = [&](int i) -> R {
            if constexpr (MRG) {
                if constexpr (sizeof(R) == 4) return gen.normal_f32(i, invn_tab);
                else return gen.normal(i);
            }
            else return inv_normal(hl[i] ^ low_word(i), invn_tab);
        };

        // Sobol words of steps i .. i + 3 (i a multiple of four)
        auto words4 = [&](int i, uint32_t* w) {
            if constexpr (SPLIT) {
                sobol_words4<kLoSplit>(lo_tab, hl, lane, i, w);
            } else {
#pragma unroll
                for (int k = 0; k < 4; ++k) w[k] = hl[i + k] ^ low_word(i + k);
            }
        };

        ProductState<R> ps;
        ps.alive = R(1); ps.pnz = R(1); ps.nzero = 0; ps.dead = false;
        bool nzw = false;   // barrier: some lane of the wave has an exactly-zero smoothing factor
        ps.euro = R(0); ps.fin_f = R(0); ps.fin_num = R(1); ps.aggp = R(0);
        // book: per barrier the state above and (after its maturity) weight x
        // vanilla, the adjoint of its survival factor; per fixing schedule
        // the running sum, replaced at its last fixing by the adjoint of each
        // fixing, and the weighted intrinsic value (numeraire adjoint)
        // (LAZY keeps one value per barrier, its registers bound the waves on a
        // compute unit: a sweep that meets the maturity before the samples
        // before it replaces the state there by its product with weight x
        // vanilla; up to then a path without a vanilla counts as breached,
        // which has no adjoint either)
        constexpr bool LAZY = ZT && CKB;
        constexpr int NBB = LAZY ? 1 : NBAR;
        R bst[NBAR], babar[NBB], gsum[NGRP], gq[NGRP];
        uint32_t zmask = 0;
        // the survival factor of barrier b
        auto bar_alive = [&](int b) -> R {
            return bst[b] > R(0) && !(ZT && ((zmask >> b) & 1u)) ? bst[b] : R(0);
        };
        // an exactly-zero factor of barrier b: the distance t = 0 that the
        // update takes it from, a first one as far below the zone (factor 1)
        auto mark_zero = [&](int b, R& t) {
            if (t != R(0)) return;
            if (!((zmask >> b) & 1u)) t = R(INFINITY);
            zmask |= 1u << b;
        };
#pragma unroll
        for (int b = 0; b < NBAR; ++b) bst[b] = R(1);
#pragma unroll
        for (int b = 0; b < NBB; ++b) babar[b] = R(0);
#pragma unroll
        for (int g = 0; g < NGRP; ++g) { gsum[g] = R(0); gq[g] = R(0); }

        // payoff `col` of this lane's path: wave sums, per-path output
        auto emit = [&](int col, R pay) {
            const double v = active ? double(pay) : 0.0;
            const double vs = wave_sum(v), vq = wave_sum(v * v);
            if (lane == kSumLane) { accw[col] += vs; accw[npay + col] += vq; }
            if (P.per_path && active) P.per_path[pidx * npay + col] = v;
            if constexpr (AD) ps.aggp = ps.aggp + R(wts[col]) * pay;
        };

        // observation of product sample s with spot S (and for Black-Scholes
        // the sample's forward factor / numeraire / discount)
        // (book: with the sample's row sm)
        auto observe = [&](int s, R S, SampleRow sm) {
            R F = S, numv = R(1), discv = R(1);
            if constexpr (!DUP) {
                F = S * R(s_ff[s]);
                numv = P.spot_measure ? R(s_num[s]) * S : R(s_num[s]);
                discv = R(s_disc[s]);
            }
            if constexpr (PRD == PRD_BARRIER) {
                // mcPrd.h:256-287, branch free: a breach kills the path, the
                // smoothing zone multiplies in (B + w - F) / 2w
                const bool live = !ps.dead;
                const bool brk = live && F > R(P.bar_smooth);
                const bool zone = live && !brk && F > R(P.minus_smooth);
                const R a_prev = ps.alive;
                ps.dead = ps.dead || brk;
                if constexpr (ZT) {
                    const R f = (R(P.bar_smooth) - F) * R(P.inv_two_smooth);
                    if (zone) ps.alive = a_prev * f;
                    // exactly-zero factors (F = B + w), rare: from the first one on,
                    // pnz holds the product of the non-zero factors
                    nzw = nzw | (__builtin_amdgcn_ballot_w64(f == R(0)) != 0);
                    if (nzw) {
                        const bool fz = zone && f == R(0);
                        if (fz) {
                            if (ps.nzero == 0) ps.pnz = a_prev;
                            ps.nzero++;
                        } else if (zone && ps.nzero > 0) {
                            ps.pnz = ps.pnz * f;
                        }
                    }
                } else {
                    const R f = max(R(P.bar_smooth) - F, tiny_d) * R(P.inv_two_smooth);
                    ps.alive = a_prev * (zone ? f : R(1));
                }
                // the vanilla of the last sample: after the path (the last
                // sample is the last timeline point)
            } else if constexpr (PRD == PRD_EUROPEAN) {
                // mcPrd.h:113-125
                const R k = R(P.strike);
                const R pay = (F - k > R(0) ? F - k : R(0)) * discv / numv;
                const double v = active ? double(pay) : 0.0;
                const double vs = wave_sum(v), vq = wave_sum(v * v);
                if (lane == kSumLane) { accw[0] += vs; accw[npay] += vq; }
                if (P.per_path && active) P.per_path[pidx * npay] = v;
                if constexpr (AD) ps.aggp = ps.aggp + R(wts[0]) * pay;
            } else if constexpr (PRD == PRD_BOOK) {
                // vanilla calls at this sample (European / Europeans parts)
                for (int k = sm.van_lo; k < sm.van_hi; ++k) {
                    const R kk = R(bk_van_strike[k]);
                    emit(bk_van_col[k], (F - kk > R(0) ? F - kk : R(0)) / numv);
                }
                // up-and-out barriers (mcPrd.h:256-287, one state per barrier,
                // in the book's order): by fours a product per barrier for all
                // lanes (bar_update), while some lane is above the lowest of
                // their zones; no state changes otherwise.  A wave vote per barrier instead, to
                // skip those with no live lane in the zone, visits half as many
                // but costs more scalar work and branches than it saves.
                const uint32_t bl = sm.bars >> 16;
                const bool all_bars = (sm.grps & kBookAllBars) != 0;
                if (all_bars && (DUP || __builtin_amdgcn_ballot_w64(F > bk_lo) != 0)) {
#pragma unroll
                    for (int b = 0; b + 3 < NBAR; b += 4) {
                        if (__builtin_amdgcn_ballot_w64(F > bk_four_c[b >> 2].lo_min[0]) == 0) continue;
                        R up[4], i2s[4];
#pragma unroll
                        for (int j = 0; j < 4; ++j) {
                            up[j] = bk_four_c[b >> 2].up[j];
                            i2s[j] = bk_four_c[b >> 2].i2s[j];
                        }
                        R t[4];
                        uint64_t zero = 0;
#pragma unroll
                        for (int j = 0; j < 4; ++j) {
                            t[j] = up[j] - F;
                            if constexpr (ZT) zero |= __builtin_amdgcn_ballot_w64(t[j] == R(0));
                        }
                        if (ZT && zero != 0) {
                            asm volatile("");   // (rare: a branch of its own)
#pragma unroll
                            for (int j = 0; j < 4; ++j) mark_zero(b + j, t[j]);
                        }
#pragma unroll
                        for (int j = 0; j < 4; ++j) bst[b + j] = bar_update(bst[b + j], t[j], i2s[j]);
                    }
                }
                if (!all_bars && sm.bars) {
#pragma unroll
                    for (int b = 0; b < NBAR; ++b) {
                        if (!(((sm.bars | bl) >> b) & 1u)) continue;
                        const BarPar bp = bar_par(b);
                        if (((sm.bars >> b) & 1u) && F > bp.lo) {
                            R t = bp.up - F;
                            if constexpr (ZT) mark_zero(b, t);
                            bst[b] = bar_update(bst[b], t, bp.i2s);
                        }
                        if ((bl >> b) & 1u) {
                            const R k = bp.k;
                            const R intrinsic = bk_bar_put[b] ? (k - F > R(0) ? k - F : R(0))
                                                                         : (F - k > R(0) ? F - k : R(0));
                            const R euro = intrinsic / numv;
                            const R alive = bar_alive(b);
                            const int col = bk_bar_col[b];
                            emit(col, alive * euro);
                            emit(col + 1, euro);
                            // weight x vanilla: the adjoint of the survival
                            // factor (the ITEM kernels keep the vanilla and
                            // weigh it before the reverse sweep)
                            if constexpr (AD) {
                                const R w = ITEM ? R(1) : R(wts[col]);
                                if constexpr (LAZY) bst[b] = euro != R(0) && w != R(0) ? bst[b] : R(-1);
                                else babar[b] = w * euro;
                            }
                        }
                    }
                }
                // arithmetic averages: running sums per fixing schedule
                const uint32_t gm = sm.grps & 0xfu, gl = (sm.grps >> 4) & 0xfu;
                if (gm) {
#pragma unroll
                    for (int g = 0; g < NGRP; ++g) {
                        if (!((gm >> g) & 1u)) continue;
                        gsum[g] = gsum[g] + F;
                        if ((gl >> g) & 1u) {
                            const R inv_n = bk_ginv[g];
                            const R avg = gsum[g] * inv_n;
                            R dsum = R(0), qsum = R(0);
                            for (int a = bk_grp_first[g]; a < bk_grp_first[g + 1]; ++a) {
                                const R k = R(bk_as_strike[a]);
                                const bool put = bk_as_put[a] != 0;
                                const R intrinsic = put ? (k - avg > R(0) ? k - avg : R(0))
                                                        : (avg - k > R(0) ? avg - k : R(0));
                                const int col = bk_as_col[a];
                                emit(col, intrinsic / numv);
                                if constexpr (AD && !ITEM) {
                                    const R w = R(wts[col]);
                                    const R d = put ? (k > avg ? R(-1) : R(0)) : (avg > k ? R(1) : R(0));
                                    dsum = dsum + w * d;
                                    qsum = qsum + w * intrinsic;
                                }
                            }
                            // the adjoint of each fixing and the weighted
                            // intrinsic values (the numeraire adjoint); the ITEM
                            // kernels keep the average and the numeraire and
                            // form both before the reverse sweep
                            if constexpr (AD) {
                                gsum[g] = ITEM ? avg : dsum * inv_n / numv;
                                gq[g] = ITEM ? numv : qsum;
                            }
                        }
                    }
                }
            } else {
                // mcPrd.h:374-399
                for (int k = pay_first[s]; k < pay_first[s + 1]; ++k) {
                    const R kk = R(pay_strike[k]);
                    const R pay = (F - kk > R(0) ? F - kk : R(0)) / numv;
                    const double v = active ? double(pay) : 0.0;
                    const double vs = wave_sum(v), vq = wave_sum(v * v);
                    if (lane == kSumLane) { accw[k] += vs; accw[npay + k] += vq; }
                    if (P.per_path && active) P.per_path[pidx * npay + k] = v;
                    if constexpr (AD) ps.aggp = ps.aggp + R(wts[k]) * pay;
                }
            }
        };

        // book: the row of sample s, at timeline point i
        auto row_of = [&](int s, int i) -> SampleRow {
            if constexpr (BOOK) return bk_rows(DUP ? i : s);
            else return SampleRow{};
        };
        // Dupire barrier: a sample other than the last one changes nothing on
        // a path that is under the smoothing zone or breached, so the spot is
        // not formed where all the wave's paths are (forward and reverse)
        constexpr bool UNDER = DUP && PRD == PRD_BARRIER;
        const R x_lo = UNDER ? R(P.bar_xlo) : R(0);
        auto zone_spot = [&](R x) -> R {
            if constexpr (NZONE) {
                if (!narrow) return exp_f64(x);
                const double d = max_f64(x - z_c, z_lo);
                const double r = fma(d * d, exp_series<8>(d), d);
                return z_e.hi + fma(z_e.hi, r, z_e.lo);
            } else {
                return state_spot(x, s0);
            }
        };
        // Dupire barrier: whether timeline points base .. base + 63 are
        // samples, one wave-uniform 64-bit mask from one ballot (bit b: point
        // base + b); the sweeps test a bit per step instead of reading the
        // sample map
        auto sample_bits = [&](int base) -> uint64_t {
            const int p = base + lane;
            return __builtin_amdgcn_ballot_w64(p <= n && step_sample[min(p, n)] >= 0);
        };
        R x;
        if (ck_mode == 2) {
            // reverse only: the end state the forward-only launch kept
            x = stq[0];
            ps.alive = stq[1 * kWave];
            ps.pnz = stq[2 * kWave];
            ps.nzero = int(stq[3 * kWave]);
            if constexpr (BOOK && ZT) zmask = uint32_t(ps.nzero);
            ps.dead = stq[4 * kWave] != R(0);
            ps.euro = stq[5 * kWave];
            ps.fin_f = stq[6 * kWave];
            ps.fin_num = stq[7 * kWave];
#pragma unroll
            for (int b = 0; b < NBAR; ++b) {
                bst[b] = stq[(8 + b) * kWave];
                if constexpr (!LAZY) babar[b] = stq[(8 + NBAR + b) * kWave];
            }
#pragma unroll
            for (int g = 0; g < NGRP; ++g) {
                gsum[g] = stq[(8 + 2 * NBAR + g) * kWave];
                gq[g] = stq[(8 + 2 * NBAR + NGRP + g) * kWave];
            }
            nzw = __builtin_amdgcn_ballot_w64(ps.nzero != 0) != 0;
        } else {
            // ---- forward sweep
            // adjoint kernels: waves in the forward (vector-ALU bound) take issue
            // priority over waves in the reverse (bound by LDS atomics)
            if constexpr (AD) __builtin_amdgcn_s_setprio(1);
            if constexpr (DUP) x = R(P.x0); else x = R(s0);   // Dupire: log-spot state; BS: spot
            {
                const int s = step_sample[0];
                if (s >= 0) observe(s, UNDER ? zone_spot(x) : DUP ? state_spot(x, s0) : x, row_of(s, 0));
            }
            // step i0 + k, with every per-step address a fixed offset (k) from a
            // base formed once per group of steps at i0.  GRP: a step of an
            // aligned group of four whose state and bracket the caller stores
            // at once (interleaved FP32 checkpoints), else stored here.
            R gx[4];
            uint32_t glo = 0;
            R gz[4];          // QW: the group's four normals, drawn before its steps
            uint64_t fbits = 0;   // UNDER: bit b, point 64 (i >> 6) + 1 + b is a sample
            uint64_t open = UNDER || BSR ? ~__builtin_amdgcn_ballot_w64(ps.dead) : 0;   // the lanes not breached
            auto fwd_step = [&](int i0, int k, auto grp, auto qw) {
                constexpr bool GRP = decltype(grp)::value, QW = decltype(qw)::value;
                const int i = i0 + k;
                SampleRow row{};
                if constexpr (BOOK && DUP) row = bk_rows(i + 1);
                R g;
                if constexpr (QW) g = gz[k];
                else if constexpr (MRG || LEAN) g = draw(i);
                else g = inv_normal(hl[i] ^ low_word(i), invn_tab);
                if constexpr (DUP) {
                    if constexpr (GRP) gx[k] = x;
                    else if constexpr (IL) ck[ck_el(i)] = x;
                    else if constexpr (ADJ == ADJ_CHECKPOINT) (ck + i0 * kWave + lane)[k * kWave] = x;
                    if constexpr (RECOMP)
                        if ((i & (kSeg - 1)) == 0) ck[(i / kSeg) * kWave + lane] = x;
                    const int lo = knot_count(x);
                    if constexpr (GRP) glo |= uint32_t(lo) << (8 * k);
                    else if constexpr (IL) { if (ck_lo) ckl[ck_el(i)] = uint8_t(lo); }
                    else if constexpr (CKB) { if (ck_lo) (ckl + i0 * kWave + lane)[k * kWave] = uint8_t(lo); }
                    const Bracket<R> b = local_vol_at(kxi, (iv + i0 * mp) + k * mp, x, lo);
                    x = euler_step(x, b.vol, g);
                } else {
                    if constexpr (ADJ == ADJ_CHECKPOINT) ck[i * kWave + lane] = g;
                    if constexpr (BSR) {
                        const R* r = bsr + i0 * kBsReals + k * kBsReals;
                        x = x * rexp(r[0] + r[1] * g);         // mcMdlBS.h:344-345
                        // (as for Dupire: a sample other than the last one
                        // changes nothing on a path under the zone or breached)
                        const R F = x * r[2];
                        if ((__builtin_amdgcn_ballot_w64(F > R(P.minus_smooth)) & open) != 0) {
                            observe(__builtin_amdgcn_readfirstlane((step_sample + i0 + 1)[k]), x, row);
                            open = ~__builtin_amdgcn_ballot_w64(ps.dead);
                        }
                        return;
                    } else {
                        x = x * rexp(drift[i] + stdv[i] * g);
                    }
                }
                // a wave-uniform test: the sample's code runs with all lanes (a lane
                // under the zone changes nothing there)
                if constexpr (UNDER) {
                    // (a group of four steps lies in one window of 64)
                    if ((QW ? k == 0 : true) && (i & 63) == 0) fbits = sample_bits(i + 1);
                    if (((fbits >> (i & 63)) & 1u) && (__builtin_amdgcn_ballot_w64(x > x_lo) & open) != 0) {
                        observe(0, zone_spot(x), SampleRow{});
                        open = ~__builtin_amdgcn_ballot_w64(ps.dead);
                    }
                } else if constexpr (BOOK && DUP) {
                    // (a plain barrier sample changes nothing while every state
                    // is under the zones)
                    if ((row.bars | row.grps) != 0 || row.van_hi > row.van_lo)
                        if (!(row.grps & kBookPlain) || __builtin_amdgcn_ballot_w64(x > bk_xlo) != 0)
                            observe(0, state_spot(x, s0), row);
                } else {
                    const int s = __builtin_amdgcn_readfirstlane((step_sample + i0 + 1)[k]);
                    if (s >= 0) observe(s, DUP ? state_spot(x, s0) : x, row_of(s, 0));
                }
            };
            // FP32 Dupire kernels other than the book: groups of four steps,
            // their Sobol words in two 16-byte reads and their four normals
            // drawn side by side (the book's sample code, four times over, and
            // FP64 measured slower).  A step is 25 vector instructions and five
            // LDS reads, from 33 and six; pricing 2^19 paths x 156 steps 0.116 ->
            // 0.101 ms, 2^20 paths' risk 0.379 -> 0.363, recompute 0.557 -> 0.395
            // (its knot search from LDS, the entry half as wide).
            constexpr int UF = ((DUP && !BOOK) || BSR) && sizeof(R) == 4 ? 4 : 1;
            int i = 0;
            if constexpr (UF > 1) {
                // (UF = 4 kernels with interleaved checkpoints: one 16-byte
                // store of the four states and one word of brackets per group)
                constexpr bool GRP = IL && UF == 4;
                // (the quads layout: the group's four Sobol words in two 16-byte reads)
                constexpr bool QW = QUADS && UF == 4;
                for (; i + UF <= n; i += UF) {
                    glo = 0;
                    if constexpr (QW) {
                        uint32_t gw[4];
                        sobol_words4(lo_tab, hl, lane, i, gw);
#pragma unroll
                        for (int k = 0; k < 4; ++k) gz[k] = inv_normal(gw[k], invn_tab);
                    }
    #pragma unroll
                    for (int k = 0; k < UF; ++k)
                        fwd_step(i, k, std::integral_constant<bool, GRP>{}, std::integral_constant<bool, QW>{});
                    if constexpr (GRP) {
                        *reinterpret_cast<float4*>(ck + ck_el(i)) = make_float4(gx[0], gx[1], gx[2], gx[3]);
                        if (ck_lo) *reinterpret_cast<uint32_t*>(ckl + ck_el(i)) = glo;
                    }
                }
            }
            // FP64: four draws at a time with the inverse normal's tail once
            // per wave (inv_normal4_p), the steps one by one (not the book:
            // its four steps' code measured slower there)
            if constexpr (sizeof(R) == 8 && !BOOK) {
                double* trow = tails + wave * TR;
                for (; i + 4 <= n; i += 4) {
                    if constexpr (MRG) {
                        double pu[4];
#pragma unroll
                        for (int k = 0; k < 4; ++k) pu[k] = gen.uniform(i + k);
                        inv_normal4_p<TR, SPLIT>(pu, gz, trow, mtab, lane);
                        if (gen.neg) {
#pragma unroll
                            for (int k = 0; k < 4; ++k) gz[k] = -gz[k];
                        }
                    } else {
                        uint32_t gw[4];
                        words4(i, gw);
                        inv_normal4_f64<TR, SPLIT>(gw, gz, trow, mtab, lane);
                    }
#pragma unroll
                    for (int k = 0; k < 4; ++k)
                        fwd_step(i, k, std::integral_constant<bool, IL>{}, std::true_type{});
                    if constexpr (IL) {
                        double2* c = reinterpret_cast<double2*>(ck + ck_el(i));
                        c[0] = make_double2(gx[0], gx[1]);
                        c[1] = make_double2(gx[2], gx[3]);
                        if (ck_lo) *reinterpret_cast<uint32_t*>(ckl + ck_el(i)) = glo;
                        glo = 0;
                    }
                }
            }
            if constexpr (sizeof(R) == 8 && BOOK) {
                // the book, FP64: the same four-draw batches, the steps
                // in a loop that is not unrolled (each takes its draw by a
                // select, so the book's step is compiled once)
                double* trow = tails + wave * TR;
                double gb[4] = {0.0, 0.0, 0.0, 0.0};
                for (; i < n; ++i) {
                    const int k = i & 3;
                    if (k == 0 && i < n4) {
                        if constexpr (MRG) {
                            double pu[4];
#pragma unroll
                            for (int j = 0; j < 4; ++j) pu[j] = gen.uniform(i + j);
                            inv_normal4_p<TR, SPLIT>(pu, gb, trow, mtab, lane);
                            if (gen.neg) {
#pragma unroll
                                for (int j = 0; j < 4; ++j) gb[j] = -gb[j];
                            }
                        } else {
                            uint32_t gw[4];
                            words4(i, gw);
                            inv_normal4_f64<TR, SPLIT>(gw, gb, trow, mtab, lane);
                        }
                    }
                    if (i < n4) gz[0] = k == 0 ? gb[0] : k == 1 ? gb[1] : k == 2 ? gb[2] : gb[3];
                    else gz[0] = draw(i);
                    fwd_step(i, 0, std::false_type{}, std::true_type{});
                }
            } else {
                for (; i < n; ++i) fwd_step(i, 0, std::false_type{}, std::false_type{});
            }

            // ---- payoffs of the barrier (known at the end of the path)
            if constexpr (PRD == PRD_BARRIER) {
                if (last >= 0) {   // mcPrd.h:281-287, at the last sample (timeline point n)
                    const R S = DUP ? state_spot(x, s0) : x;
                    const R F = DUP ? S : S * R(s_ff[last]);
                    const R numv = DUP ? R(1) : (P.spot_measure ? R(s_num[last]) * S : R(s_num[last]));
                    const R k = R(P.strike);
                    const R intrinsic = P.put ? (k - F > R(0) ? k - F : R(0)) : (F - k > R(0) ? F - k : R(0));
                    ps.euro = intrinsic / numv;
                    ps.fin_f = F;
                    ps.fin_num = numv;
                }
                const R p0 = ps.dead ? R(0) : ps.alive * ps.euro;
                const R p1 = ps.euro;
                const double v0 = active ? double(p0) : 0.0, v1 = active ? double(p1) : 0.0;
                const double a0 = wave_sum(v0), a1 = wave_sum(v1), b0 = wave_sum(v0 * v0), b1 = wave_sum(v1 * v1);
                if (lane == kSumLane) { accw[0] += a0; accw[1] += a1; accw[npay] += b0; accw[npay + 1] += b1; }
                if (P.per_path && active) { P.per_path[pidx * 2] = v0; P.per_path[pidx * 2 + 1] = v1; }
                if constexpr (AD) ps.aggp = R(wts[0]) * p0 + R(wts[1]) * p1;
            }
        }
        if constexpr (AD) {
            __builtin_amdgcn_s_setprio(0);
            if (ck_mode != 2) {
                const double agg = active ? double(ps.aggp) : 0.0;
                const double as = wave_sum(agg), aq = wave_sum(agg * agg);
                if (lane == kSumLane) { accw[2 * npay] += as; accw[2 * npay + 1] += aq; }
                if (P.per_path_agg && active) P.per_path_agg[pidx] = agg;
            }
            if (ck_mode == 1) {
                // forward only: keep the end state for the reverse-only launches
                stq[0] = x;
                stq[1 * kWave] = ps.alive;
                stq[2 * kWave] = ps.pnz;
                stq[3 * kWave] = R(BOOK ? int(zmask) : ps.nzero);
                stq[4 * kWave] = ps.dead ? R(1) : R(0);
                stq[5 * kWave] = ps.euro;
                stq[6 * kWave] = ps.fin_f;
                stq[7 * kWave] = ps.fin_num;
#pragma unroll
                for (int b = 0; b < NBAR; ++b) {
                    stq[(8 + b) * kWave] = bst[b];
                    if constexpr (!LAZY) stq[(8 + NBAR + b) * kWave] = babar[b];
                }
#pragma unroll
                for (int g = 0; g < NGRP; ++g) {
                    stq[(8 + 2 * NBAR + g) * kWave] = gsum[g];
                    stq[(8 + 2 * NBAR + NGRP + g) * kWave] = gq[g];
                }
                continue;
            }
            if constexpr (BOOK && ITEM) {
                // the weighted adjoints: each barrier's weight x vanilla (the
                // adjoint of its survival factor); per fixing schedule, from
                // the average and the numeraire, the adjoint of each fixing
                // sum_a w_a d max(.)/d avg / n / numeraire and the weighted
                // intrinsic values (the numeraire adjoint)
#pragma unroll
                for (int b = 0; b < NBAR; ++b)
                    if (b < P.bk.n_bar) {
                        const R w = R(wts[bk_bar_col[b]]);
                        if constexpr (LAZY) bst[b] = w != R(0) ? bst[b] : R(-1);
                        else babar[b] = w * babar[b];
                    }
#pragma unroll
                for (int g = 0; g < NGRP; ++g) {
                    if (g >= P.bk.n_grp) continue;
                    const R avg = gsum[g], numv = gq[g], inv_n = bk_ginv[g];
                    R dsum = R(0), qsum = R(0);
                    for (int a = bk_grp_first[g]; a < bk_grp_first[g + 1]; ++a) {
                        const R k = R(bk_as_strike[a]);
                        const bool put = bk_as_put[a] != 0;
                        const R intrinsic = put ? (k - avg > R(0) ? k - avg : R(0)) : (avg - k > R(0) ? avg - k : R(0));
                        const R w = R(wts[bk_as_col[a]]);
                        const R d = put ? (k > avg ? R(-1) : R(0)) : (avg > k ? R(1) : R(0));
                        dsum = dsum + w * d;
                        qsum = qsum + w * intrinsic;
                    }
                    gsum[g] = dsum * inv_n / numv;
                    gq[g] = qsum;
                }
            }

            const R w0 = R(wts[0]);
            const R w1 = npay > 1 ? R(wts[1]) : R(0);
            // A path whose adjoint is zero at the last point and stays zero
            // adds nothing: the barrier's vanilla out of the money, or breached
            // and no weight on the vanilla; the European out of the money.
            // Its lane issues no atomics, the load of the LDS pipe in these
            // kernels (2^20 paths x 156 steps, strike 120 on a spot of 100: FP32
            // 0.53 -> 0.38 ms, FP64 0.92 -> 0.80, FP32 recompute 0.63 -> 0.56).
            // (A state or weight out of range is not left out.)
            bool live = active;
            if constexpr ((DUP && (PRD == PRD_BARRIER || PRD == PRD_EUROPEAN)) || BSR) {
                const R F = DUP ? state_spot(x, s0) : ps.fin_f, k = R(P.strike);
                const bool in = PRD == PRD_BARRIER && P.put ? k > F : F > k;
                const bool zero = PRD == PRD_EUROPEAN ? ns == 1 && !in : !in || (ps.dead && w1 == R(0));
                live = active && !(zero && x - x == R(0) && F - F == R(0) && (w0 + w1) - (w0 + w1) == R(0));
            }
            // PK: the swept paths of up to ck_slots blocks are gathered, each
            // lane of a sweep reading the checkpoints and the end state of its
            // own block's slot (the end state in the slot's guard rows), until
            // they fill a wave, their slots are all taken or the wave's last
            // block is done; pk_cnt: the paths of the sweep.
            int pk_cnt = kWave;
            uint32_t src = uint32_t(lane);
            bool pk_last = false;
            if (PK && ck_slots > 1) {
                ck[lane - kWave] = x;
                if constexpr (PRD == PRD_BARRIER) {
                    // (the product of the factors, with zero ones that of the others)
                    ck[lane - 2 * kWave] = ps.nzero == 0 ? ps.alive : ps.pnz;
                    ck[lane - 3 * kWave] = ps.euro;
                }
                // (other lanes read the slot: after its stores)
                __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
                const uint64_t lm = __builtin_amdgcn_ballot_w64(live);
                const int nl = __builtin_popcountll(lm), total = pk_n + nl;
                // the live lanes from lane pk_n on, the others behind them
                auto rank = [&](uint64_t mk) {
                    return int(__builtin_amdgcn_mbcnt_hi(uint32_t(mk >> 32), __builtin_amdgcn_mbcnt_lo(uint32_t(mk), 0u)));
                };
                const int dst = pk_n + (live ? rank(lm) : nl + rank(~lm));
                const uint32_t mine = uint32_t(lane) | uint32_t(pk_slot) << 6 | uint32_t(min(ps.nzero, 2)) << 28 |
                                      (ps.dead ? 1u << 30 : 0u);
                const uint32_t got = uint32_t(__builtin_amdgcn_ds_permute((dst & (kWave - 1)) << 2, int(mine)));
                src = lane < pk_n ? pk_src : got;
                pk_last = q + int64_t(nblk) * waves > qe;
                bool kept;
                if (total >= kWave) {
                    pk_src = got;
                    pk_n = total - kWave;
                    kept = pk_n > 0;
                    pk_used = kept ? 1 : 0;
                } else {
                    pk_src = src;
                    pk_used += nl > 0 ? 1 : 0;
                    pk_cnt = pk_last || pk_used == ck_slots ? total : 0;
                    kept = nl > 0 && pk_cnt == 0;
                    pk_n = total;
                    if (pk_cnt > 0) { pk_n = 0; pk_used = 0; }
                }
                if (kept) {
                    pk_slot = pk_slot + 1 == ck_slots ? 0 : pk_slot + 1;
                    ck = ck0 + size_t(pk_slot) * ck_rows * kWave;
                    ckl = ckl0 + size_t(pk_slot) * ck_rows * kWave * sizeof(R);
                }
            } else if constexpr (PK) {
                if (__builtin_amdgcn_ballot_w64(live) == 0) pk_cnt = 0;
            }

            // (one sweep, two where the wave's last block leaves a rest; the
            // body, to the end of the block's work, is not indented further)
            for (bool more = pk_cnt > 0; more;) {
            more = false;
            // the lane's path of the sweep: its lane in the block and its slot
            int rl = lane;
            uint32_t so = 0;
            if (PK && ck_slots > 1) {
                live = lane < pk_cnt;
                if (!live) src = __builtin_amdgcn_readfirstlane(src);
                rl = int(src & 63u);
                so = ((src >> 6) & 63u) * uint32_t(ck_rows * kWave);
                const R* e = ck0 + (so + uint32_t(rl));
                x = e[-kWave];
                if constexpr (PRD == PRD_BARRIER) {
                    ps.nzero = int((src >> 28) & 3u);
                    ps.dead = (src >> 30) != 0;
                    ps.pnz = e[-2 * kWave];
                    ps.alive = ps.nzero == 0 ? ps.pnz : R(0);
                    ps.euro = e[-3 * kWave];
                    nzw = __builtin_amdgcn_ballot_w64(ps.nzero != 0) != 0;
                }
                if (pk_last && pk_n > 0) { more = true; src = pk_src; pk_cnt = pk_n; pk_n = 0; }
            }
            // checkpoints of the lane's path: byte offsets of the states and
            // brackets of an aligned group of four, and of a state row
            const uint32_t vx = (so + uint32_t(rl << 2)) * uint32_t(sizeof(R));
            const uint32_t vb4 = so * uint32_t(sizeof(R)) + uint32_t(rl << 2);
            auto at = [](const void* base, uint32_t off) -> const char* {
                return static_cast<const char*>(base) + off;
            };
            const R* const ckr = PK ? ck0 : ck;
            const uint8_t* const cklr = PK ? ckl0 : ckl;

            // book: the spot above which barrier b has an adjoint on this
            // lane, the lower end of its zone, or +infinity (breached, the
            // vanilla out of the money or without weight).  Kept per barrier in
            // a register (FP64 in float, under the zone by more than its
            // rounding), so that a sample's test is one comparison: as masks
            // they would spill from scalar registers.  rv_lo, rv_x: the lowest
            // of them, as a spot and as a state.
            float rth[NBAR];
            R rv_lo = R(INFINITY), rv_x = R(INFINITY);
            if constexpr (BOOK) {
                float lo_min = INFINITY;
#pragma unroll
                for (int b0 = 0; b0 + 3 < NBAR; b0 += 4) {
#pragma unroll
                    for (int b = b0; b < b0 + 4; ++b) rth[b] = INFINITY;
                    if (b0 >= P.bk.n_bar) continue;
#pragma unroll
                    for (int b = b0; b < b0 + 4; ++b) {
                        const float lo = float(bk_four_c[b >> 2].lo[b & 3]);
                        const float th = sizeof(R) == 4 ? lo : lo - 1e-6f * fabsf(lo);
                        if constexpr (LAZY) rth[b] = bst[b] > R(0) ? th : INFINITY;
                        else rth[b] = bst[b] > R(0) && babar[b] != R(0) ? th : INFINITY;
                        lo_min = fminf(lo_min, rth[b]);
                    }
                }
                rv_lo = R(lo_min);
                if constexpr (DUP) {
                    const R xl = sizeof(R) == 4 ? R(__logf(lo_min / float(s0))) : R(log(double(lo_min)));
                    rv_x = lo_min > 0.0f ? xl - R(sizeof(R) == 4 ? 1e-4 : 1e-10) * (R(1) + fabs(xl)) : R(-INFINITY);
                    if (!(lo_min < INFINITY)) rv_x = R(INFINITY);
                }
            }

            const bool zany = BOOK && ZT && __builtin_amdgcn_ballot_w64(zmask != 0) != 0;

            // adjoints of the forward, numeraire and discount at sample s
            const R alive_eff = ps.dead ? R(0) : ps.alive;
            const R euro_bar = w0 * alive_eff + w1;       // barrier: adjoint of the vanilla
            const R alive_bar = w0 * ps.euro;             // barrier: adjoint of alive
            // at_last: s is the last sample (the last timeline point); the
            // sweeps pass a constant false inside their step loops
            // Fz: the spot the forward took the barrier's smoothing factor at
            // sm: the book's row of the sample
            auto sample_adj = [&](int s, SampleRow sm, R F, R Fz, R numv, R discv, R& Fb, R& nb, R& db, bool at_last) {
                Fb = R(0); nb = R(0); db = R(0);
                if constexpr (PRD == PRD_BARRIER) {
                    // d alive / dF = -(product of the other factors) / 2w: alive / f
                    // without a zero factor; with one, pnz for the zero factor
                    // and 0 for the others; 0 with two or more
                    const bool zone = !ps.dead && Fz > R(P.minus_smooth);
                    const R f = (ZT ? R(P.bar_smooth) - Fz : max(R(P.bar_smooth) - Fz, tiny_d)) * R(P.inv_two_smooth);
                    R others = recip_mul(ps.alive, f);
                    if (ZT && __builtin_expect(nzw, 0))
                        others = ps.nzero == 0 ? others : ((ps.nzero == 1 && f == R(0)) ? ps.pnz : R(0));
                    if (zone) Fb -= alive_bar * others * R(P.inv_two_smooth);
                    if (at_last) {
                        const R k = R(P.strike);
                        const R dmax = P.put ? (k > F ? R(-1) : R(0)) : (F > k ? R(1) : R(0));
                        Fb += euro_bar * dmax / numv;
                        nb += -euro_bar * ps.euro / numv;
                    }
                } else if constexpr (PRD == PRD_EUROPEAN) {
                    const R k = R(P.strike);
                    const R ind = F > k ? R(1) : R(0);
                    const R intrinsic = F > k ? F - k : R(0);
                    Fb = w0 * ind * discv / numv;
                    db = w0 * intrinsic / numv;
                    nb = -w0 * intrinsic * discv / (numv * numv);
                } else if constexpr (PRD == PRD_BOOK) {
                    for (int k = sm.van_lo; k < sm.van_hi; ++k) {
                        const R kk = R(bk_van_strike[k]);
                        const R wk = R(wts[bk_van_col[k]]);
                        if (F > kk) {
                            Fb += wk / numv;
                            nb += -wk * (F - kk) / (numv * numv);
                        }
                    }
                    // d alive / dF = -(product of the other factors) / 2w: the
                    // state over the factor without a zero factor; with one,
                    // its product for the zero factor and 0 for the others
                    auto zone_adj = [&](int b, R up, R i2s) {
                        if constexpr (ZT) {
                            // v: the weighted vanilla times the state
                            const R v = LAZY ? bst[b] : babar[LAZY ? 0 : b] * bst[b], d = up - F;
                            R a = recip_mul(v, d);
                            if (zany) {
                                asm volatile("");   // (rare: a branch of its own)
                                if ((zmask >> b) & 1u) a = d == R(0) ? v * i2s : R(0);
                            }
                            Fb -= a;
                        } else {
                            // FP32 (factors at least 1e-30)
                            const R f = max((up - F) * i2s, R(1e-30));
                            Fb -= babar[b] * i2s * recip_mul(bst[b], f);
                        }
                    };
                    const uint32_t bm = sm.bars & 0xffffu;
                    uint32_t bl = sm.bars >> 16;
                    const float Ff = float(F);
                    const bool above = bm && __builtin_amdgcn_ballot_w64(F > rv_lo) != 0;
                    if (bl || (!DUP && above)) {
                        // (opaque: the tests of the mask's bits stay here,
                        // where some barrier matures)
                        asm volatile("" : "+s"(bl));
#pragma unroll
                        for (int b = 0; b < NBAR; ++b) {
                            if (!(((bm | bl) >> b) & 1u)) continue;
                            const BarPar bp = bar_par(b);
                            if ((bl >> b) & 1u) {
                                const int col = bk_bar_col[b];
                                const R k = bp.k;
                                const bool put = bk_bar_put[b] != 0;
                                const R intrinsic = put ? (k - F > R(0) ? k - F : R(0))
                                                        : (F - k > R(0) ? F - k : R(0));
                                const R dmax = put ? (k > F ? R(-1) : R(0)) : (F > k ? R(1) : R(0));
                                // (one expression, one rounding)
                                const R euro_bar = R(wts[col]) * bar_alive(b) + R(wts[col + 1]);
                                Fb += euro_bar * dmax / numv;
                                nb += -euro_bar * (intrinsic / numv) / numv;
                                if constexpr (LAZY) bst[b] = R(wts[col]) * intrinsic * bst[b];
                            }
                            if (Ff > rth[b] && F > bp.lo && ((bm >> b) & 1u)) zone_adj(b, bp.up, bp.i2s);
                        }
                    } else if (DUP && above) {
                        // some lane is above the lowest zone that its path
                        // has an adjoint in (one sample in three of the
                        // 55-payoff book); then few barriers have one.
                        // (Black-Scholes takes the loop above for both, a copy
                        // of the zones' code less in kernels of some 90 KB
                        // beside an instruction cache of 64: FP64 risk of 5
                        // steps 98 -> 95 us.)
#pragma unroll
                        for (int b = 0; b < NBAR; ++b) {
                            if (Ff > rth[b]) {
                                if ((bm >> b) & 1u) {
                                    const R lo = bk_four_c[b >> 2].lo[b & 3];
                                    if (sizeof(R) == 4 || F > lo)
                                        zone_adj(b, bk_four_c[b >> 2].up[b & 3], bk_four_c[b >> 2].i2s[b & 3]);
                                }
                            }
                        }
                    }
                    const uint32_t gm = sm.grps & 0xfu, gl = (sm.grps >> 4) & 0xfu;
                    if (gm) {
#pragma unroll
                        for (int g = 0; g < NGRP; ++g) {
                            if (!((gm >> g) & 1u)) continue;
                            Fb += gsum[g];
                            if ((gl >> g) & 1u) nb += -gq[g] / (numv * numv);
                        }
                    }
                } else {
                    for (int k = pay_first[s]; k < pay_first[s + 1]; ++k) {
                        const R kk = R(pay_strike[k]);
                        const R wk = R(wts[k]);
                        if (F > kk) {
                            Fb += wk / numv;
                            nb += -wk * (F - kk) / (numv * numv);
                        }
                    }
                }
            };

            // Dupire barrier, a sample before the last: S x d payoff / dF for spot S,
            // = -alive_bar (product of the other factors) S / 2w in the zone.
            // Without a zero factor the other factors' product is alive / f with
            // f = (B + w - S) / 2w, so the adjoint is kz S / (B + w - S),
            // kz = -alive_bar alive; with one, pnz at the zero factor
            const R kz = -alive_bar * (ps.dead ? R(0) : ps.alive);
            auto barrier_sf = [&](R S) -> R {
                const bool zone = !ps.dead && S > R(P.minus_smooth);
                const R d = ZT ? R(P.bar_smooth) - S : max(R(P.bar_smooth) - S, tiny_d);
                R sf = kz * recip_mul(S, d);
                if (ZT && __builtin_expect(nzw, 0))
                    sf = ps.nzero == 0 ? sf
                                       : ((ps.nzero == 1 && d * R(P.inv_two_smooth) == R(0))
                                              ? -alive_bar * ps.pnz * R(P.inv_two_smooth) * S : R(0));
                return zone ? sf : R(0);
            };

            const R x_adj = UNDER ? (ps.dead || ps.euro == R(0) ? R(INFINITY) : x_lo) : R(0);

            if constexpr (DUP && RECOMP) {
                // ---- reverse sweep, recompute variant: segments of kSeg steps
                // from the last one back; each segment is first re-simulated
                // from its stored state (Sobol point, inverse normal, local
                // vol), keeping in registers the step's local derivatives
                //   abar_i = abar_{i+1} (1 + (g - vol) dvol/dx) + sample adjoint
                //   vol adjoint = abar_{i+1} (g - vol), split on the two nodes
                R abar = R(0);
                {
                    const int s = step_sample[n];
                    if (s >= 0) {
                        const R S = state_spot(x, s0);
                        R Fb, nb, db;
                        sample_adj(s, row_of(s, n), S, zone_spot(x), R(1), R(1), Fb, nb, db, true);   // step_sample[n] is the last sample
                        abar = S * Fb;
                    }
                }
                const int nseg = (n + kSeg - 1) / kSeg;
                for (int sg = nseg - 1; sg >= 0; --sg) {
                    const int i0 = sg * kSeg;
                    R xi = ck[sg * kWave + lane];
                    R ca[kSeg], cb[kSeg], cw[kSeg], cv[kSeg];
                    int cj[kSeg];
                    // quads layout: the segment's Sobol words, four at a time
                    // (a group from step n on is not read)
                    uint32_t sw[kSeg];
                    if constexpr (QUADS) {
                        static_assert(kSeg % 4 == 0, "segments of whole groups of four");
#pragma unroll
                        for (int q4 = 0; q4 < kSeg; q4 += 4)
                            if (i0 + q4 < n) sobol_words4(lo_tab, hl, lane, i0 + q4, sw + q4);
                    }
                    // mrg32k3a: the segment's normals drawn top down, so the
                    // generator only steps back over the reverse sweep; FP64
                    // Sobol: the segment's four draws with the inverse
                    // normal's tail once per wave (steps from n on draw 1/2)
                    R mz[kSeg];
                    if constexpr (MRG && sizeof(R) == 8) {
                        static_assert(kSeg == 4, "FP64 segments of four draws");
                        double pu[4];
#pragma unroll
                        for (int k = 3; k >= 0; --k) pu[k] = i0 + k < n ? gen.uniform(i0 + k) : 0.5;
                        inv_normal4_p<TR, SPLIT>(pu, mz, tails + wave * TR, mtab, lane);
                        if (gen.neg) {
#pragma unroll
                            for (int k = 0; k < 4; ++k) mz[k] = -mz[k];
                        }
                    } else if constexpr (MRG) {
#pragma unroll
                        for (int k = kSeg - 1; k >= 0; --k) mz[k] = i0 + k < n ? draw(i0 + k) : R(0);
                    } else if constexpr (sizeof(R) == 8) {
                        static_assert(kSeg == 4, "FP64 segments of four draws");
                        uint32_t gw[4];
#pragma unroll
                        for (int k = 0; k < 4; ++k) gw[k] = 0x80000000u;
                        if (i0 + 4 <= n) {
                            words4(i0, gw);
                        } else {
#pragma unroll
                            for (int k = 0; k < 3; ++k)
                                if (i0 + k < n) gw[k] = hl[i0 + k] ^ low_word(i0 + k);
                        }
                        inv_normal4_f64<TR, SPLIT>(gw, mz, tails + wave * TR, mtab, lane);
                    }
#pragma unroll
                    for (int k = 0; k < kSeg; ++k) {
                        const int i = i0 + k;
                        ca[k] = R(1);
                        cb[k] = R(0);
                        cw[k] = R(0);
                        cv[k] = R(0);
                        cj[k] = 0;
                        if (i >= n) continue;
                        R g;
                        if constexpr (QUADS) g = inv_normal(sw[k], invn_tab);
                        else if constexpr (MRG || sizeof(R) == 8) g = mz[k];
                        else g = draw(i);
                        const Bracket<R> b = local_vol_at(kxi, iv + i * mp, xi, knot_count(xi));
                        const R ws = g - b.vol;    // d x_{i+1} / d vol
                        ca[k] = R(1) + ws * b.slope;
                        cw[k] = ws * b.wa;
                        cv[k] = ws * b.wb;
                        cj[k] = b.j;
                        const int smp = __builtin_amdgcn_readfirstlane(step_sample[i]);
                        if constexpr (UNDER) {
                            if (smp >= 0 && __builtin_amdgcn_ballot_w64(xi > x_adj) != 0)
                                cb[k] = barrier_sf(zone_spot(xi));
                        } else if (smp >= 0) {
                            const SampleRow row = row_of(smp, i);
                            if (!(row.grps & kBookPlain) || __builtin_amdgcn_ballot_w64(xi > rv_x) != 0) {
                                const R S = state_spot(xi, s0);
                                R Fb, nb, db;
                                sample_adj(smp, row, S, S, R(1), R(1), Fb, nb, db, false);
                                cb[k] = S * Fb;
                            }
                        }
                        xi = euler_step(xi, b.vol, g);
                    }
#pragma unroll
                    for (int k = kSeg - 1; k >= 0; --k) {
                        const int i = i0 + k;
                        if (i >= n) continue;
                        if (live) {
                            double* row = ivbl + i * mp;
                            atomicAdd(row + cj[k], double(abar * cw[k]));
                            atomicAdd(row + cj[k] + 1, double(abar * cv[k]));
                        }
                        abar = abar * ca[k] + cb[k];
                    }
                }
                if (live) padj[0] += double(abar) / s0;      // d log(S0) / d S0
            } else if constexpr (DUP) {
                // ---- reverse sweep over the Euler steps (mcMdlDupire.h:259-279)
                R abar = R(0);   // adjoint of the log-spot state at the current point
                {
                    const int s = step_sample[n];
                    if (s >= 0) {
                        const R S = state_spot(x, s0);
                        R Fb, nb, db;
                        sample_adj(s, row_of(s, n), S, zone_spot(x), R(1), R(1), Fb, nb, db, true);   // step_sample[n] is the last sample
                        abar = S * Fb;
                    }
                }
                R xnext = x;     // state at point i + 1
                // every local-vol node at least the recovery threshold: no
                // normal is drawn again
                const bool iv_recover = P.iv_recover != 0;
                const R vmin = R(sizeof(R) == 8 ? kRecoverVolF64 : kRecoverVolF32);
                // groups of U steps, top down to top - U + 1; the checkpoint
                // loads of the next group are issued before the current group
                // is worked (the book, with more registers: U = 1; FP64 below).
                // FP32 groups of four are the aligned groups of the interleaved
                // checkpoints (steps 4g .. 4g + 3), one 16-byte load of states
                // and one word of brackets each; the top group may be partial
                // (steps from n on are skipped).  The prefetch below step 0
                // reads the slot's guard rows (never used).
                constexpr int U = sizeof(R) == 8 ? 1 : (BOOK ? 1 : 4);
                constexpr bool VG = IL && U == 4;
                static_assert(U == 1 || VG, "groups of four steps read interleaved checkpoints");
                static_assert(U <= kCkptGuardRows, "the prefetch reads at most kCkptGuardRows rows below 0");
                R buf[U];
                int lbuf[U];
                SampleRow prow{};       // book: the row of the group's step, read a step ahead
                int rwin = -1;          // UNDER: window of 64 points held in rbits
                uint64_t rbits = 0;
                // states and brackets of steps top, top - 1, ..., top - U + 1
                auto load_group = [&](int top, R* xb, int* lb) {
                    if constexpr (VG) {
                        const int e = (top - 3) * kWave;   // an aligned group
                        const float4 v = *reinterpret_cast<const float4*>(at(ckr + e, vx));
                        xb[0] = v.w;
                        xb[1] = v.z;
                        xb[2] = v.y;
                        xb[3] = v.x;
                        const uint32_t w = ck_lo ? *reinterpret_cast<const uint32_t*>(at(cklr + e, vb4)) : 0u;
#pragma unroll
                        for (int k = 0; k < 4; ++k) lb[k] = int((w >> (8 * (3 - k))) & 0xffu);
                    } else {
                        const int e = ck_el(top);
                        xb[0] = ck[e];
                        lb[0] = ck_lo ? int(ckl[e]) : 0;
                    }
                };
                auto group = [&](int top, auto partial) {
                    constexpr bool PART = decltype(partial)::value;
                    R nbuf[U];
                    int nlbuf[U];
                    load_group(top - U, nbuf, nlbuf);
                    SampleRow nrow{};
                    if constexpr (BOOK) nrow = bk_rows(max(top - 1, 0));
                    // phase 1, independent of the adjoint chain: brackets, the
                    // derivative of each step to its vol, the sample adjoints
                    R ws[U], sl[U], wa[U], wb[U], sf[U];
                    int js[U];
                    // the sample index of each step (aligned groups: one 16-byte
                    // read); the Dupire barrier tests the window's sample bits
                    // (a group lies in one window of 64 points)
                    int smps[U];
                    if constexpr (UNDER) {
                        if ((top >> 6) != rwin) {
                            rwin = top >> 6;
                            rbits = sample_bits(rwin << 6);
                        }
#pragma unroll
                        for (int k = 0; k < U; ++k) smps[k] = int(((rbits >> ((top - k) & 63)) & 1u)) - 1;
                    } else if constexpr (VG) {
                        const int4 v = *reinterpret_cast<const int4*>(step_sample + (top - 3));
                        smps[0] = v.w;
                        smps[1] = v.z;
                        smps[2] = v.y;
                        smps[3] = v.x;
                    } else {
                        smps[0] = BOOK ? 0 : step_sample[top];
                    }
#pragma unroll
                    for (int k = 0; k < U; ++k) {
                        const int i = top - k;
                        const int smp = UNDER ? smps[k] : __builtin_amdgcn_readfirstlane(smps[k]);
                        ws[k] = R(0);
                        sl[k] = R(0);
                        wa[k] = R(0);
                        wb[k] = R(0);
                        sf[k] = R(0);
                        js[k] = 0;
                        if (PART && i >= n) continue;
                        const R xi = buf[k];
                        const int lo = ck_lo ? lbuf[k] : knot_count(xi);
                        const Bracket<R> b = local_vol_at(kxi, iv + i * mp, xi, lo);
                        // d x_{i+1} / d vol = g - vol, recovered from the two states:
                        // x_{i+1} - x_i = vol (g - vol / 2) up to the rounding of
                        // x_{i+1}; where a local vol is below the recovery
                        // threshold (rare; a wave-uniform test) the normal is
                        // drawn again
                        ws[k] = recip_mul(xnext - xi, b.vol) - R(0.5) * b.vol;
                        if (!iv_recover && __builtin_amdgcn_ballot_w64(b.vol < vmin) != 0)
                            if (b.vol < vmin) ws[k] = draw(i) - b.vol;
                        sl[k] = b.slope;
                        wa[k] = b.wa;
                        wb[k] = b.wb;
                        js[k] = b.j;
                        if constexpr (UNDER) {
                            if (smp >= 0 && __builtin_amdgcn_ballot_w64(xi > x_adj) != 0)
                                sf[k] = barrier_sf(zone_spot(xi));
                        } else {
                            const SampleRow row = BOOK ? prow : SampleRow{};
                            const bool on = BOOK ? (row.bars | row.grps) != 0 || row.van_hi > row.van_lo : smp >= 0;
                            if (on && (!(row.grps & kBookPlain) || __builtin_amdgcn_ballot_w64(xi > rv_x) != 0)) {
                                const R S = state_spot(xi, s0);
                                R Fb, nb, db;
                                sample_adj(smp, row, S, S, R(1), R(1), Fb, nb, db, false);
                                sf[k] = S * Fb;
                            }
                        }
                        xnext = xi;
                    }
                    // phase 2: the adjoint of the state, step by step backwards
                    R vb[U];
#pragma unroll
                    for (int k = 0; k < U; ++k) {
                        vb[k] = abar * ws[k];
                        abar = abar + vb[k] * sl[k];
                        abar = abar + sf[k];
                    }
                    // phase 3: scatter onto the two bracketing local-vol nodes
                    // (rows top - U + 1 .. top at fixed offsets from one base)
                    if (live) {
                        double* rows = ivbl + (top - (U - 1)) * mp;
#pragma unroll
                        for (int k = 0; k < U; ++k) {
                            if (PART && top - k >= n) continue;
                            double* row = rows + (U - 1 - k) * mp;
                            atomicAdd(row + js[k], double(vb[k] * wa[k]));
                            atomicAdd(row + js[k] + 1, double(vb[k] * wb[k]));
                        }
                    }
#pragma unroll
                    for (int k = 0; k < U; ++k) { buf[k] = nbuf[k]; lbuf[k] = nlbuf[k]; }
                    prow = nrow;
                };
                if constexpr (IL && sizeof(R) == 8) {
                    // FP64: the steps run one by one, their checkpoints loaded
                    // in groups of four one group ahead.  (A load one step
                    // ahead has some 1,000 cycles to come from HBM, less than
                    // its latency under load.  2^20 paths x 156 steps, 30 x 36
                    // grid, with the tail table in LDS: 1.04 -> 0.93 ms a call;
                    // 2^16 paths on the 60 x 36 grid 0.286 -> 0.258.)
                    if (n > 0) {
                        const int last = min(n - 1, P.rev_point);
                        if (last + 1 < n) xnext = ck[ck_el(last + 1)];
                        auto step = [&](int i, R xi, int lo, auto recover) {
                            constexpr bool REC = decltype(recover)::value;
                            int smp;
                            if constexpr (UNDER) {
                                if ((i >> 6) != rwin) {
                                    rwin = i >> 6;
                                    rbits = sample_bits(rwin << 6);
                                }
                                smp = int(((rbits >> (i & 63)) & 1u)) - 1;
                            } else {
                                smp = __builtin_amdgcn_readfirstlane(step_sample[i]);
                            }
                            if (!ck_lo) lo = knot_count(xi);
                            const Bracket<R> b = local_vol_at(kxi, iv + i * mp, xi, lo);
                            R ws = recip_mul(xnext - xi, b.vol) - R(0.5) * b.vol;
                            if constexpr (!REC)
                                if (!iv_recover && __builtin_amdgcn_ballot_w64(b.vol < vmin) != 0)
                                    if (b.vol < vmin) ws = draw(i) - b.vol;
                            R sf = R(0);
                            if constexpr (UNDER) {
                                if (smp >= 0 && __builtin_amdgcn_ballot_w64(xi > x_adj) != 0)
                                    sf = barrier_sf(zone_spot(xi));
                            } else if (smp >= 0) {
                                const R S = state_spot(xi, s0);
                                R Fb, nb, db;
                                sample_adj(smp, SampleRow{}, S, S, R(1), R(1), Fb, nb, db, false);
                                sf = S * Fb;
                            }
                            const R vb = abar * ws;
                            abar = abar + vb * b.slope;
                            abar = abar + sf;
                            if (live) {
                                double* row = ivbl + i * mp;
                                atomicAdd(row + b.j, double(vb * b.wa));
                                atomicAdd(row + b.j + 1, double(vb * b.wb));
                            }
                            xnext = xi;
                        };
                        double2 c0, c1;
                        uint32_t cw;
                        auto load4 = [&](int g) {   // (below step 0: the slot's guard rows, never used)
                            const double2* c = reinterpret_cast<const double2*>(at(ckr + (g << 8), vx));
                            c0 = c[0];
                            c1 = c[1];
                            cw = ck_lo ? *reinterpret_cast<const uint32_t*>(at(cklr + (g << 8), vb4)) : 0u;
                        };
                        auto sweep = [&](auto recover) {
                            int top = last;
                            for (; top >= n4; --top) {
                                const uint32_t e = so + uint32_t(rl);
                                step(top, (ckr + top * kWave)[e],
                                     ck_lo ? int((cklr + top * kWave)[e + so * uint32_t(sizeof(R) - 1)]) : 0, recover);
                            }
                            if (top < 0) return;
                            load4(top >> 2);
                            for (int g = top >> 2; g >= 0; --g) {
                                const double2 a0 = c0, a1 = c1;
                                const uint32_t w = cw;
                                load4(g - 1);
                                const int i = g << 2;
                                if (i + 3 <= top) step(i + 3, a1.y, int(w >> 24), recover);
                                if (i + 2 <= top) step(i + 2, a1.x, int((w >> 16) & 0xffu), recover);
                                if (i + 1 <= top) step(i + 1, a0.y, int((w >> 8) & 0xffu), recover);
                                step(i, a0.x, int(w & 0xffu), recover);
                            }
                        };
                        if (iv_recover) sweep(std::true_type{}); else sweep(std::false_type{});
                    }
                } else if (n > 0) {
                    // the sweep starts at the last point whose sample carries
                    // weight (one payoff's reverse of itemized risk: later
                    // steps have no adjoint), the next state from its checkpoint
                    const int last = min(n - 1, P.rev_point);
                    int top = VG ? ((last >> 2) << 2) + 3 : last;
                    if (top + 1 < n) xnext = ck[ck_el(top + 1)];
                    load_group(top, buf, lbuf);
                    if constexpr (BOOK) prow = bk_rows(top);
                    if (VG && top >= n) {
                        group(top, std::true_type{});
                        top -= U;
                    }
                    for (; top >= U - 1; top -= U) group(top, std::false_type{});
                }
                if (live) padj[0] += double(abar) / s0;      // d log(S0) / d S0
            } else {
                // ---- Black-Scholes: forward tangents of the spot with respect
                // to (spot, vol, rate, div), replaying the checkpointed normals
                // (mcMdlBS.h:203-225, :240-275, :288-349)
                const double* tl = P.bs_aux;     // sample times
                const double* tf = tl + ns;      // forward maturity - sample time
                const double* td = tf + ns;      // discount maturity - sample time
                const double* dt = td + ns;      // step lengths
                const double vol = P.bs_vol;
                R spot = R(s0);
                R tau[4] = {R(1.0 / s0), R(0), R(0), R(0)};   // d spot / spot
                auto accumulate = [&](int s, R S) {
                    const R ff = R(s_ff[s]);
                    const R F = S * ff;
                    const R numv = P.spot_measure ? R(s_num[s]) * S : R(s_num[s]);
                    const R discv = R(s_disc[s]);
                    R Fb, nb, db;
                    sample_adj(s, row_of(s, 0), F, F, numv, discv, Fb, nb, db, s == last);
                    // dF = F (tau + dff/ff), ff = exp(mu (Tf - t))
                    const R tfs = R(tf[s]), tds = R(td[s]), ts = R(tl[s]);
                    R dF[4] = {F * tau[0], F * tau[1], F * (tau[2] + tfs), F * (tau[3] - tfs)};
                    R dD[4] = {R(0), R(0), -tds * discv, R(0)};
                    R dN[4];
                    if (P.spot_measure) {
                        // num = exp(div t) / S0 * spot
                        dN[0] = numv * (tau[0] - R(1.0 / s0));
                        dN[1] = numv * tau[1];
                        dN[2] = numv * tau[2];
                        dN[3] = numv * (tau[3] + ts);
                    } else {
                        dN[0] = R(0); dN[1] = R(0); dN[2] = numv * ts; dN[3] = R(0);
                    }
                    if (live)
                        for (int c = 0; c < 4; ++c) padj[c] += double(Fb * dF[c] + db * dD[c] + nb * dN[c]);
                };
                {
                    const int s = step_sample[0];
                    if (s >= 0) accumulate(s, spot);
                }
                const int nrev = min(n, P.rev_point);   // samples after it carry no weight
                // barrier: only the last sample and those where a path that
                // has a survival adjoint is above the zone's lower end.  (A
                // step's numbers in the kernel's precision from one row in LDS;
                // every sample worked, sqrt(dt) and the conversions formed at
                // each step: the three risk calls of a serving burst 180 us on
                // average, now 106; the two pricing calls 173, now 122.)
                const uint64_t some = BSR ? __builtin_amdgcn_ballot_w64(live) : 0;
                const uint64_t zoned = BSR ? __builtin_amdgcn_ballot_w64(live && !ps.dead && ps.euro != R(0)) : 0;
                if constexpr (BSR) {
                    auto step = [&](int i, R g) {
                        const R* r = bsr + i * kBsReals;
                        spot = spot * rexp(r[0] + r[1] * g);
                        tau[1] = tau[1] + r[4] + r[5] * g;
                        tau[2] = tau[2] + r[6];
                        tau[3] = tau[3] - r[6];
                        const R F = spot * r[2];
                        if (i == n - 1 || (__builtin_amdgcn_ballot_w64(F > R(P.minus_smooth)) & zoned) != 0) {
                            const int s = __builtin_amdgcn_readfirstlane(step_sample[i + 1]);
                            if (s >= 0) accumulate(s, spot);
                        }
                    };
                    int i = 0;
                    if (some != 0) {
                        // (four normals at a time)
                        R g4[4] = {R(0), R(0), R(0), R(0)};
                        auto normals4 = [&](int at) {
                            if constexpr (QUADS && RECOMP) {
                                uint32_t gw[4];
                                sobol_words4(lo_tab, hl, lane, at, gw);
#pragma unroll
                                for (int k = 0; k < 4; ++k) g4[k] = inv_normal(gw[k], invn_tab);
                            } else {
#pragma unroll
                                for (int k = 0; k < 4; ++k) g4[k] = RECOMP ? draw(at + k) : ck[(at + k) * kWave + lane];
                            }
                        };
                        for (; i + 4 <= nrev; i += 4) {
                            normals4(i);
#pragma unroll
                            for (int k = 0; k < 4; ++k) step(i + k, g4[k]);
                        }
                        for (; i < nrev; ++i) step(i, RECOMP ? draw(i) : ck[i * kWave + lane]);
                    }
                } else {
                    for (int i = 0; i < nrev; ++i) {
                        R g;
                        if constexpr (RECOMP) g = draw(i);   // regenerated
                        else g = ck[i * kWave + lane];
                        spot = spot * rexp(drift[i] + stdv[i] * g);
                        const R dti = R(dt[i]);
                        const R sq = R(sqrt(dt[i]));
                        tau[1] = tau[1] + (P.spot_measure ? R(vol) * dti : -R(vol) * dti) + sq * g;
                        tau[2] = tau[2] + dti;
                        tau[3] = tau[3] - dti;
                        const int s = step_sample[i + 1];
                        if (s >= 0) accumulate(s, spot);
                    }
                }
            }
            }   // (the sweeps of this block)
        }
    }

    // ---- parameter adjoints: wave, then per-wave accumulators
    if constexpr (AD) {
        for (int c = 0; c < kMaxParamAdj; ++c) {
            const double v = wave_sum(padj[c]);
            if (lane == kSumLane) accw[2 * npay + 2 + c] += v;
        }
    }
    __syncthreads();
    for (int c = tid; c < stride; c += nthr) {
        double s = 0.0;
        for (int w = 0; w < waves; ++w) s += acc[w * stride + c];
        // (through to the memory that all caches share: see below)
        __hip_atomic_store(P.block_out + size_t(bid) * stride + c, s, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    if constexpr (!(AD && DUP)) {
        // the last block to get here sums the rows, in the order in which the
        // reduction kernel sums them (phase l of rows l, l + 64, ..., then the
        // phases), so the result does not depend on which block it is.  The
        // rows' stores and loads bypass the caches that are not shared and are
        // waited for, which orders them; a device-wide fence in each wave
        // instead writes back and drops its L2 (2^19 paths: 100 us more).
        if (P.blocks_done) {
            asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
            __syncthreads();
            int* is_last = reinterpret_cast<int*>(smem);   // (the tables are done with)
            if (tid == 0) *is_last = atomicInc(P.blocks_done, unsigned(nblk - 1)) == unsigned(nblk - 1) ? 1 : 0;
            __syncthreads();
            if (*is_last) {
                // (the columns of a wave, up to four at a time: their loads
                // and their chains of additions overlap)
                const int cols = fused_cols(npay, AD);
                auto sum = [&](auto at) {
                    constexpr int N = decltype(at)::value;
                    for (int c0 = wave; c0 < cols; c0 += N * waves) {
                        double s[N] = {}, t[N] = {};
                        for (int r = lane; r < nblk; r += kWave)
#pragma unroll
                            for (int j = 0; j < N; ++j)
                                if (c0 + j * waves < cols)
                                    s[j] += __hip_atomic_load(P.block_out + size_t(r) * stride + c0 + j * waves,
                                                              __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
#pragma unroll 16
                        for (int k = 0; k < kWave; ++k)
#pragma unroll
                            for (int j = 0; j < N; ++j) {
                                const uint64_t b = __builtin_bit_cast(uint64_t, s[j]);
                                const uint32_t lo = __builtin_amdgcn_readlane(uint32_t(b), k);
                                const uint32_t hi = __builtin_amdgcn_readlane(uint32_t(b >> 32), k);
                                t[j] += __builtin_bit_cast(double, uint64_t(hi) << 32 | lo);
                            }
#pragma unroll
                        for (int j = 0; j < N; ++j)
                            if (lane == 0 && c0 + j * waves < cols) P.reduced[c0 + j * waves] = t[j];
                    }
                };
                if (cols <= waves) sum(std::integral_constant<int, 1>{});
                else if (cols <= 2 * waves) sum(std::integral_constant<int, 2>{});
                else sum(std::integral_constant<int, 4>{});
            }
        }
    }
    if constexpr (AD && DUP) {
        double* dst = P.ivbar_blocks + size_t(bid) * n * m;
        // padded columns back onto the grid nodes: column j + 1 is node j,
        // the end columns 0 and m + 1 belong to the first and last node
        for (int e = tid; e < n * m; e += nthr) {
            const int i = e / m, j = e - i * m;
            double v = 0.0;
            for (int c = 0; c < P.ivbar_copies; ++c) {
                const double* r = ivbar + size_t(c) * ivbar_copy_stride(n, m) + size_t(i) * mp;
                v += r[j + 1];
                if (j == 0) v += r[0];
                if (j == m - 1) v += r[m + 1];
            }
            dst[e] = v;
        }
    }
}

#ifndef CF_PATH_KERNEL_ATTR
#define CF_PATH_KERNEL_ATTR
#endif

// Waves a SIMD has to hold at least (beside those that a block implies): the
// FP32 recompute book on Black-Scholes with mrg32k3a normals, bound by its
// waves, takes more than 128 registers without the limit, three waves instead
// of four (2^19 paths, 5 steps 124 against 92 us, 52 steps 409 against 264).
// The Sobol kernel needs 120 by itself, and the limit only costs it (5 steps
// 53.7 against 51.5 us, 52 steps 211 against 190).
constexpr int min_waves(int model, int prd, int real_bytes, int adj, bool mrg)
{
    return model == MODEL_BS && prd == PRD_BOOK && real_bytes == 4 && adj == ADJ_RECOMPUTE && mrg ? 4 : 1;
}

template <typename R, int MODEL, int PRD, int ADJ, bool LEAN, bool MRG, bool ITEM>
__global__ void __launch_bounds__(book_block_limit(PRD, int(sizeof(R)), ADJ), min_waves(MODEL, PRD, int(sizeof(R)), ADJ, MRG))
CF_PATH_KERNEL_ATTR path_kernel(const LaunchParams P)
{
    path_body<R, MODEL, PRD, ADJ, LEAN, MRG, ITEM>(P, int(blockIdx.x), int(gridDim.x));
}

// Several calls of one kernel in one launch: blocks [first[r], first[r + 1])
// run call r (Sobol normals, no itemized modes).  The calls' parameters sit in
// the kernel arguments, read with scalar loads like the single call's.
template <typename R, int MODEL, int PRD, int ADJ, bool LEAN>
__global__ void __launch_bounds__(book_block_limit(PRD, int(sizeof(R)), ADJ)) CF_PATH_KERNEL_ATTR
path_kernel_packed(const PackArgs A)
{
    const int b = int(blockIdx.x);
    int r = 0;
    while (r + 1 < A.n && b >= A.first[r + 1]) ++r;
    r = __builtin_amdgcn_readfirstlane(r);
    path_body<R, MODEL, PRD, ADJ, LEAN, false, false>(A.p[r], b - A.first[r], A.first[r + 1] - A.first[r]);
}

}  // namespace cfk

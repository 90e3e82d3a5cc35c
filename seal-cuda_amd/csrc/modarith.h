// modarith.h -- exact 64-bit modular arithmetic for gfx950 VALU.
//
// CDNA4 has no 64x64 multiply; every product below is lowered by the compiler to
// 32-bit v_mad_u64_u32 / v_mul_hi_u32 / v_mul_lo_u32 chains.  Moduli are < 2^61,
// so the lazy ranges [0,2q) and [0,4q) used by the NTT never overflow 64 bits.
//
// Semantics follow the reference's small-modulus arithmetic
// (src/utils/uintarithsmallmod.h:95-230, device twins src/kernelutils.cuh:99-189):
//   * Shoup multiply by a precomputed operand (w, floor(w 2^64 / q)),
//   * Barrett reduction of 64- and 128-bit values with floor(2^128 / q).
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace shc {

struct u128 {
    uint64_t lo, hi;
};

__device__ __forceinline__ uint64_t mulhi64(uint64_t a, uint64_t b) { return __umul64hi(a, b); }

__device__ __forceinline__ u128 mul64x64(uint64_t a, uint64_t b) {
    u128 r;
    r.lo = a * b;
    r.hi = __umul64hi(a, b);
    return r;
}

__device__ __forceinline__ void add128(u128 &acc, u128 v) {
    uint64_t lo = acc.lo + v.lo;
    acc.hi += v.hi + (lo < acc.lo ? 1ull : 0ull);
    acc.lo = lo;
}

// x * w mod q in [0, 2q), for any 64-bit x and w < q (Shoup, lazy).
__device__ __forceinline__ uint64_t shoup_lazy(uint64_t x, uint64_t w, uint64_t wq, uint64_t q) {
    uint64_t hi = mulhi64(x, wq);
    return x * w - hi * q;
}

// floor(x * y / 2^64) - e with e in {0, 1, 2}: the high word without the carries of
// the two middle partial products' low halves and of x_lo * y_lo (3 multiplies).
__host__ __device__ __forceinline__ uint64_t mulhi64_approx(uint64_t x, uint64_t y) {
    const uint32_t xl = (uint32_t)x, xh = (uint32_t)(x >> 32), yl = (uint32_t)y, yh = (uint32_t)(y >> 32);
    const uint64_t mid = ((uint64_t)xh * yl >> 32) + ((uint64_t)xl * yh >> 32);
    return (uint64_t)xh * yh + mid;
}

// x * w mod q in [0, 4q), for any 64-bit x, w < q < 2^62, wq = floor(w 2^64 / q) and
// neg_q = 2^64 - q.  The quotient estimate is Shoup's minus at most 2, so the remainder
// x w - Q q lies in [0, 4q) and equals its low 64 bits, computed as x w + Q neg_q with
// only the low halves of the cross products (9 multiplies in all).  The four cross products
// reach the high word alone: a chain of v_mad_u64_u32 and one 32-bit add (a v_mad_u64_u32
// issues in 5.1 cycles, a v_mul_lo_u32 in 4.7 and a v_add3_u32 in 4.4, so four and an add
// take 23 where four products and two three-way adds take 28), in inline assembly since the
// compiler turns the chain back into them.  UNI: w and wq are the same in every lane (scalar
// operands, one per instruction); neg_q always is.
template <bool UNI = false>
__host__ __device__ __forceinline__ uint64_t shoup_lazier(uint64_t x, uint64_t w, uint64_t wq, uint64_t neg_q) {
    const uint64_t Q = mulhi64_approx(x, wq);
    const uint32_t xl = (uint32_t)x, xh = (uint32_t)(x >> 32), wl = (uint32_t)w, wh = (uint32_t)(w >> 32);
    const uint32_t ql = (uint32_t)Q, qh = (uint32_t)(Q >> 32), nl = (uint32_t)neg_q, nh = (uint32_t)(neg_q >> 32);
    const uint64_t p = (uint64_t)xl * wl + (uint64_t)ql * nl;
#if defined(__HIP_DEVICE_COMPILE__)
    uint64_t c, sd;
    if constexpr (UNI)
        asm("v_mad_u64_u32 %0, %1, %2, %3, 0\n\tv_mad_u64_u32 %0, %1, %4, %5, %0\n\t"
            "v_mad_u64_u32 %0, %1, %6, %7, %0\n\tv_mad_u64_u32 %0, %1, %8, %9, %0"
            : "=&v"(c), "=&s"(sd)
            : "v"(xl), "s"(wh), "v"(xh), "s"(wl), "v"(ql), "s"(nh), "v"(qh), "s"(nl));
    else
        asm("v_mad_u64_u32 %0, %1, %2, %3, 0\n\tv_mad_u64_u32 %0, %1, %4, %5, %0\n\t"
            "v_mad_u64_u32 %0, %1, %6, %7, %0\n\tv_mad_u64_u32 %0, %1, %8, %9, %0"
            : "=&v"(c), "=&s"(sd)
            : "v"(xl), "v"(wh), "v"(xh), "v"(wl), "v"(ql), "s"(nh), "v"(qh), "s"(nl));
    uint32_t hi = (uint32_t)(p >> 32) + (uint32_t)c;
    asm("" : "+v"(hi));  // keeps the 32-bit add from being widened back to 64 bits
#else
    const uint32_t hi = (uint32_t)(p >> 32) + xl * wh + xh * wl + ql * nh + qh * nl;
#endif
    return ((uint64_t)hi << 32) | (uint32_t)p;
}

__device__ __forceinline__ uint64_t shoup(uint64_t x, uint64_t w, uint64_t wq, uint64_t q) {
    uint64_t r = shoup_lazy(x, w, wq, q);
    return r >= q ? r - q : r;
}

__device__ __forceinline__ uint64_t csub(uint64_t x, uint64_t q) { return x >= q ? x - q : x; }

// x mod q for any 64-bit x, using the high word of floor(2^128/q) (barrettReduce64).
__device__ __forceinline__ uint64_t barrett64(uint64_t x, uint64_t q, uint64_t ratio_hi) {
    uint64_t est = mulhi64(x, ratio_hi);
    uint64_t r = x - est * q;
    return r >= q ? r - q : r;
}

// v - c, or v if that is negative (neg_c = 2^64 - c; the difference in [-2^63, 2^63)).
__host__ __device__ __forceinline__ uint64_t sub_not_below(uint64_t v, uint64_t neg_c) {
    const uint64_t t = v + neg_c;
    return (int32_t)(t >> 32) < 0 ? v : t;
}

// (hi:lo) mod q for any 128-bit value and q < 2^61 (the remainder of barrettReduce128,
// uintarithsmallmod.h:95-126).  With c = 2^64 mod q the value is hi c + lo, and the halves of
// floor(2^128 / q) are the quotient constants of both terms: ratio_hi = floor(2^64 / q) is
// lo's and ratio_lo = floor(c 2^64 / q) is c's Shoup constant.  Each estimate is at most 3
// short (1 and mulhi64_approx's 2), so the remainder lies in [0, 8q) and equals its low 64
// bits.  Against the exact 128-bit quotient: no carries between products
// (128 products at N = 2^16, L = 24: 40.4 -> 39.6 ms with the sums' own).
__host__ __device__ __forceinline__ uint64_t barrett128(u128 x, uint64_t q, uint64_t ratio_lo, uint64_t ratio_hi) {
    const uint64_t c = 0 - ratio_hi * q;
    const uint64_t Q = mulhi64_approx(x.hi, ratio_lo) + mulhi64_approx(x.lo, ratio_hi);
    const uint32_t hl = (uint32_t)x.hi, hh = (uint32_t)(x.hi >> 32), cl = (uint32_t)c, ch = (uint32_t)(c >> 32);
    const uint64_t nq = 0 - q;
    const uint32_t ql = (uint32_t)Q, qh = (uint32_t)(Q >> 32), nl = (uint32_t)nq, nh = (uint32_t)(nq >> 32);
    const uint64_t p = x.lo + (uint64_t)hl * cl + (uint64_t)ql * nl;
    const uint32_t hi = (uint32_t)(p >> 32) + hl * ch + hh * cl + ql * nh + qh * nl;
    const uint64_t r = (uint64_t)hi << 32 | (uint32_t)p;
    return sub_not_below(sub_not_below(sub_not_below(r, nq << 2), nq << 1), nq);
}

__device__ __forceinline__ uint64_t mulmod(uint64_t a, uint64_t b, uint64_t q, uint64_t ratio_lo,
                                           uint64_t ratio_hi) {
    return barrett128(mul64x64(a, b), q, ratio_lo, ratio_hi);
}

__device__ __forceinline__ uint64_t addmod(uint64_t a, uint64_t b, uint64_t q) {
    uint64_t s = a + b;
    return s >= q ? s - q : s;
}

__device__ __forceinline__ uint64_t submod(uint64_t a, uint64_t b, uint64_t q) {
    return a >= b ? a - b : a + q - b;
}

__device__ __forceinline__ uint64_t negmod(uint64_t a, uint64_t q) { return a ? q - a : 0; }

}  // namespace shc

// accum.h -- sums of 64 x 64-bit products without carry chains (key-switch inner
// products).
//
// A sum of products t * k with t, k < 2^63 is kept as three 64-bit words
//   value = al + ml * 2^32 + h * 2^64,
// where each product adds
//   al += lo32(tl kl),  ml += hi32(tl kl) + lo32(m),  h += th kh + hi32(m),
//   m = th kl + tl kh
// (tl, th, kl, kh: 32-bit halves).  m < 2^64 because th, kh < 2^31; al grows by less
// than 2^32 and ml by less than 2^33 per product; h stays below 2^64 while the value is
// below 2^128, which key switching guarantees: its terms are below 8q * q < 2^123
// (q < 2^60) and a level has at most 31 digits at that size (63 below 4q * q) plus one
// correction term.  Every step is one v_mad_u64_u32 (a 32-bit word joins a 64-bit sum
// as word * 1 + sum; 64-bit products take one each): 8 VALU instructions per product,
// with no carry chains and no 64-bit shifts.  The device code states the eight
// multiply-adds in inline assembly, since the compiler otherwise re-associates the
// 32-bit pieces into 64-bit adds and register moves; they go in three groups (the two
// products of tl, then the ones that need those products' halves, then the rest)
// because the compiler puts a wait state between consecutive inline-assembly
// statements that share a register.  The same
// sums as the reference's 128-bit accumulation of key-switch products
// (src/evaluator.cpp:2520-2590: multiply_uint64 + add_uint128, then barrett_reduce_128).
#pragma once
#include "common.h"
#include "modarith.h"

namespace shc {

struct Acc3 {
    uint64_t al, ml, h;
};

// value + t * k.  KU: k is uniform across the wave (an SGPR operand, e.g. a conversion
// table entry; one per instruction, the constant-bus limit).
template <bool KU = false>
__host__ __device__ __forceinline__ void mac(Acc3 &a, uint64_t t, uint64_t k) {
    const uint32_t tl = (uint32_t)t, th = (uint32_t)(t >> 32), kl = (uint32_t)k, kh = (uint32_t)(k >> 32);
#if defined(__HIP_DEVICE_COMPILE__)
    uint64_t p, m, c;
    if constexpr (KU)
        asm("v_mad_u64_u32 %0, %2, %3, %4, 0\n\tv_mad_u64_u32 %1, %2, %3, %5, 0"
            : "=&v"(p), "=&v"(m), "=&s"(c) : "v"(tl), "s"(kl), "s"(kh));
    else
        asm("v_mad_u64_u32 %0, %2, %3, %4, 0\n\tv_mad_u64_u32 %1, %2, %3, %5, 0"
            : "=&v"(p), "=&v"(m), "=&s"(c) : "v"(tl), "v"(kl), "v"(kh));
    if constexpr (KU)
        asm("v_mad_u64_u32 %0, %3, %4, %5, %0\n\tv_mad_u64_u32 %1, %3, %6, 1, %1\n\tv_mad_u64_u32 %2, %3, %7, 1, %2"
            : "+v"(m), "+v"(a.al), "+v"(a.ml), "=&s"(c) : "v"(th), "s"(kl), "v"((uint32_t)p), "v"((uint32_t)(p >> 32)));
    else
        asm("v_mad_u64_u32 %0, %3, %4, %5, %0\n\tv_mad_u64_u32 %1, %3, %6, 1, %1\n\tv_mad_u64_u32 %2, %3, %7, 1, %2"
            : "+v"(m), "+v"(a.al), "+v"(a.ml), "=&s"(c) : "v"(th), "v"(kl), "v"((uint32_t)p), "v"((uint32_t)(p >> 32)));
    if constexpr (KU)
        asm("v_mad_u64_u32 %0, %2, %3, 1, %0\n\tv_mad_u64_u32 %1, %2, %4, 1, %1\n\tv_mad_u64_u32 %1, %2, %5, %6, %1"
            : "+v"(a.ml), "+v"(a.h), "=&s"(c) : "v"((uint32_t)m), "v"((uint32_t)(m >> 32)), "v"(th), "s"(kh));
    else
        asm("v_mad_u64_u32 %0, %2, %3, 1, %0\n\tv_mad_u64_u32 %1, %2, %4, 1, %1\n\tv_mad_u64_u32 %1, %2, %5, %6, %1"
            : "+v"(a.ml), "+v"(a.h), "=&s"(c) : "v"((uint32_t)m), "v"((uint32_t)(m >> 32)), "v"(th), "v"(kh));
#else
    const uint64_t p = (uint64_t)tl * kl;
    a.al += (uint32_t)p;
    a.ml += p >> 32;
    const uint64_t m = (uint64_t)th * kl + (uint64_t)tl * kh;
    a.ml += (uint32_t)m;
    a.h += (uint64_t)th * kh + (m >> 32);
#endif
}

// value + x for x < 2^64 (one more term, e.g. a correction).
__host__ __device__ __forceinline__ void acc_add(Acc3 &a, uint64_t x) {
    a.al += (uint32_t)x;
    a.ml += x >> 32;
}

__host__ __device__ __forceinline__ u128 acc_value(const Acc3 &a) {
    const uint64_t lo = a.al + (a.ml << 32);
    return u128{lo, a.h + (a.ml >> 32) + (lo < a.al ? 1ull : 0ull)};
}

// value mod q (< q).
__device__ __forceinline__ uint64_t acc_reduce(const Acc3 &a, const DevPrime &Q) {
    return barrett128(acc_value(a), Q.q, Q.ratio_lo, Q.ratio_hi);
}

// Replaces the value by value mod q (for sums longer than the 128-bit bound allows).
__device__ __forceinline__ void acc_fold(Acc3 &a, const DevPrime &Q) {
    const uint64_t r = acc_reduce(a, Q);
    a = Acc3{(uint32_t)r, r >> 32, 0};
}

// The same sums for primes below 2^50 and t < 2^52, as three words at weights 1, 2^26 and
// 2^52 (t and k cut at 26 bits: every partial product is below 2^52, so 64-bit words hold
// over 1,000 of them without carries): 4 multiply-adds per product instead of 8, after a
// cut of each operand (2 instructions) that serves every product it enters.
struct Cut26 {
    uint32_t lo, hi;
};
__host__ __device__ __forceinline__ Cut26 cut26(uint64_t x) {
    return Cut26{(uint32_t)x & 0x3ffffffu, (uint32_t)(x >> 26)};
}
struct Acc26 {
    uint64_t a0, a1, a2;
};
__host__ __device__ __forceinline__ void mac(Acc26 &a, Cut26 t, Cut26 k) {
    a.a0 += (uint64_t)t.lo * k.lo;
    a.a1 += (uint64_t)t.lo * k.hi;
    a.a1 += (uint64_t)t.hi * k.lo;
    a.a2 += (uint64_t)t.hi * k.hi;
}
__host__ __device__ __forceinline__ void acc_add(Acc26 &a, uint64_t x) {  // x < 2^58
    a.a0 += (uint32_t)x & 0x3ffffffu;
    a.a1 += x >> 26;
}
// (values below 2^116: what passes 26 bits of each word moves up, then the words are cut
// together without compares)
__host__ __device__ __forceinline__ u128 acc_value(const Acc26 &a) {
    const uint64_t a1 = a.a1 + (a.a0 >> 26), a2 = a.a2 + (a1 >> 26);
    const uint32_t lo = (uint32_t)a1 << 26 | ((uint32_t)a.a0 & 0x3ffffffu);
    const uint32_t hi = (uint32_t)a2 << 20 | ((uint32_t)a1 >> 6 & 0xfffffu);
    return u128{(uint64_t)hi << 32 | lo, a2 >> 12};
}
// The value mod q for q of b bits, 2 < b <= 50, and values below 2^(b + 60): 2^(58 - b) products
// of t < 4q and k < q, 256 at b = 50 (key switches and rotations sum at most 63 and two terms
// more, plain products fold every 64 of t < q).  One quotient estimate: with t = value >> (b - 2) < 2^62 and
// ratio = floor(2^(b + 62) / q) < 2^63, mulhi64_approx(t, ratio) is short by less than
// 1/2 (t) + 1/4 (ratio) + 1 (floor) + 2 (approx), so the remainder lies in [0, 4q).  About
// 55 instructions with the sum's own against 95 for a 128-bit quotient: plain_dot_tiles 4.86 ->
// 4.62 ms (1,024 diagonals, 16 ciphertexts, N = 2^15, L = 15), the products of 31 key switches
// of them 13.1 -> 12.9.
__host__ __device__ __forceinline__ uint64_t acc_reduce26(const Acc26 &a, uint64_t q, uint64_t ratio_lo,
                                                          uint64_t ratio_hi) {
    const int b = 64 - __builtin_clzll(q);
    const uint64_t ratio = ratio_hi << (b - 2) | ratio_lo >> (66 - b);
    const u128 v = acc_value(a);
    const uint64_t t = v.hi << (66 - b) | v.lo >> (b - 2);
    const uint64_t est = mulhi64_approx(t, ratio), nq = 0 - q;
    const uint32_t ql = (uint32_t)est, qh = (uint32_t)(est >> 32), nl = (uint32_t)nq, nh = (uint32_t)(nq >> 32);
    const uint64_t p = v.lo + (uint64_t)ql * nl;
    const uint32_t hi = (uint32_t)(p >> 32) + ql * nh + qh * nl;
    return sub_not_below(sub_not_below((uint64_t)hi << 32 | (uint32_t)p, nq << 1), nq);
}
__device__ __forceinline__ uint64_t acc_reduce(const Acc26 &a, const DevPrime &Q) {
    return acc_reduce26(a, Q.q, Q.ratio_lo, Q.ratio_hi);
}

__device__ __forceinline__ void acc_fold(Acc26 &a, const DevPrime &Q) {
    const Cut26 r = cut26(acc_reduce(a, Q));
    a = Acc26{r.lo, r.hi, 0};
}

}  // namespace shc

// butterfly_fp.h -- the forward NTT's butterflies in fp64 for primes below 2^50 (host and
// device).
//
// CDNA4 issues v_fma_f64 at the rate of a 32-bit multiply-add, so for a prime that leaves a
// few bits of a double's 53 free, a modular product takes 6 instructions instead of the 13
// of the 64-bit integer form (shoup_lazier: nine 32-bit multiplies and their adds), and a
// butterfly 8 instead of 17-21.  Every value is an integer held exactly in a double:
//
//   h = RN(y w), l = y w - h (exact, one fma), b = rint(RN(y RN(w/q))),
//   v = (h - b q) + l = y w - b q   exactly.
//
// (The error-free product by fma, Ogita, Rump and Oishi, "Accurate sum and dot product", 2005,
// and the modular product with a quotient from a precomputed inverse that van der Hoeven,
// Lecerf and Quintin build on it, "Modular SIMD arithmetic in Mathemagix", 2016; the bounds and
// schedules below are for this transform.)
//
// With q < 2^50, |y| <= c q, c <= 8 and |w| <= q/2 (centred): RN(y RN(w/q)) is within
// |y w / q| 2^-52 <= c 2^-3 of the quotient, so |v| <= (0.5 + c/8) q <= 1.5 q; |h| < 2^102,
// so |l| <= 2^49, and h - b q = v - l is an integer below 2^52: both additions are exact.
// The outputs x +- v are below 2^53 in magnitude as long as their bound stays <= 8 q.  With
// c_in at the input of a pass, a layer takes c to c + 0.5 + c/8, or to 1 + c/8 when x is
// first reduced to |x| <= q/2 (3 instructions: fp_center); the schedules
//   columns pass (K = 6..8 layers), c_in <= 2, x reduced at local layer 5: max 6.9, out < 3.5
//   rows pass (K = 7..9), c_in < 3.5, x reduced at layers 3 and K - 1: max 6.6, out < 1.7
// keep c below 7 (checked with extreme operands by tests/test_butterfly_bounds.py).
#pragma once
#include <hip/hip_runtime.h>
#include <math.h>
#include <stdint.h>

namespace shc {

// Primes below this take the fp64 schedule (their DevPrime has fp twiddles).
constexpr uint64_t FP_PRIME_LIMIT = uint64_t(1) << 50;

__host__ __device__ __forceinline__ double fp_center(double x, double q, double qinv) {
#pragma clang fp contract(off)
    return fma(-rint(x * qinv), q, x);
}

// y w - rint(y w / q) q, wq = RN(w / q).
__host__ __device__ __forceinline__ double fp_mulmod(double y, double w, double wq, double q) {
#pragma clang fp contract(off)
    const double h = y * w;
    const double l = fma(y, w, -h);
    const double b = rint(y * wq);
    return fma(-b, q, h) + l;
}

// (x, y) -> (x + w y, x - w y); w = (w, RN(w / q)).
__host__ __device__ __forceinline__ void fp_butterfly(double &x, double &y, double2 w, double q, double qinv,
                                                      bool center) {
#pragma clang fp contract(off)
    const double u = center ? fp_center(x, q, qinv) : x;
    const double v = fp_mulmod(y, w.x, w.y, q);
    x = u + v;
    y = u - v;
}

// Local layers of a pass that reduce x first.
__host__ __device__ constexpr bool fp_centers(bool rows, int K, int s) {
    return rows ? s == 3 || s == K - 1 : s == 5;
}

// A residue below 2^52 as a double, and a value of (-2q, 2q) as the residue x + 2q in
// (0, 4q) (below 2^52): the exponent word of 2^52 makes the mantissa the integer itself.
__host__ __device__ __forceinline__ double fp_from_u52(uint64_t x) {
    union { uint64_t u; double d; } c;
    c.u = x | 0x4330000000000000ull;
    return c.d - 4503599627370496.0;
}
__host__ __device__ __forceinline__ uint64_t fp_to_u52(double x, double two52_plus_2q) {
    union { double d; uint64_t u; } c;
    c.d = x + two52_plus_2q;
    return c.u & 0xfffffffffffffull;
}

}  // namespace shc

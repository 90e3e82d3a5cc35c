// rotations.hip -- hoisted rotation and summation, exact against separate rotations.
//
// A rotation (Evaluator::applyGaloisInplace, src/evaluator.cpp:2210-2250; GPU
// src/evaluator_cuda.cu:2011-2104) switches the key of sigma(c1), whose digits are the
// canonical residues of sigma applied to c1's coefficients.  Hoisting transforms c1's
// digits once: T_ij = NTT_i(d_j mod q_i), and sigma(T_ij) (an NTT-domain permutation)
// is the transform of sigma(d_j) mod q_i -- except where sigma negates a coefficient.
// There the reference's digit is q_j - d (for d != 0), which is q_j mod q_i above the
// hoisted -d mod q_i.  So, per target prime i and with S_sigma the 0/1 polynomial of
// negated positions,
//   sum_j NTT_i(digit_j) key_j
//     = sigma(sum_j T_ij sigma^-1(key_j)) + NTT_i(S_sigma) sum_j (q_j mod q_i) key_j
//     = sigma(sum_j T_ij key'_j + corr')
// with key' = sigma^-1(key) and corr' = sigma^-1(NTT_i(S_sigma) sum_j (q_j mod q_i) key_j),
// prepared once per key and level.  A zero digit d_j[p] = 0 at a position sigma negates
// has the reference digit 0, not q_j: corr' counted (q_j mod q_i) X^sigma(p) there, whose
// preimage under sigma is -X^p.  Each such zero is put right in the products before the
// permutation, P += (q_j mod q_i) NTT_i(X^p) key'_j (the NTT of a monomial is a power of
// the root at each slot), and a ciphertext whose digits are all zero has products zero.
// The zeros are listed on the device, so no decision waits for the host.  Each rotation
// then costs one inner product, one permutation of the 2(L+1) product limbs and one
// ModDown instead of a full ModUp (L x L transforms for CKKS, L(L+1) for BFV).
#include "rotations.h"
#include "elementwise.h"
#include "galois.h"
#include "hostmath.h"
#include "accum.h"
#include "modarith.h"
#include "ntt.h"
#include "rns_ops.h"
#include "workspaces.h"
#include <algorithm>
#include <type_traits>

namespace shc {
namespace {

constexpr int TPB = 256;

inline uint32_t blocks_for(size_t n) {
    const size_t b = (n + TPB - 1) / TPB;
    return (uint32_t)(b < (size_t(1) << 20) ? b : (size_t(1) << 20));
}

// neg[l][k] = 1 where sigma_elt negates the coefficient that lands at k (the source
// i = k elt^-1 mod N moves to i elt mod 2N, negated when that is >= N), in each limb.
__global__ void negated_positions_kernel(uint64_t *__restrict__ neg, uint32_t elt, uint32_t elt_inv, int logn,
                                         size_t total) {
    const uint32_t n = 1u << logn;
    for (size_t idx = (size_t)blockIdx.x * TPB + threadIdx.x; idx < total; idx += (size_t)gridDim.x * TPB) {
        const uint32_t k = (uint32_t)(idx & (n - 1));
        const uint32_t i = (uint32_t)(((uint64_t)k * elt_inv) & (n - 1));
        neg[idx] = (((uint64_t)i * elt) >> logn) & 1;
    }
}

// C[k][i][c] = negntt[i][c] * sum_{j<L} (q_j mod q_i) key[j][k][ki][c] mod q_i, i <= L
// (ki = i, or the special prime's key limb K-1 for i == L).
__global__ void correction_kernel(const uint64_t *__restrict__ negntt, const uint64_t *__restrict__ key,
                                  uint64_t *__restrict__ C, const DevPrime *__restrict__ targets,
                                  const DevPrime *__restrict__ data, uint32_t L, uint32_t K, int logn, size_t total) {
    const size_t n = (size_t)1 << logn;
    for (size_t idx = (size_t)blockIdx.x * TPB + threadIdx.x; idx < total; idx += (size_t)gridDim.x * TPB) {
        const size_t c = idx & (n - 1);
        const size_t r = idx >> logn;
        const uint32_t i = (uint32_t)(r % (L + 1));
        const uint32_t k = (uint32_t)(r / (L + 1));
        const DevPrime &Q = targets[i];
        const uint32_t ki = i == L ? K - 1 : i;
        Acc3 acc{0, 0, 0};
        for (uint32_t j = 0; j < L; j++) {
            const uint64_t cij = barrett64(data[j].q, Q.q, Q.ratio_hi);
            mac(acc, cij, key[(((size_t)j * 2 + k) * K + ki) * n + c]);
        }
        const uint64_t s = acc_reduce(acc, Q);
        C[idx] = mulmod(s, negntt[(size_t)i * n + c], Q.q, Q.ratio_lo, Q.ratio_hi);
    }
}

// Products of R rotations at once, each T word read once for all of them:
//   P_r[ct][k][i] = sum_j T[i][ct][j] key'_r[j][k][ki] + corr'_r[k][i]   (S_r for i == L)
// and with fold.ct (N >= 2^13), P_r[ct][0][i] += p c0[ct][i]: the ModDown then writes the
// rotation without a pass that permutes and adds c0.
// One thread per (i, c) position and RG ciphertexts (each key word it loads serves RG
// products); the loads of digit j + 1 go out before the products of digit j, and in a
// partial last group the missing ciphertext repeats the last one (in bounds, not stored).
// With diag, T holds no limb (i, i) for i < L and that term is the NTT-form input limb
// diag[ct * diag_stride + i * N].  The waves of a block take WG groups of the same
// positions, so that a key line is fetched once per block and its other readers hit the
// CU's cache; blocks of one tile run on one XCD (XCD = block % 8), whose L2 serves the
// tile's key words to the other blocks.  Sums are Acc3, or (MIXED, a block of a prime
// below 2^50: T holds words below 4 q) Acc26 at half the instructions.
constexpr int RMAX = ROT_MAX;
static_assert(RMAX <= (int)PERM_MAX, "a pass's rotations fit one permuted ModDown");
constexpr int RG = 2;
struct RotBatch {
    const uint64_t *key[RMAX];   // prepared keys; corr' follows at corr_off words
    uint64_t *P[RMAX], *S[RMAX];
    uint32_t elt[RMAX];          // their Galois elements
};
struct RotArgs {
    const uint64_t *T;
    size_t corr_off;
    const DevPrime *targets;
    uint32_t L, K;
    int logn;
    uint32_t count, tiles;
    const uint64_t *diag;
    size_t diag_stride;
    KsFold fold;                 // ct: c0 of ciphertext g at ct + g * ct_stride
};

template <int R, bool FP>
__device__ __forceinline__ void rotation_products_core(const RotBatch &rb, const RotArgs &a, uint32_t i, size_t c,
                                                       uint32_t ct0, int gv) {
    using Acc = std::conditional_t<FP, Acc26, Acc3>;
    using Word = std::conditional_t<FP, Cut26, uint64_t>;
    auto word = [](uint64_t x) -> Word {
        if constexpr (FP) return cut26(x);
        else return x;
    };
    const uint32_t L = a.L;
    const size_t n = (size_t)1 << a.logn;
    const uint32_t ki = (i == L) ? a.K - 1 : i;
    const DevPrime &Q = a.targets[i];
    const bool short_row = a.diag && i < L;  // uniform over the block
    const uint32_t Lt = short_row ? L - 1 : L;
    const uint64_t *Ti = a.T + (((size_t)i * a.count * L + (size_t)ct0 * Lt) << a.logn) + c;
    const size_t kstride = (size_t)a.K << a.logn;
    size_t goff[RG];
    const uint64_t *dp[RG];
#pragma unroll
    for (int g = 0; g < RG; g++) {
        goff[g] = ((size_t)min(g, gv - 1) * Lt) << a.logn;
        dp[g] = short_row ? a.diag + (ct0 + min(g, gv - 1)) * a.diag_stride + ((size_t)i << a.logn) + c : nullptr;
    }
    Acc a0[R][RG], a1[R][RG];
#pragma unroll
    for (int r = 0; r < R; r++)
#pragma unroll
        for (int g = 0; g < RG; g++) a0[r][g] = a1[r][g] = Acc{0, 0, 0};
    uint64_t tn[RG], k0n[R], k1n[R];
    auto fetch = [&](uint32_t j) {
        const bool dj = short_row && j == i;
        const size_t jt = short_row && j > i ? j - 1 : j;
#pragma unroll
        for (int g = 0; g < RG; g++) tn[g] = *(dj ? dp[g] : Ti + goff[g] + (jt << a.logn));
#pragma unroll
        for (int r = 0; r < R; r++) {
            const uint64_t *kp = rb.key[r] + (size_t)ki * n + c;
            k0n[r] = kp[(2 * j) * kstride];
            k1n[r] = kp[(2 * j + 1) * kstride];
        }
    };
    fetch(0);
    for (uint32_t j = 0; j < L; j++) {
        Word t[RG], k0[R], k1[R];
#pragma unroll
        for (int g = 0; g < RG; g++) t[g] = word(tn[g]);
#pragma unroll
        for (int r = 0; r < R; r++) k0[r] = word(k0n[r]), k1[r] = word(k1n[r]);
        fetch(j + 1 < L ? j + 1 : j);
#pragma unroll
        for (int r = 0; r < R; r++)
#pragma unroll
            for (int g = 0; g < RG; g++) {
                mac(a0[r][g], t[g], k0[r]);
                mac(a1[r][g], t[g], k1[r]);
            }
    }
    if (a.fold.ct && i < L) {
        const Word pm = word(a.fold.dc[i].p_mod);
#pragma unroll
        for (int g = 0; g < RG; g++) {
            const Word w = word(a.fold.ct[(ct0 + min(g, gv - 1)) * a.fold.ct_stride + ((size_t)i << a.logn) + c]);
#pragma unroll
            for (int r = 0; r < R; r++) mac(a0[r][g], w, pm);
        }
    }
#pragma unroll
    for (int r = 0; r < R; r++) {
        const uint64_t *corr = rb.key[r] + a.corr_off;
        const uint64_t c0 = corr[(size_t)i * n + c], c1 = corr[((size_t)(L + 1) + i) * n + c];
#pragma unroll
        for (int g = 0; g < RG; g++) {
            if (g >= gv) continue;
            const size_t ct = ct0 + g;
            acc_add(a0[r][g], c0);
            acc_add(a1[r][g], c1);
            const uint64_t r0 = acc_reduce(a0[r][g], Q), r1 = acc_reduce(a1[r][g], Q);
            if (i == L) {
                rb.S[r][(ct * 2 + 0) * n + c] = r0;
                rb.S[r][(ct * 2 + 1) * n + c] = r1;
            } else {
                rb.P[r][((ct * 2 + 0) * L + i) * n + c] = r0;
                rb.P[r][((ct * 2 + 1) * L + i) * n + c] = r1;
            }
        }
    }
}

template <int R, int WG, bool MIXED>
__global__ __launch_bounds__(TPB) void rotation_products_kernel(RotBatch rb, RotArgs a) {
    constexpr int PB = TPB / WG;  // positions per block
    const uint32_t groups = (a.count + RG - 1) / RG, chunks = (groups + WG - 1) / WG;
    const uint32_t xcd = blockIdx.x & 7, q8 = blockIdx.x >> 3;
    const uint32_t tile = (q8 / chunks) * 8 + xcd;
    if (tile >= a.tiles) return;
    const uint32_t group = (q8 % chunks) * WG + threadIdx.x / PB;
    const size_t flat = (size_t)tile * PB + threadIdx.x % PB;
    if (group >= groups || flat >= (size_t)(a.L + 1) << a.logn) return;
    const uint32_t i = uniform_row(flat, a.logn);
    const size_t c = flat & (((size_t)1 << a.logn) - 1);
    const uint32_t ct0 = group * RG;
    const int gv = (int)min<uint32_t>(RG, a.count - ct0);
    if constexpr (MIXED) {
        if (a.targets[i].fwd_fp) {  // uniform
            rotation_products_core<R, true>(rb, a, i, c, ct0, gv);
            return;
        }
    }
    rotation_products_core<R, false>(rb, a, i, c, ct0, gv);
}

// The products of nr rotations; the waves of a block share positions where there are
// groups enough for them.
void launch_rotation_products(const RotBatch &rb, RotArgs a, uint32_t nr, bool mixed, hipStream_t st) {
    const uint32_t groups = (a.count + RG - 1) / RG;
    uint32_t wg = a.logn < 6 || groups < 2 ? 1 : groups < 4 ? 2 : 4;
    uint64_t blocks;
    for (;; wg = 1) {
        a.tiles = (uint32_t)((((size_t)(a.L + 1) << a.logn) + TPB / wg - 1) / (TPB / wg));
        blocks = (uint64_t)((a.tiles + 7) / 8) * 8 * ((groups + wg - 1) / wg);
        if (wg == 1 || blocks * TPB < (uint64_t(1) << 32)) break;
    }
    if (blocks * TPB >= (uint64_t(1) << 32)) fail(ERR_INVALID_ARGUMENT, "rotation batch too large for one call");
    auto go = [&](auto r, auto w) {
        constexpr int R = decltype(r)::value, WG = decltype(w)::value;
        if (mixed) rotation_products_kernel<R, WG, true><<<(uint32_t)blocks, TPB, 0, st>>>(rb, a);
        else rotation_products_kernel<R, WG, false><<<(uint32_t)blocks, TPB, 0, st>>>(rb, a);
    };
    auto with_r = [&](auto w) {
        switch (nr) {
            case 1: go(std::integral_constant<int, 1>{}, w); break;
            case 2: go(std::integral_constant<int, 2>{}, w); break;
            case 3: go(std::integral_constant<int, 3>{}, w); break;
            default: go(std::integral_constant<int, 4>{}, w); break;
        }
    };
    switch (wg) {
        case 1: with_r(std::integral_constant<int, 1>{}); break;
        case 2: with_r(std::integral_constant<int, 2>{}); break;
        default: with_r(std::integral_constant<int, 4>{}); break;
    }
    launch_check("rotation_products");
}

// The sum over a pass's rotations of their permuted products, Psum[g] (+)= sum_q
// sigma_q(P_q[g]) for polynomials g < polys of L limbs, and of their rounded special limbs,
// V[g] (+)= sum_q [S_q[g] + floor(p/2)]_p as whole numbers (at most 15 of them below 2^60):
// what one ModDown needs for all of them.  HBM: reads each product once.
struct SumArgs {
    const uint64_t *P, *S;       // rotation q's at + q * polys limbs * L (1)
    uint64_t *Psum, *V;
    uint32_t elt[RMAX];
    uint64_t p;
};
__global__ void sum_products_kernel(SumArgs a, uint32_t nr, const DevPrime *__restrict__ primes, uint32_t L, int logn,
                                    uint32_t polys, bool first, size_t total) {
    const uint32_t n = 1u << logn;
    for (size_t idx = (size_t)blockIdx.x * TPB + threadIdx.x; idx < total; idx += (size_t)gridDim.x * TPB) {
        const uint32_t r = uniform_row(idx, logn), g = r / (L + 1), i = r - g * (L + 1);
        const uint32_t off = (uint32_t)(idx & (n - 1));
        if (i == L) {
            uint64_t v = first ? 0 : a.V[((size_t)g << logn) + off];
            for (uint32_t q = 0; q < nr; q++) {
                const uint64_t s = a.S[((size_t)(q * polys + g) << logn) + off] + (a.p >> 1);
                v += s >= a.p ? s - a.p : s;
            }
            a.V[((size_t)g << logn) + off] = v;
            continue;
        }
        const uint64_t q_i = primes[i].q;
        const size_t limb = (size_t)g * L + i;
        uint64_t v = first ? 0 : a.Psum[(limb << logn) + off];
        const uint32_t rev = __brev(n + off) >> (31 - logn);
        for (uint32_t q = 0; q < nr; q++) {
            const uint32_t src = __brev((a.elt[q] * rev >> 1) & (n - 1)) >> (32 - logn);
            v = addmod(v, a.P[(((size_t)q * polys * L + limb) << logn) + src], q_i);
        }
        a.Psum[(limb << logn) + off] = v;
    }
}

// out c0 = (first ? 0 : out c0) + s0, out c1 = first ? 0 : out c1; s0: [count][L][N].
__global__ void accumulate_c0_kernel(uint64_t *__restrict__ out, const uint64_t *__restrict__ s0,
                                     const DevPrime *__restrict__ primes, uint32_t L, int logn, bool first,
                                     size_t total) {
    const size_t lw = (size_t)L << logn;
    for (size_t idx = (size_t)blockIdx.x * TPB + threadIdx.x; idx < total; idx += (size_t)gridDim.x * TPB) {
        const size_t ct = idx / lw, r = idx % lw;
        uint64_t *c0 = out + ct * 2 * lw + r;
        const uint64_t v = s0[idx];
        if (first) {
            *c0 = v;
            c0[lw] = 0;
        } else {
            *c0 = addmod(*c0, v, primes[r >> logn].q);
        }
    }
}

__global__ void clear_flag_kernel(unsigned long long *flag) { *flag = 0; }

// A prepared key ends with two header words: HOISTED_TAG | L, and the Galois element.
constexpr uint64_t HOISTED_TAG = 0x484f4953ull << 32;  // "HOIS"
__global__ void write_hoisted_header_kernel(uint64_t *hdr, uint32_t L, uint32_t elt) {
    hdr[0] = HOISTED_TAG | L;
    hdr[1] = elt;
}

// flag |= 2 if a prepared key's header does not name level L and element elts[r].
constexpr int HDR_CHUNK = 16;
struct HeaderBatch {
    const uint64_t *hdr[HDR_CHUNK];
    uint32_t elt[HDR_CHUNK];
};
__global__ void check_hoisted_headers_kernel(HeaderBatch hb, uint32_t nr, uint32_t L, unsigned long long *flag) {
    const uint32_t r = threadIdx.x;
    if (r >= nr) return;
    if (hb.hdr[r][0] != (HOISTED_TAG | L) || hb.hdr[r][1] != hb.elt[r]) atomicOr(flag, 2ull);
}

// Zero digits of the batch: zc[0] counts them and entry e < zc[0] of `list` is
// (ct << 32) | (j << 24) | p; zc[2 + ct] counts ciphertext ct's (the list has room for
// every digit word, so it cannot overflow).
__global__ void zero_list_kernel(const uint64_t *__restrict__ digits, size_t dstride, uint32_t L, int logn,
                                 unsigned long long *__restrict__ zc, uint64_t *__restrict__ list, size_t total) {
    const size_t per_ct = (size_t)L << logn;
    for (size_t idx = (size_t)blockIdx.x * TPB + threadIdx.x; idx < total; idx += (size_t)gridDim.x * TPB) {
        const size_t ct = idx / per_ct, r = idx % per_ct;
        if (digits[ct * dstride + r] != 0) continue;
        const unsigned long long e = atomicAdd(zc, 1ull);
        atomicAdd(zc + 2 + ct, 1ull);
        list[e] = ((uint64_t)ct << 32) | ((uint64_t)(r >> logn) << 24) | (r & ((size_t(1) << logn) - 1));
    }
}

__global__ void clear_words_kernel(unsigned long long *w, size_t words) {
    for (size_t i = (size_t)blockIdx.x * TPB + threadIdx.x; i < words; i += (size_t)gridDim.x * TPB) w[i] = 0;
}

// The zero-digit fix of R rotations' products (before their permutations): at target
// i, slot s (one thread each),
//   P_r[ct][k][i][s] += sum over zeros (ct, j, p) that sigma_r negates, j's prime not i,
//                       of (q_j mod q_i) psi_i^((2 brev(s) + 1) p) key'_r[j][k][ki][s],
// psi_i^((2 brev(s)+1) p) being slot s of NTT_i(X^p); products of a ciphertext whose
// L N digit words are all zero are set to zero (its exact products; p c0 where that is
// folded in).  Exits at once
// when the batch has no zero digit.
template <int R>
__global__ __launch_bounds__(TPB) void zero_digit_fix_kernel(RotBatch rb, const unsigned long long *__restrict__ zc,
                                                             const uint64_t *__restrict__ list,
                                                             const DevPrime *__restrict__ targets,
                                                             const DevPrime *__restrict__ data, uint32_t L, uint32_t K,
                                                             int logn, uint32_t count, KsFold fold) {
    const unsigned long long z = zc[0];
    if (z == 0) return;
    const size_t n = (size_t)1 << logn;
    const size_t flat = (size_t)blockIdx.x * TPB + threadIdx.x;
    if (flat >= (size_t)(L + 1) << logn) return;
    const uint32_t i = (uint32_t)(flat >> logn);
    const uint32_t s = (uint32_t)(flat & (n - 1));
    const uint32_t ki = (i == L) ? K - 1 : i;
    const DevPrime &Q = targets[i];
    const uint64_t all = (uint64_t)L << logn;
    auto out = [&](int r, size_t ct, int k) -> uint64_t * {
        return i == L ? rb.S[r] + (ct * 2 + k) * n + s : rb.P[r] + ((ct * 2 + k) * L + i) * n + s;
    };
    for (uint32_t ct = 0; ct < count; ct++) {
        if (zc[2 + ct] != all) continue;
        const uint64_t pc0 = fold.ct && i < L ? mulmod(fold.ct[ct * fold.ct_stride + flat], fold.dc[i].p_mod, Q.q,
                                                       Q.ratio_lo, Q.ratio_hi)
                                              : 0;
#pragma unroll
        for (int r = 0; r < R; r++) {
            *out(r, ct, 0) = pc0;
            *out(r, ct, 1) = 0;
        }
    }
    const uint64_t two_bs1 = 2 * (uint64_t)(__brev(s) >> (32 - logn)) + 1;
    const size_t kstride = (size_t)K << logn;
    for (unsigned long long e = 0; e < z; e++) {
        const uint64_t w = list[e];
        const size_t ct = w >> 32;
        if (zc[2 + ct] == all) continue;
        const uint32_t j = (uint32_t)(w >> 24) & 0xff, p = (uint32_t)w & 0xffffff;
        if (j == i) continue;  // q_j mod q_j = 0
        const uint64_t qji = barrett64(data[j].q, Q.q, Q.ratio_hi);
        const uint64_t ex = (two_bs1 * p) & (2 * n - 1);
        const uint64_t m = ex & (n - 1);
        const uint64_t root = Q.fwd[__brev((uint32_t)m) >> (32 - logn)].x;
        const uint64_t psi = ex >= n ? Q.q - root : root;
        const uint64_t f = mulmod(qji, psi, Q.q, Q.ratio_lo, Q.ratio_hi);
#pragma unroll
        for (int r = 0; r < R; r++) {
            if (((((uint64_t)p * rb.elt[r]) >> logn) & 1) == 0) continue;  // sigma_r keeps p's sign
            const uint64_t *kp = rb.key[r] + (size_t)ki * n + s;
#pragma unroll
            for (int k = 0; k < 2; k++) {
                const uint64_t t = mulmod(f, kp[(2 * (size_t)j + k) * kstride], Q.q, Q.ratio_lo, Q.ratio_hi);
                uint64_t *o = out(r, ct, k);
                *o = addmod(*o, t, Q.q);
            }
        }
    }
}

void check_level(const Context &c, uint32_t L) {
    if (c.key_count() < 2) fail(ERR_LOGIC, "keyswitching is not supported by the context");
    if (L < 1 || L > c.key_count() - 1) fail(ERR_INVALID_ARGUMENT, "level out of range for key switching");
}

}  // namespace

size_t hoisted_key_words(const Context &c, uint32_t L) {
    const size_t K = c.key_count();
    return ((K - 1) * 2 * K + 2 * ((size_t)L + 1)) * c.n + 2;
}

size_t hoisted_key_workspace(const Context &c, uint32_t L) { return 3 * ((size_t)L + 1) * c.n * 8; }

void hoisted_key_prepare(const Context &c, const uint64_t *galois_key, uint32_t elt, uint32_t L, uint64_t *out,
                         void *ws, size_t ws_bytes, hipStream_t st) {
    check_level(c, L);
    const uint64_t m = 2 * c.n;
    if (!(elt & 1) || elt >= m) fail(ERR_INVALID_ARGUMENT, "Galois element is not valid");
    if (!ws || ws_bytes < hoisted_key_workspace(c, L)) fail(ERR_INVALID_ARGUMENT, "workspace too small");
    const uint32_t K = (uint32_t)c.key_count();
    const size_t n = c.n;
    const uint32_t elt_inv = (uint32_t)hm::invmod(elt, m);
    // key' = sigma^-1(key), limb by limb
    apply_galois(c, galois_key, K * n, out, K * n, (K - 1) * 2, K, elt_inv, true, st);
    // corr' = sigma^-1(NTT_i(S_sigma) * sum_j (q_j mod q_i) key_j[i])
    uint64_t *neg = static_cast<uint64_t *>(ws);
    uint64_t *C = neg + ((size_t)L + 1) * n;
    const size_t nw = ((size_t)L + 1) * n;
    negated_positions_kernel<<<blocks_for(nw), TPB, 0, st>>>(neg, elt, elt_inv, c.logn, nw);
    launch_check("negated_positions");
    const DevPrime *targets = c.keyswitch_primes(L);
    ntt_forward_grid(neg, LimbGrid{1, L + 1, L + 1, 1}, targets, c.logn, NTT_FULL, st);
    correction_kernel<<<blocks_for(2 * nw), TPB, 0, st>>>(neg, galois_key, C, targets, c.primes(), L, K, c.logn,
                                                          2 * nw);
    launch_check("correction");
    apply_galois(c, C, nw, out + (size_t)(K - 1) * 2 * K * n, nw, 2, L + 1, elt_inv, true, st);
    write_hoisted_header_kernel<<<1, 1, 0, st>>>(out + hoisted_key_words(c, L) - 2, L, elt);
    launch_check("hoisted key header");
    std::lock_guard<std::mutex> g(c.hoisted_mu);
    c.hoisted_keys[out] = {L, elt};
}

size_t rotate_sum_workspace(const Context &c, uint32_t count, uint32_t L) { return rot_layout(c.logn, count, L).total; }

namespace {

// The hoisted rotations of `in`, summed into out (sum) or each into its own
// out + r * count * 2L N (!sum).
void rotate_hoisted(const Context &c, const uint64_t *in, uint32_t count, uint32_t L, const uint32_t *elts,
                    const uint64_t *const *hoisted, const uint64_t *const *keys, uint32_t rotations, uint64_t *out,
                    void *ws, size_t ws_bytes, hipStream_t st, bool sum) {
    check_level(c, L);
    if (!count) return;
    if (!rotations || !elts || !hoisted || !keys) fail(ERR_INVALID_ARGUMENT, "no rotations given");
    KernelProbe probe{nullptr, nullptr};
    const bool armed = c.take_probe(probe);  // brackets the first pass of hoisted products
    const RotLayout lay = rot_layout(c.logn, count, L);
    if (!ws || ws_bytes < lay.total) fail(ERR_INVALID_ARGUMENT, "workspace too small for rotation sums");
    if (in == out) fail(ERR_INVALID_ARGUMENT, "rotate_sum cannot run in place");
    const uint64_t max_cts = ((uint64_t(1) << 34) >> c.logn) / ((uint64_t)L * (L + 1));
    if ((uint64_t)count > max_cts) fail(ERR_INVALID_ARGUMENT, "rotation batch too large for one call");
    const bool ckks = c.scheme == SCHEME_CKKS;
    const int logn = c.logn;
    const size_t n = c.n, lw = (size_t)L * n;
    char *base = static_cast<char *>(ws);
    auto at = [base](size_t off) { return reinterpret_cast<uint64_t *>(base + off); };
    uint64_t *T = at(lay.T), *list = at(lay.list), *U = at(sum ? lay.U_sum : lay.U), *S2 = at(lay.S2);
    uint64_t *c_limbs = at(lay.c);  // CKKS: the digits; BFV, N >= 2^13: c0 in NTT form
    uint64_t *Pm = at(lay.Pm), *Sm = at(sum ? lay.Sm_sum : lay.Sm);
    auto *flag = reinterpret_cast<unsigned long long *>(base + lay.flag);

    // each prepared key must be the one of this level and element: checked on the
    // host for keys prepared through this context; other keys' header words are read
    // back from the device (the only case that waits for the stream)
    const size_t hdr_off = hoisted_key_words(c, L) - 2;
    std::vector<uint32_t> unknown;
    {
        std::lock_guard<std::mutex> g(c.hoisted_mu);
        for (uint32_t r = 0; r < rotations; r++) {
            if (!hoisted[r] || !keys[r]) fail(ERR_INVALID_ARGUMENT, "null key pointer");
            auto it = c.hoisted_keys.find(hoisted[r]);
            if (it == c.hoisted_keys.end()) unknown.push_back(r);
            else if (it->second.first != L || it->second.second != elts[r])
                fail(ERR_INVALID_ARGUMENT, "a hoisted key was prepared for another level or Galois element");
        }
    }
    if (!unknown.empty()) {
        clear_flag_kernel<<<1, 1, 0, st>>>(flag);
        for (size_t r0 = 0; r0 < unknown.size(); r0 += HDR_CHUNK) {
            HeaderBatch hb{};
            const uint32_t nr = (uint32_t)std::min<size_t>(unknown.size() - r0, HDR_CHUNK);
            for (uint32_t q = 0; q < nr; q++) {
                hb.hdr[q] = hoisted[unknown[r0 + q]] + hdr_off;
                hb.elt[q] = elts[unknown[r0 + q]];
            }
            check_hoisted_headers_kernel<<<1, 64, 0, st>>>(hb, nr, L, flag);
            launch_check("hoisted key headers");
        }
        unsigned long long flags = 0;
        SHC_HIP(hipMemcpyAsync(&flags, flag, 8, hipMemcpyDeviceToHost, st));
        SHC_HIP(hipStreamSynchronize(st));
        if (flags & 2)
            fail(ERR_INVALID_ARGUMENT, "a hoisted key was prepared for another level or Galois element");
    }
    // 1. digits of c1 in coefficient form (CKKS: transformed into the workspace; c1 itself, in NTT
    // form, supplies the own-prime terms of the products)
    const uint64_t *digits = in + lw;
    size_t dstride = 2 * lw;
    if (ckks) {
        ntt_inverse_from(in + lw, LimbGrid{1, 2 * L, L, count}, c_limbs, LimbGrid{1, L, L, count}, c.primes(), logn,
                         NTT_FULL, st);
        digits = c_limbs;
        dstride = lw;
    }
    // 2. zero digits, listed for the products' fix (the list has room for every word)
    auto *zc = reinterpret_cast<unsigned long long *>(base + lay.zc);
    clear_words_kernel<<<1, TPB, 0, st>>>(zc, 2 + (size_t)count);
    zero_list_kernel<<<blocks_for(count * lw), TPB, 0, st>>>(digits, dstride, L, logn, zc, list, count * lw);
    launch_check("zero digits");
    const size_t ct_words = (size_t)count * 2 * lw;
    // 3. one ModUp for every rotation
    const bool skipped = modup_to_T(c, digits, dstride, T, count, L, st, nullptr, ckks);
    // T words below 4 q_i where the fp64 transforms (N >= 2^13) or full reduction made them
    const bool acc26 = c.fp_primes;
    const uint64_t *diag = skipped ? in + lw : nullptr;
    const DevPrime *targets = c.keyswitch_primes(L);
    const size_t K = c.key_count();
    const size_t corr_off = (K - 1) * 2 * K * n;
    // N >= 2^13: c0 joins the products (in NTT form: BFV's c0 is transformed once for all
    // rotations), the products are permuted as the ModDown reads them, and a pass's
    // rotations -- or, when summing, up to 15 of them -- take one ModDown
    KsFold fold{};
    if (lay.batched) {
        fold = KsFold{in, 2 * lw, c.ks_consts()};
        if (!ckks) {
            const NttGroup g{c_limbs, in, LimbGrid{1, L, L, count}, LimbGrid{1, 2 * L, L, count}, c.primes()};
            ntt_forward_groups(&g, 1, logn, NTT_FULL, st);
            fold = KsFold{c_limbs, lw, c.ks_consts()};
        }
    }
    const RotArgs args{T, corr_off, targets, L, (uint32_t)K, logn, count, 0, diag, 2 * lw, fold};
    // rotations per pass: RMAX, fewer where one launch cannot hold their limbs
    uint32_t pass = RMAX;
    while (lay.batched && pass > 1 && (uint64_t)pass * count * 2 * L > ((uint64_t(1) << 34) >> logn)) pass--;
    const uint64_t p = c.moduli[K - 1];
    uint32_t summed = 0;  // rotations in Psum, V
    for (uint32_t r0 = 0; r0 < rotations; r0 += pass) {
        const uint32_t nr = std::min(rotations - r0, pass);
        // products with the prepared keys (corrections included), RMAX rotations per pass over T
        RotBatch rb{};
        for (uint32_t q = 0; q < nr; q++) {
            rb.key[q] = hoisted[r0 + q];
            rb.P[q] = Pm + (size_t)q * count * 2 * lw;
            rb.S[q] = Sm + (size_t)q * count * 2 * n;
            rb.elt[q] = elts[r0 + q];
        }
        if (armed && r0 == 0) SHC_HIP(hipEventRecord(probe.begin, st));
        launch_rotation_products(rb, args, nr, acc26, st);
        if (armed && r0 == 0) SHC_HIP(hipEventRecord(probe.end, st));
        const uint32_t fix_blocks = (uint32_t)((((size_t)(L + 1) << logn) + TPB - 1) / TPB);
        switch (nr) {
            case 1: zero_digit_fix_kernel<1><<<fix_blocks, TPB, 0, st>>>(rb, zc, list, targets, c.primes(), L, (uint32_t)K, logn, count, fold); break;
            case 2: zero_digit_fix_kernel<2><<<fix_blocks, TPB, 0, st>>>(rb, zc, list, targets, c.primes(), L, (uint32_t)K, logn, count, fold); break;
            case 3: zero_digit_fix_kernel<3><<<fix_blocks, TPB, 0, st>>>(rb, zc, list, targets, c.primes(), L, (uint32_t)K, logn, count, fold); break;
            default: zero_digit_fix_kernel<4><<<fix_blocks, TPB, 0, st>>>(rb, zc, list, targets, c.primes(), L, (uint32_t)K, logn, count, fold); break;
        }
        launch_check("zero_digit_fix");
        if (!lay.batched) {
            uint64_t *C0 = at(lay.C0), *P2 = at(lay.P2);
            for (uint32_t q = 0; q < nr; q++) {
                const uint32_t r = r0 + q;
                uint64_t *dst = sum ? out : out + r * ct_words;
                // (sigma(c0), 0) into dst (accumulated when summing)
                apply_galois(c, in, 2 * lw, C0, lw, count, L, elts[r], ckks, st);
                accumulate_c0_kernel<<<blocks_for(count * lw), TPB, 0, st>>>(dst, C0, c.primes(), L, logn,
                                                                             !sum || r == 0, count * lw);
                launch_check("accumulate_c0");
                // the products permuted by sigma, then this rotation's ModDown added into dst
                apply_galois(c, rb.P[q], lw, P2, lw, count * 2, L, elts[r], true, st);
                apply_galois(c, rb.S[q], n, S2, n, count * 2, 1, elts[r], true, st);
                moddown_into(c, P2, S2, U, dst, 2 * lw, count, L, st);
            }
            continue;
        }
        GaloisPerm perm{2 * count, {}};
        for (uint32_t q = 0; q < nr; q++) {
            if (!(elts[r0 + q] & 1) || elts[r0 + q] >= 2 * n) fail(ERR_INVALID_ARGUMENT, "Galois element is not valid");
            perm.elt[q] = elts[r0 + q];
        }
        const uint32_t polys = 2 * count * nr;
        ntt_inverse_galois(Sm, LimbGrid{1, 1, 1, polys}, perm, S2, LimbGrid{1, 1, 1, polys}, targets + L, logn, st);
        ModDownArgs md{S2, Pm, out + r0 * ct_words, 2 * lw, c.ks_consts(), p, L, true};
        if (!sum) {
            md.perm = perm;
            ntt_moddown(ckks, U, md, count * nr, c.primes(), logn, st);
            continue;
        }
        uint64_t *Psum = at(lay.Psum), *V = at(lay.V);
        SumArgs sa{Pm, S2, Psum, V, {}, p};
        for (uint32_t q = 0; q < nr; q++) sa.elt[q] = elts[r0 + q];
        const size_t total = (size_t)2 * count * (L + 1) * n;
        sum_products_kernel<<<blocks_for(total), TPB, 0, st>>>(sa, nr, c.primes(), L, logn, 2 * count, summed == 0, total);
        launch_check("sum_products");
        summed += nr;
        const uint32_t next = std::min(rotations - (r0 + nr), pass);
        if (!next || summed + next > SUM_MAX) {
            md.S = V;
            md.P = Psum;
            md.ct = out;
            md.folded = r0 + nr == summed;  // the first sums write out, later ones add
            md.presum = summed;
            ntt_moddown(ckks, ckks ? U : Psum, md, count, c.primes(), logn, st);
            summed = 0;
        }
    }
}

}  // namespace

void rotate_sum(const Context &c, const uint64_t *in, uint32_t count, uint32_t L, const uint32_t *elts,
                const uint64_t *const *hoisted, const uint64_t *const *keys, uint32_t rotations, uint64_t *out,
                void *ws, size_t ws_bytes, hipStream_t st) {
    rotate_hoisted(c, in, count, L, elts, hoisted, keys, rotations, out, ws, ws_bytes, st, true);
}

void rotate_many(const Context &c, const uint64_t *in, uint32_t count, uint32_t L, const uint32_t *elts,
                 const uint64_t *const *hoisted, const uint64_t *const *keys, uint32_t rotations, uint64_t *out,
                 void *ws, size_t ws_bytes, hipStream_t st) {
    rotate_hoisted(c, in, count, L, elts, hoisted, keys, rotations, out, ws, ws_bytes, st, false);
}

// ---- sums of rotations of different ciphertexts --------------------------------------
namespace {

// The c0 part of a rotation sum, and the ciphertexts that stay as they are:
//   out[ct][0] (+)= sum_h sigma_h(in[h][ct][0]),  out[ct][1] (+)= sum_{h: elt 1} in[h][ct][1]
constexpr uint32_t C0_MAX = 16;
struct SumC0Args {
    const uint64_t *in;   // [n][count][2][L][N]
    uint64_t *out;        // [count][2][L][N]
    uint32_t elt[C0_MAX], elt_inv[C0_MAX];
    uint32_t n, count, L;
    int logn;
    bool first;
};
template <bool NTT>
__global__ void sum_c0_kernel(SumC0Args a, const DevPrime *__restrict__ primes, size_t total) {
    const uint32_t n = 1u << a.logn;
    const size_t lw = (size_t)a.L << a.logn, ctw = 2 * lw;
    for (size_t idx = (size_t)blockIdx.x * TPB + threadIdx.x; idx < total; idx += (size_t)gridDim.x * TPB) {
        const uint32_t r = uniform_row(idx, a.logn), ct = r / a.L, i = r - ct * a.L;
        const uint32_t off = (uint32_t)(idx & (n - 1));
        const uint64_t q = primes[i].q;
        const size_t limb = (size_t)ct * ctw + ((size_t)i << a.logn);
        uint64_t v0 = a.first ? 0 : a.out[limb + off], v1 = a.first ? 0 : a.out[limb + lw + off];
        for (uint32_t h = 0; h < a.n; h++) {
            const uint64_t *src = a.in + (size_t)h * a.count * ctw + limb;
            const uint32_t e = a.elt[h];
            uint64_t x;
            if constexpr (NTT) {
                x = src[galois_slot(off, e, a.logn)];
            } else {
                const uint32_t k = (uint32_t)(((uint64_t)off * a.elt_inv[h]) & (n - 1));
                x = src[k];
                if (((uint64_t)k * e >> a.logn) & 1) x = negmod(x, q);
            }
            v0 = addmod(v0, x, q);
            if (e == 1) v1 = addmod(v1, src[lw + off], q);
        }
        a.out[limb + off] = v0;
        a.out[limb + lw + off] = v1;
    }
}

// d[h][ct][i] = sigma_h(in[h][ct][1][i]) in coefficient form, h < n (at most PERM_MAX).
__global__ void galois_digits_kernel(SumC0Args a, uint64_t *__restrict__ d, const DevPrime *__restrict__ primes,
                                     size_t total) {
    const uint32_t n = 1u << a.logn;
    for (size_t idx = (size_t)blockIdx.x * TPB + threadIdx.x; idx < total; idx += (size_t)gridDim.x * TPB) {
        const uint32_t r = uniform_row(idx, a.logn), g = r / a.L, i = r - g * a.L, h = g / a.count;
        const uint32_t off = (uint32_t)(idx & (n - 1));
        const uint32_t k = (uint32_t)(((uint64_t)off * a.elt_inv[h]) & (n - 1));
        uint64_t x = a.in[((((size_t)g * 2 + 1) * a.L + i) << a.logn) + k];
        if (((uint64_t)k * a.elt[h] >> a.logn) & 1) x = negmod(x, primes[i].q);
        d[idx] = x;
    }
}

}  // namespace

size_t rotate_accumulate_workspace(const Context &c, uint32_t count, uint32_t L) {
    return acc_workspace(c.logn, count, L);
}

void rotate_accumulate(const Context &c, const uint64_t *in, uint32_t count, uint32_t L, const uint32_t *elts,
                       const uint64_t *const *keys, uint32_t n, uint64_t *out, void *ws, size_t ws_bytes,
                       hipStream_t st) {
    check_level(c, L);
    if (!count) return;
    if (!n || !elts || !keys) fail(ERR_INVALID_ARGUMENT, "no rotations given");
    const uint32_t most_nb = ws ? acc_rotations(c.logn, count, L, ws_bytes) : 0;
    if (!most_nb) fail(ERR_INVALID_ARGUMENT, "workspace too small for rotation sums");
    const AccLayout lay = acc_layout(c.logn, count, L, most_nb);
    const size_t N = c.n, lw = (size_t)L * N, ctw = 2 * lw, step = (size_t)count * ctw;
    // (the sums are written while later ciphertexts' permuted words are still to be read)
    if (out < in + n * step && in < out + step) fail(ERR_INVALID_ARGUMENT, "rotate_accumulate cannot run in place");
    for (uint32_t h = 0; h < n; h++) {
        if (!(elts[h] & 1) || elts[h] >= 2 * N) fail(ERR_INVALID_ARGUMENT, "Galois element is not valid");
        if (elts[h] != 1 && !keys[h]) fail(ERR_INVALID_ARGUMENT, "null key pointer");
    }
    char *base = static_cast<char *>(ws);
    auto at = [base](size_t off) { return reinterpret_cast<uint64_t *>(base + off); };
    const bool ckks = c.scheme == SCHEME_CKKS;
    const int logn = c.logn;
    if (!lay.batched) {
        // (sigma(c0), 0) joins the sum, and the switch of sigma(c1) adds into it
        uint64_t *sigma = at(lay.d), *C0 = at(lay.C0);
        for (uint32_t h = 0; h < n; h++) {
            const uint64_t *x = in + h * step;
            if (elts[h] == 1) {
                if (h) poly_add(c, out, x, out, count * 2, L, st);
                else SHC_HIP(hipMemcpyAsync(out, x, step * 8, hipMemcpyDeviceToDevice, st));
                continue;
            }
            apply_galois(c, x + lw, ctw, sigma, lw, count, L, elts[h], ckks, st);
            apply_galois(c, x, ctw, C0, lw, count, L, elts[h], ckks, st);
            accumulate_c0_kernel<<<blocks_for(count * lw), TPB, 0, st>>>(out, C0, c.primes(), L, logn, h == 0, count * lw);
            launch_check("accumulate_c0");
            switch_key(c, sigma, lw, out, ctw, keys[h], count, L, base + lay.ks, lay.total - lay.ks, st);
        }
        return;
    }
    SumC0Args ca{in, out, {}, {}, 0, count, L, logn, true};
    for (uint32_t h0 = 0; h0 < n; h0 += C0_MAX) {
        ca.in = in + h0 * step;
        ca.n = std::min(n - h0, C0_MAX);
        ca.first = h0 == 0;
        for (uint32_t h = 0; h < ca.n; h++) {
            ca.elt[h] = elts[h0 + h];
            ca.elt_inv[h] = (uint32_t)hm::invmod(elts[h0 + h], 2 * N);
        }
        const size_t total = (size_t)count * lw;
        if (ckks) sum_c0_kernel<true><<<blocks_for(total), TPB, 0, st>>>(ca, c.primes(), total);
        else sum_c0_kernel<false><<<blocks_for(total), TPB, 0, st>>>(ca, c.primes(), total);
        launch_check("sum_c0");
    }
    const DevPrime *targets = c.keyswitch_primes(L);
    const uint32_t K = (uint32_t)c.key_count();
    uint64_t *d = at(lay.d), *T = at(lay.T), *P = at(lay.P), *S = at(lay.S), *Psum = at(lay.Psum), *V = at(lay.V);
    uint32_t summed = 0, left = 0;  // key switches in Psum, V; and still to come
    for (uint32_t h = 0; h < n; h++) left += elts[h] != 1;
    for (uint32_t h0 = 0; h0 < n;) {
        if (elts[h0] == 1) {
            h0++;
            continue;
        }
        uint32_t nb = 1;  // consecutive switches, at most a summed ModDown's 15 in all
        while (nb < most_nb && h0 + nb < n && elts[h0 + nb] != 1 && summed + nb < SUM_MAX) nb++;
        const uint64_t *x = in + h0 * step;
        GaloisPerm perm{count, {}};
        InnerKeys ik{};
        ik.n = nb;
        ik.per = count;
        SumC0Args ga{x, nullptr, {}, {}, nb, count, L, logn, true};
        for (uint32_t h = 0; h < nb; h++) {
            perm.elt[h] = ga.elt[h] = ik.elt[h] = elts[h0 + h];
            ga.elt_inv[h] = (uint32_t)hm::invmod(elts[h0 + h], 2 * N);
            ik.key[h] = keys[h0 + h];
        }
        // digits of sigma(c1): CKKS through the permutation on load (c1 itself, permuted on
        // load, supplies the own-prime terms), BFV permuted in coefficient form
        if (ckks) {
            ntt_inverse_galois(x + lw, LimbGrid{1, 2 * L, L, nb * count}, perm, d, LimbGrid{1, L, L, nb * count},
                               c.primes(), logn, st);
        } else {
            const size_t total = (size_t)nb * count * lw;
            galois_digits_kernel<<<blocks_for(total), TPB, 0, st>>>(ga, d, c.primes(), total);
            launch_check("galois_digits");
        }
        if (acc_fused(logn)) {
            for (uint32_t h = 0; h < nb; h++)
                ntt_modup_keyprod(d + h * count * lw, lw, T, ik.key[h], P + h * step, S + (size_t)h * count * 2 * N,
                                  ckks ? x + h * step + lw : nullptr, ctw, count, L, K, targets, c.primes(), logn,
                                  c.fp_primes, st, nullptr, c.ks_shape(L, count),
                                  KsFold{nullptr, 0, nullptr, false, ik.elt[h]});
        } else {
            const bool skipped = modup_to_T(c, d, lw, T, nb * count, L, st, nullptr, ckks);
            keyswitch_inner_products(c, T, ik, P, S, L, st, skipped ? x + lw : nullptr, ctw);
        }
        ntt_inverse(S, nb * count * 2, 1, targets + L, logn, NTT_FULL, st);
        const SumArgs sa{P, S, Psum, V, {1, 1, 1, 1}, c.moduli[K - 1]};
        const size_t total = (size_t)2 * count * (L + 1) * N;
        sum_products_kernel<<<blocks_for(total), TPB, 0, st>>>(sa, nb, c.primes(), L, logn, 2 * count, summed == 0, total);
        launch_check("sum_products");
        summed += nb;
        left -= nb;
        h0 += nb;
        if (summed == SUM_MAX || !left) {
            ModDownArgs md{V, Psum, out, ctw, c.ks_consts(), c.moduli[K - 1], L, false};
            md.presum = summed;
            ntt_moddown(ckks, ckks ? at(lay.U) : Psum, md, count, c.primes(), logn, st);
            summed = 0;
        }
    }
}

}  // namespace shc

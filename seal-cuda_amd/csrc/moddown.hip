// moddown.hip -- the ModDown / rescale correction and CKKS encryption fused into their
// transforms (N = 2^13 .. 2^17; the passes are those of ntt_device.h).
#include "ntt_device.h"

namespace shc {
namespace {

// ---- ModDown by the special prime p, fused into the transforms (switch_key step 5):
//   u_i = ([s + floor(p/2)]_p mod q_i) - (floor(p/2) mod q_i)     (s: special limb, coeff)
//   ct_k[i] += (P_k[i] - u_i) * p^-1 mod q_i
// CKKS runs it as the forward NTT of u (first pass computes u from s on load, last pass
// adds into ct on store); BFV as the inverse NTT of P (last pass subtracts u and adds).
// Limb (i, j): prime i < L, j = 2 ct + k.
__device__ __forceinline__ uint64_t moddown_prep(uint64_t s, uint64_t p, const DevPrime &Q, const DivRoundConst &d) {
    uint64_t v = s + (p >> 1);
    v = v >= p ? v - p : v;
    return submod(barrett64(v, Q.q, Q.ratio_hi), d.half_mod, Q.q);
}

// f(u) with u(i, s) = u_i of a ModDown at word s of its special limbs, for a limb of its own or a
// sum of them (15 floor(p/2) mod q_i < 2^64).  The branch is one per block: inside a pass's load
// it kept a thread's 16 loads from going out together (1,452 -> 1,695 us for 256 limbs of 2^16 to
// 23 primes), inside its store the special limbs' (26.6 -> 29.8 us for 16 limbs of 2^17, BFV).
template <class F>
__device__ __forceinline__ void with_moddown_u(const ModDownArgs &a, const DevPrime *__restrict__ primes, const F &f) {
    if (a.presum)
        f([&](uint32_t i, uint64_t s) {
            const DevPrime &Q = primes[i];
            return submod(barrett64(s, Q.q, Q.ratio_hi), barrett64(a.presum * a.dc[i].half_mod, Q.q, Q.ratio_hi), Q.q);
        });
    else
        f([&](uint32_t i, uint64_t s) { return moddown_prep(s, a.p, primes[i], a.dc[i]); });
}

// Word (limb i of polynomial j, coefficient off) of a ModDown's P.
template <int LOGN>
__device__ __forceinline__ uint64_t moddown_p(const ModDownArgs &a, uint32_t i, uint32_t j, size_t off) {
    if (a.perm.polys) off = galois_slot((uint32_t)off, a.perm.elt[j / a.perm.polys], LOGN);  // uniform
    if (a.p_lpp)  // uniform
        return a.P[(size_t)(j >> 1) * a.p_ct_stride + ((size_t)((j & 1) * a.p_lpp + i) << LOGN) + off];
    return a.P[((size_t)(j * a.L + i) << LOGN) + off];
}

template <int LOGN>
__device__ __forceinline__ void moddown_add(const ModDownArgs &a, uint32_t i, uint32_t j, size_t off, uint64_t pv,
                                            uint64_t u, const DevPrime &Q) {
    uint64_t *dst = a.ct + (size_t)(j >> 1) * a.ct_stride + ((size_t)((j & 1) * a.L + i) << LOGN) + off;
    const uint64_t v = shoup(submod(pv, u, Q.q), a.dc[i].inv, a.dc[i].inv_shoup, Q.q);
    if (a.folded) *dst = v;  // uniform: the ciphertext's words are already in P
    else *dst = addmod(*dst, v, Q.q);
}

// Columns pass of u_i = the rounded special limb's residue, on load.  Every prime reads the same
// special limb: i fastest keeps it in L2.
template <int LOGN, int K, int E, int SUBS>
__device__ __forceinline__ void cols_moddown_prep(uint64_t *tile, uint32_t bid, uint64_t *__restrict__ U,
                                                  const DevPrime *__restrict__ primes, const ModDownArgs &a,
                                                  uint32_t jn) {
    with_moddown_u(a, primes, [&](const auto &u) {
        cols_body_t<LOGN, K, E, SUBS, false, true>(
            tile, bid, primes, 0, jn,
            [&](uint32_t i, uint32_t j, size_t off) { return u(i, a.S[((size_t)j << LOGN) + off]); },
            [&](uint32_t i, uint32_t j, size_t off, uint64_t x) { U[((size_t)(j * a.L + i) << LOGN) + off] = x; }, a.L);
    });
}

template <int LOGN, int K, int E, int SUBS>
__global__ __launch_bounds__(SUBS << (K - E)) void ntt_cols_moddown_prep_kernel(uint64_t *__restrict__ U,
                                                                               const DevPrime *__restrict__ primes,
                                                                               ModDownArgs a, uint32_t jn) {
    __shared__ uint64_t tile[SUBS << K];
    cols_moddown_prep<LOGN, K, E, SUBS>(tile, blockIdx.x, U, primes, a, jn);
}

template <int LOGN, int K, int E, int SUBS, bool MX>
__global__ __launch_bounds__(SUBS << (K - E)) void ntt_rows_moddown_kernel(const uint64_t *__restrict__ U,
                                                                          const DevPrime *__restrict__ primes,
                                                                          ModDownArgs a, uint32_t jn) {
    rows_body<LOGN, K, E, SUBS, false, false, MX>(
        blockIdx.x, primes, a.L, 0, jn, [&](uint32_t i, uint32_t j, size_t off) { return U[((size_t)(j * a.L + i) << LOGN) + off]; },
        [&](uint32_t i, uint32_t j, size_t off, uint64_t x) {
            const DevPrime &Q = primes[i];
            moddown_add<LOGN>(a, i, j, off, moddown_p<LOGN>(a, i, j, off), finish<false, true>(x, Q), Q);
        });
}

// ---- CKKS public-key encryption fused into the error term's forward transform ----
__device__ __forceinline__ uint64_t enc_lift(int64_t v, uint64_t q) { return v < 0 ? q - (uint64_t)(-v) : (uint64_t)v; }

// Columns pass of the transforms of signed bytes: every prime of polynomial j reads the same
// bytes (i fastest), lifted on load.
template <int LOGN, int K, int E, int SUBS>
__global__ __launch_bounds__(SUBS << (K - E)) void ntt_cols_small_kernel(const int8_t *__restrict__ Us,
                                                                        uint64_t *__restrict__ U,
                                                                        const DevPrime *__restrict__ primes,
                                                                        uint32_t L1, uint32_t m) {
    cols_body<LOGN, K, E, SUBS, false, true>(
        blockIdx.x, primes, 0, m,
        [&](uint32_t i, uint32_t j, size_t off) { return enc_lift(Us[((size_t)j << LOGN) + off], primes[i].q); },
        [&](uint32_t i, uint32_t j, size_t off, uint64_t x) { U[((size_t)(j * L1 + i) << LOGN) + off] = x; }, L1);
}

template <int LOGN, bool SMALL>
void launch_small_as(const int8_t *Us, uint64_t *U, uint32_t L1, uint32_t m, uint32_t rows_from,
                     const DevPrime *primes, hipStream_t st) {
    using S = PassShape<LOGN, SMALL>;
    constexpr int K1 = S::K1, K2 = S::K2, E = S::E, CS = S::CS, RS = S::RS;
    const bool mx = rows_mixed<LOGN, K2, RS>(m);
    const uint32_t rows = L1 - rows_from;  // primes whose rows pass runs
    const uint32_t row_blocks = rows * rows_blocks_per_prime<LOGN, K2, E, RS>(m, mx);
    ntt_cols_small_kernel<LOGN, K1, E, CS><<<L1 * m * ((1u << K2) / CS), CS << (K1 - E), 0, st>>>(Us, U, primes, L1, m);
    if (!rows) return;
    const LimbGrid lg{1, L1, rows, m};
    with_bool(mx, [&](auto x) {
        ntt_rows_kernel<LOGN, K2, E, RS, false, true, true, decltype(x)::value><<<row_blocks, RS << (K2 - E), 0, st>>>(
            U + ((size_t)rows_from << LOGN), primes + rows_from, lg, 0, m);
    });
}

template <int LOGN, int K, int E, int SUBS>
__global__ __launch_bounds__(SUBS << (K - E)) void ntt_cols_encrypt_kernel(const DevPrime *__restrict__ primes,
                                                                          EncArgs a, uint32_t jn) {
    // every prime of polynomial j reads the same error and last-limb words: i fastest
    cols_body<LOGN, K, E, SUBS, false, true>(
        blockIdx.x, primes, 0, jn,
        [&](uint32_t i, uint32_t j, size_t off) {
            const DevPrime &Q = primes[i];
            const size_t w = ((size_t)j << LOGN) + off;
            const int64_t e = a.Es[w];
            uint64_t x = enc_lift(e, Q.q);
            if (a.drop) x = submod(x, moddown_prep(addmod(a.Pl[w], enc_lift(e, a.p), a.p), a.p, Q, a.dc[i]), Q.q);
            return x;
        },
        [&](uint32_t i, uint32_t j, size_t off, uint64_t x) { a.out[((size_t)(j * a.L + i) << LOGN) + off] = x; },
        a.L);
}

template <int LOGN, int K, int E, int SUBS, bool MX>
__global__ __launch_bounds__(SUBS << (K - E)) void ntt_rows_encrypt_kernel(const DevPrime *__restrict__ primes,
                                                                          EncArgs a, uint32_t jn) {
    rows_body<LOGN, K, E, SUBS, false, false, MX>(
        blockIdx.x, primes, a.L, 0, jn,
        [&](uint32_t i, uint32_t j, size_t off) { return a.out[((size_t)(j * a.L + i) << LOGN) + off]; },
        [&](uint32_t i, uint32_t j, size_t off, uint64_t x) {
            const DevPrime &Q = primes[i];
            const uint32_t g = j >> 1, k = j & 1;
            const uint64_t pu = mulmod(a.pk[((size_t)(k * a.K + i) << LOGN) + off],
                                       a.U[((size_t)(g * a.L1 + i) << LOGN) + off], Q.q, Q.ratio_lo, Q.ratio_hi);
            uint64_t v = addmod(pu, finish<false, true>(x, Q), Q.q);
            if (a.drop) v = shoup(v, a.dc[i].inv, a.dc[i].inv_shoup, Q.q);
            if (a.plain && k == 0) v = addmod(v, a.plain[((size_t)(g * a.L + i) << LOGN) + off], Q.q);
            a.out[((size_t)(j * a.L + i) << LOGN) + off] = v;
        });
}

// The rows pass for batches: a block owns row g of prime i for SUBS ciphertexts and runs the
// rows of their u, e0 and e1 one after another, so that NTT(u) stays in registers (16 words per
// thread) instead of in memory, and the public key's words -- a thread's position is the same
// in every ciphertext -- get Shoup constants once per block: their quotients come from
// floor(2^128 / q), at most 1 short, which leaves the products in [0, 5q) (q < 2^60; with the
// transform's [0, 8q) they fit a word).  128 ciphertexts at N = 2^16, L = 24: u's rows pass
// 0.78 + e's 3.87 ms -> 3.46 in all, still VALU issue (24 layers and 3 products per word).
template <int LOGN, int K, int E, int SUBS>
__global__ __launch_bounds__(SUBS << (K - E), 4) void ntt_rows_encrypt_batch_kernel(const DevPrime *__restrict__ primes,
                                                                                EncArgs a, uint32_t m) {
    constexpr int T = 1 << (K - E), RPL = LOGN - K;
    static_assert(SUBS * T == 1 << K, "one position of the row per thread");
    __shared__ uint64_t tile[SUBS * row_words(K)];
    const int tid = threadIdx.x, sub = tid / T, t = tid % T;
    const uint32_t chunks = (m + SUBS - 1) / SUBS;
    const uint32_t g0 = blockIdx.x % chunks * SUBS, r = blockIdx.x / chunks;
    const int row = (int)(r & ((1u << RPL) - 1));
    const uint32_t i = r >> RPL;
    const int nsub = (int)min<uint32_t>(SUBS, m - g0);
    const bool active = sub < nsub;
    const uint32_t mine = g0 + (uint32_t)(active ? sub : 0);
    const size_t row_off = (size_t)row << K;
    const DevPrime &Q = primes[i];
    const BfConst bc = bf_const(Q);
    const ulonglong2 *table = Q.fwd;
    auto addr = [sub](int idx) { return sub * row_words(K) + row_slot(idx); };
    auto transform = [&](const uint64_t *in) {
        asm volatile("" : "+s"(table));  // twiddles are loaded again rather than kept
        const GlobalTw<LOGN, false, ulonglong2> tw{table, row, RPL};
        auto load = [in](int idx, int) { return in[idx]; };
        auto stage = [&](int idx, uint64_t x) { tile[addr(idx)] = x; };
        run_phases<K, E, false, true>(tile, addr, load, stage, t, tw, bc, active);
        __syncthreads();
    };
    transform(a.U + (((size_t)mine * a.L1 + i) << LOGN) + row_off);
    // word v of the thread: position tid of the block's ciphertext v
    uint64_t u[SUBS];
#pragma unroll
    for (int v = 0; v < SUBS; v++) u[v] = tile[v * row_words(K) + row_slot(tid)];
    const size_t limb = ((size_t)i << LOGN) + row_off, ct_words = (size_t)a.L << LOGN;
#pragma unroll 1
    for (uint32_t k = 0; k < 2; k++) {
        __syncthreads();  // the tile has been read
        transform(a.out + (2 * mine + k) * ct_words + limb);
        const uint64_t pk = a.pk[((size_t)(k * a.K + i) << LOGN) + row_off + tid];
        const uint64_t pkq = pk * Q.ratio_hi + mulhi64(pk, Q.ratio_lo);
        const bool add = a.plain && k == 0;
#pragma unroll
        for (int v = 0; v < SUBS; v++) {
            if (v >= nsub) break;  // uniform
            uint64_t x = shoup_lazier(u[v], pk, pkq, bc.neg_q) + tile[v * row_words(K) + row_slot(tid)];
            if (a.drop) x = shoup(x, a.dc[i].inv, a.dc[i].inv_shoup, Q.q);
            else x = barrett64(x, Q.q, Q.ratio_hi);
            // (uniform slices: the thread's part of the addresses is tid alone)
            if (add) x = addmod(x, (a.plain + (g0 + v) * ct_words + limb)[tid], Q.q);
            (a.out + (2 * (g0 + v) + k) * ct_words + limb)[tid] = x;
        }
    }
}

// The ciphertexts of such a block, and the fewest it is taken for (N = 2^15, 2^16: rows of 256;
// the 32 rows of 128 and the 8 of 512 that a block of 256 threads has need more than one
// position per thread, and registers that spill).
constexpr uint32_t ENC_BATCH = 16;

template <int LOGN, bool SMALL>
void launch_encrypt_as(const EncArgs &a, uint32_t jn, const DevPrime *primes, hipStream_t st) {
    using S = PassShape<LOGN, SMALL>;
    constexpr int K1 = S::K1, K2 = S::K2, E = S::E, CS = S::CS, RS = S::RS;
    const uint32_t col_blocks = a.L * jn * ((1u << K2) / CS);
    const bool mx = rows_mixed<LOGN, K2, RS>(jn);
    const uint32_t row_blocks = a.L * rows_blocks_per_prime<LOGN, K2, E, RS>(jn, mx);
    ntt_cols_encrypt_kernel<LOGN, K1, E, CS><<<col_blocks, CS << (K1 - E), 0, st>>>(primes, a, jn);
    if constexpr (!SMALL && RS == ENC_BATCH) {
        if (a.u_cols) {
            const uint32_t m = jn / 2;
            ntt_rows_encrypt_batch_kernel<LOGN, K2, E, RS>
                <<<(a.L << K1) * ((m + RS - 1) / RS), RS << (K2 - E), 0, st>>>(primes, a, m);
            return;
        }
    }
    if (mx)
        ntt_rows_encrypt_kernel<LOGN, K2, E, RS, true><<<row_blocks, RS << (K2 - E), 0, st>>>(primes, a, jn);
    else
        ntt_rows_encrypt_kernel<LOGN, K2, E, RS, false><<<row_blocks, RS << (K2 - E), 0, st>>>(primes, a, jn);
}

template <int LOGN>
void launch_encrypt(const EncArgs &a, uint32_t jn, const DevPrime *primes, hipStream_t st) {
    with_shape<LOGN>((uint64_t)a.L * jn, [&](auto s) {
        launch_encrypt_as<LOGN, decltype(s)::value>(a, jn, primes, st);
    });
}

struct ModDownGroupDev {
    uint64_t *U;
    ModDownArgs a;
    uint32_t jn;
};
struct ModDownGroups {
    uint32_t n;
    uint32_t start[MAX_GROUPS + 1];
    ModDownGroupDev g[MAX_GROUPS];
};

template <int LOGN, int K, int E, int SUBS>
__global__ __launch_bounds__(SUBS << (K - E)) void ntt_cols_moddown_prep_grouped_kernel(
    const DevPrime *__restrict__ primes, ModDownGroups mg) {
    const uint32_t gi = group_of(mg.start, mg.n, blockIdx.x);
    const ModDownGroupDev &gr = mg.g[gi];
    const ModDownArgs &a = gr.a;
    __shared__ uint64_t tile[SUBS << K];
    cols_moddown_prep<LOGN, K, E, SUBS>(tile, blockIdx.x - mg.start[gi], gr.U, primes, a, gr.jn);
}

template <int LOGN, int K, int E, int SUBS, bool MX>
__global__ __launch_bounds__(SUBS << (K - E)) void ntt_rows_moddown_grouped_kernel(const DevPrime *__restrict__ primes,
                                                                                  ModDownGroups mg) {
    const uint32_t gi = group_of(mg.start, mg.n, blockIdx.x);
    const ModDownGroupDev &gr = mg.g[gi];
    const ModDownArgs &a = gr.a;
    const uint64_t *U = gr.U;
    rows_body<LOGN, K, E, SUBS, false, false, MX>(
        blockIdx.x - mg.start[gi], primes, a.L, 0, gr.jn,
        [&](uint32_t i, uint32_t j, size_t off) { return U[((size_t)(j * a.L + i) << LOGN) + off]; },
        [&](uint32_t i, uint32_t j, size_t off, uint64_t x) {
            const DevPrime &Q = primes[i];
            moddown_add<LOGN>(a, i, j, off, moddown_p<LOGN>(a, i, j, off), finish<false, true>(x, Q), Q);
        });
}

template <int LOGN, int K, int E, int SUBS>
__global__ __launch_bounds__(SUBS << (K - E)) void ntt_cols_moddown_kernel(const uint64_t *__restrict__ Pt,
                                                                          const DevPrime *__restrict__ primes,
                                                                          ModDownArgs a, uint32_t jn) {
    __shared__ uint64_t tile[SUBS << K];
    with_moddown_u(a, primes, [&](const auto &u) {
        cols_body_t<LOGN, K, E, SUBS, true>(
            tile, blockIdx.x, primes, 0, jn,
            [&](uint32_t i, uint32_t j, size_t off) { return Pt[((size_t)(j * a.L + i) << LOGN) + off]; },
            [&](uint32_t i, uint32_t j, size_t off, uint64_t x) {
                const DevPrime &Q = primes[i];
                moddown_add<LOGN>(a, i, j, off, finish<true, true>(x, Q), u(i, a.S[((size_t)j << LOGN) + off]), Q);
            });
    });
}

// Rows pass of an inverse transform of sigma(src).
template <int LOGN, int K, int E, int SUBS, bool MX>
__global__ __launch_bounds__(SUBS << (K - E)) void ntt_rows_galois_kernel(const uint64_t *__restrict__ src,
                                                                         LimbGrid slg, GaloisPerm perm,
                                                                         uint64_t *__restrict__ data,
                                                                         const DevPrime *__restrict__ primes,
                                                                         LimbGrid lg) {
    const GridAccess g{data, lg, LOGN};
    const GridAccess s{const_cast<uint64_t *>(src), slg, LOGN};
    rows_body<LOGN, K, E, SUBS, true, false, MX>(
        blockIdx.x, primes, lg.I, 0, lg.J,
        [&](uint32_t i, uint32_t j, size_t off) {
            return *s.at(i, j, galois_slot((uint32_t)off, perm.elt[j / perm.polys], LOGN));
        },
        [&](uint32_t i, uint32_t j, size_t off, uint64_t x) { *g.at(i, j, off) = x; });
}

template <int LOGN, bool SMALL>
void launch_inverse_galois_as(const uint64_t *src, LimbGrid slg, const GaloisPerm &perm, uint64_t *data, LimbGrid lg,
                           const DevPrime *primes, hipStream_t st) {
    using S = PassShape<LOGN, SMALL>;
    constexpr int K1 = S::K1, K2 = S::K2, E = S::E, CS = S::CS, RS = S::RS;
    const bool mx = rows_mixed<LOGN, K2, RS>(lg.J);
    const uint32_t row_blocks = lg.I * rows_blocks_per_prime<LOGN, K2, E, RS>(lg.J, mx);
    const uint32_t col_blocks = lg.I * lg.J * ((1u << K2) / CS);
    with_bool(mx, [&](auto m) {
        ntt_rows_galois_kernel<LOGN, K2, E, RS, decltype(m)::value>
            <<<row_blocks, RS << (K2 - E), 0, st>>>(src, slg, perm, data, primes, lg);
    });
    ntt_cols_kernel<LOGN, K1, E, CS, true, true, true><<<col_blocks, CS << (K1 - E), 0, st>>>(data, primes, lg, 0, lg.J);
}

template <int LOGN>
void launch_inverse_galois(const uint64_t *src, LimbGrid slg, const GaloisPerm &perm, uint64_t *data, LimbGrid lg,
                           const DevPrime *primes, hipStream_t st) {
    with_shape<LOGN>((uint64_t)lg.I * lg.J, [&](auto s) {
        launch_inverse_galois_as<LOGN, decltype(s)::value>(src, slg, perm, data, lg, primes, st);
    });
}

template <int LOGN, bool SMALL>
void launch_moddown_as(bool ckks, uint64_t *buf, const ModDownArgs &a, uint32_t jn, const DevPrime *primes,
                    hipStream_t st) {
    using S = PassShape<LOGN, SMALL>;
    constexpr int K1 = S::K1, K2 = S::K2, E = S::E, CS = S::CS, RS = S::RS;
    const uint32_t col_blocks = a.L * jn * ((1u << K2) / CS);
    const bool mx = rows_mixed<LOGN, K2, RS>(jn);
    const uint32_t row_blocks = a.L * rows_blocks_per_prime<LOGN, K2, E, RS>(jn, mx);
    if (ckks) {
        ntt_cols_moddown_prep_kernel<LOGN, K1, E, CS><<<col_blocks, CS << (K1 - E), 0, st>>>(buf, primes, a, jn);
        if (mx)
            ntt_rows_moddown_kernel<LOGN, K2, E, RS, true><<<row_blocks, RS << (K2 - E), 0, st>>>(buf, primes, a, jn);
        else
            ntt_rows_moddown_kernel<LOGN, K2, E, RS, false><<<row_blocks, RS << (K2 - E), 0, st>>>(buf, primes, a, jn);
    } else {
        const LimbGrid lg{1, a.L, a.L, jn};
        if (a.perm.polys)
            with_bool(mx, [&](auto m) {
                ntt_rows_galois_kernel<LOGN, K2, E, RS, decltype(m)::value>
                    <<<row_blocks, RS << (K2 - E), 0, st>>>(a.P, lg, a.perm, buf, primes, lg);
            });
        else if (mx)
            ntt_rows_kernel<LOGN, K2, E, RS, true, false, true, true>
                <<<row_blocks, RS << (K2 - E), 0, st>>>(buf, primes, lg, 0, jn);
        else
            ntt_rows_kernel<LOGN, K2, E, RS, true, false, true, false>
                <<<row_blocks, RS << (K2 - E), 0, st>>>(buf, primes, lg, 0, jn);
        ntt_cols_moddown_kernel<LOGN, K1, E, CS><<<col_blocks, CS << (K1 - E), 0, st>>>(buf, primes, a, jn);
    }
}

template <int LOGN>
void launch_moddown(bool ckks, uint64_t *buf, const ModDownArgs &a, uint32_t jn, const DevPrime *primes,
                    hipStream_t st) {
    with_shape<LOGN>((uint64_t)a.L * jn, [&](auto s) {
        launch_moddown_as<LOGN, decltype(s)::value>(ckks, buf, a, jn, primes, st);
    });
}

uint64_t group_limbs(const ModDownGroup *gs, uint32_t n) {
    uint64_t limbs = 0;
    for (uint32_t g = 0; g < n; g++) limbs += (uint64_t)gs[g].a.L * 2 * gs[g].count;
    return limbs;
}

template <int LOGN, bool SMALL>
void launch_moddown_groups_as(const ModDownGroup *gs, uint32_t n, const DevPrime *primes, hipStream_t st) {
    using S = PassShape<LOGN, SMALL>;
    constexpr int K1 = S::K1, K2 = S::K2, E = S::E, CS = S::CS, RS = S::RS;
    ModDownGroups cols{}, rmx{}, rfull{};
    std::vector<uint64_t> csz, msz, fsz;
    for (uint32_t g = 0; g < n; g++) {
        const uint32_t jn = 2 * gs[g].count;
        const ModDownGroupDev d{gs[g].U, gs[g].a, jn};
        cols.g[g] = d;
        csz.push_back((uint64_t)gs[g].a.L * jn * ((1u << K2) / CS));
        const bool mx = rows_mixed<LOGN, K2, RS>(jn);
        const uint64_t rb = (uint64_t)gs[g].a.L * rows_blocks_per_prime<LOGN, K2, E, RS>(jn, mx);
        if (mx) {
            rmx.g[msz.size()] = d;
            msz.push_back(rb);
        } else {
            rfull.g[fsz.size()] = d;
            fsz.push_back(rb);
        }
    }
    const uint32_t cb = fill_starts(cols, csz);
    ntt_cols_moddown_prep_grouped_kernel<LOGN, K1, E, CS><<<cb, CS << (K1 - E), 0, st>>>(primes, cols);
    if (!msz.empty()) {
        const uint32_t b = fill_starts(rmx, msz);
        ntt_rows_moddown_grouped_kernel<LOGN, K2, E, RS, true><<<b, RS << (K2 - E), 0, st>>>(primes, rmx);
    }
    if (!fsz.empty()) {
        const uint32_t b = fill_starts(rfull, fsz);
        ntt_rows_moddown_grouped_kernel<LOGN, K2, E, RS, false><<<b, RS << (K2 - E), 0, st>>>(primes, rfull);
    }
}

template <int LOGN>
void launch_moddown_groups(const ModDownGroup *gs, uint32_t n, const DevPrime *primes, hipStream_t st) {
    with_shape<LOGN>(group_limbs(gs, n), [&](auto s) {
        launch_moddown_groups_as<LOGN, decltype(s)::value>(gs, n, primes, st);
    });
}

}  // namespace

namespace {
bool moddown_jn(bool ckks, uint64_t *buf, const ModDownArgs &a, uint32_t jn, const DevPrime *primes, int logn,
                hipStream_t st) {
    if (logn < 13 || logn > 17 || jn == 0) return false;
    if ((uint64_t)jn * a.L > ((uint64_t(1) << 34) >> logn)) fail(ERR_INVALID_ARGUMENT, "batch too large for one launch");
    if (a.p_lpp && !ckks) fail(ERR_LOGIC, "a strided ModDown input is for the NTT form");
    switch (logn) {
        case 13: launch_moddown<13>(ckks, buf, a, jn, primes, st); break;
        case 14: launch_moddown<14>(ckks, buf, a, jn, primes, st); break;
        case 15: launch_moddown<15>(ckks, buf, a, jn, primes, st); break;
        case 16: launch_moddown<16>(ckks, buf, a, jn, primes, st); break;
        case 17: launch_moddown<17>(ckks, buf, a, jn, primes, st); break;
    }
    launch_check("ntt moddown launch");
    return true;
}
}  // namespace

bool ntt_moddown(bool ckks, uint64_t *buf, const ModDownArgs &a, uint32_t count, const DevPrime *primes, int logn,
                 hipStream_t st) {
    return moddown_jn(ckks, buf, a, 2 * count, primes, logn, st);
}

void ntt_inverse_galois(const uint64_t *src, LimbGrid slg, const GaloisPerm &perm, uint64_t *data, LimbGrid lg,
                        const DevPrime *primes, int logn, hipStream_t st) {
    if (logn < 13 || logn > 17) fail(ERR_LOGIC, "permuted inverse transforms take N = 2^13 .. 2^17");
    if (slg.I != lg.I || slg.J != lg.J || !perm.polys || lg.J > perm.polys * PERM_MAX)
        fail(ERR_LOGIC, "transform source and destination shapes differ");
    if ((uint64_t)lg.I * lg.J > ((uint64_t(1) << 34) >> logn)) fail(ERR_INVALID_ARGUMENT, "batch too large for one launch");
    switch (logn) {
        case 13: launch_inverse_galois<13>(src, slg, perm, data, lg, primes, st); break;
        case 14: launch_inverse_galois<14>(src, slg, perm, data, lg, primes, st); break;
        case 15: launch_inverse_galois<15>(src, slg, perm, data, lg, primes, st); break;
        case 16: launch_inverse_galois<16>(src, slg, perm, data, lg, primes, st); break;
        case 17: launch_inverse_galois<17>(src, slg, perm, data, lg, primes, st); break;
    }
    launch_check("permuted inverse ntt launch");
}

bool ntt_forward_small(const int8_t *Us, uint64_t *U, uint32_t L1, uint32_t m, uint32_t rows_from,
                       const DevPrime *primes, int logn, hipStream_t st) {
    if (logn < 13 || logn > 17 || m == 0 || (uint64_t)L1 * m > ((uint64_t(1) << 34) >> logn)) return false;
    auto go = [&](auto n) {
        constexpr int LOGN = decltype(n)::value;
        with_shape<LOGN>((uint64_t)L1 * m, [&](auto s) {
            launch_small_as<LOGN, decltype(s)::value>(Us, U, L1, m, rows_from, primes, st);
        });
    };
    switch (logn) {
        case 13: go(std::integral_constant<int, 13>{}); break;
        case 14: go(std::integral_constant<int, 14>{}); break;
        case 15: go(std::integral_constant<int, 15>{}); break;
        case 16: go(std::integral_constant<int, 16>{}); break;
        case 17: go(std::integral_constant<int, 17>{}); break;
    }
    launch_check("small ntt launch");
    return true;
}

bool ntt_encrypt_takes_columns(uint32_t m, uint32_t L, uint32_t L1, int logn) {
    const uint64_t most = (uint64_t(1) << 34) >> logn;
    return (logn == 15 || logn == 16) && m >= ENC_BATCH && (uint64_t)2 * m * L <= most &&
           (uint64_t)m * L1 <= most && ((uint64_t)2 * m * L << logn) > SMALL_WORDS;
}

bool ntt_encrypt_ckks(const EncArgs &a, uint32_t m, const DevPrime *primes, int logn, hipStream_t st) {
    if (logn < 13 || logn > 17 || m == 0) return false;
    const uint32_t jn = 2 * m;
    if ((uint64_t)jn * a.L > ((uint64_t(1) << 34) >> logn)) return false;
    switch (logn) {
        case 13: launch_encrypt<13>(a, jn, primes, st); break;
        case 14: launch_encrypt<14>(a, jn, primes, st); break;
        case 15: launch_encrypt<15>(a, jn, primes, st); break;
        case 16: launch_encrypt<16>(a, jn, primes, st); break;
        case 17: launch_encrypt<17>(a, jn, primes, st); break;
    }
    launch_check("ntt encrypt launch");
    return true;
}

bool ntt_moddown_polys(uint64_t *U, const ModDownArgs &a, uint32_t polys, const DevPrime *primes, int logn,
                       hipStream_t st) {
    return moddown_jn(true, U, a, polys, primes, logn, st);
}

bool ntt_moddown_groups(const ModDownGroup *gs, uint32_t n, const DevPrime *primes, int logn, hipStream_t st) {
    if (logn < 13 || logn > 17) return false;
    if (n > MAX_GROUPS) fail(ERR_INVALID_ARGUMENT, "too many groups for one launch");
    if (n == 0) return true;
    switch (logn) {
        case 13: launch_moddown_groups<13>(gs, n, primes, st); break;
        case 14: launch_moddown_groups<14>(gs, n, primes, st); break;
        case 15: launch_moddown_groups<15>(gs, n, primes, st); break;
        case 16: launch_moddown_groups<16>(gs, n, primes, st); break;
        case 17: launch_moddown_groups<17>(gs, n, primes, st); break;
    }
    launch_check("grouped moddown launch");
    return true;
}

}  // namespace shc

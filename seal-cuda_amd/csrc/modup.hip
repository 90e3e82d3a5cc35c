// modup.hip -- the key switch's ModUp transforms, alone and fused with the products by the
// key (N = 2^13 .. 2^17; the passes are those of ntt_device.h, the schedules ntt.hip's).
#include "accum.h"
#include "launch_limits.h"
#include "ntt_device.h"

namespace shc {
namespace {

// A pointer that is the same in every lane, as a scalar.
__device__ __forceinline__ const void *uniform_ptr(const void *p) {
    const uint64_t a = (uint64_t)p;
    const uint32_t lo = (uint32_t)__builtin_amdgcn_readfirstlane((uint32_t)a);
    const uint32_t hi = (uint32_t)__builtin_amdgcn_readfirstlane((uint32_t)(a >> 32));
    return (const void *)((uint64_t)hi << 32 | lo);
}

// The key switch's ModUp rows pass fused with the products by the key (N = 2^13 .. 2^16):
// a block owns RW adjacent rows of target prime i for CG ciphertexts (NS = CG x RW
// slots).  Each step transforms SUBS rows of T -- NS slots x SUBS/NS digits, the last K
// layers with the wide schedule -- stages them in LDS, and then every thread multiplies
// its coefficient of those rows by the key words of their digits and adds into
// three-word sums (one per slot and key component), so the transformed limbs never
// return to HBM:
//   P[ct][k][i][c] = sum_j NTT_i(T[i][ct][j])[c] * key[j][k][ki][c]   (S for i == L).
// With diag (CKKS, T without its own-prime limbs), the term j == i is the NTT-form input
// limb diag[ct * diag_stride + i * N].  The groups start at ciphertext ct_base.  A step
// past the last digit, or a ciphertext past the batch, transforms a repeated row and
// does not add or store it.  Groups of 4 and 2 ciphertexts take one row (RW = 1); a
// single ciphertext takes two rows (RW = 2), so that a step holds 8 of its digits
// instead of 16 (24 digits in 3 steps, not 2 with a third of the rows wasted).  With
// RW = 2 the slots run slot-major (each wave's rows share one row index, so its twiddle
// loads stay scalar).  Blocks of one tile run one after another on one XCD, so its key
// slice comes from that XCD's L2.
// Sum bound: up to 31 digits the transformed words (< 8q) enter the sums directly
// (31 * 8q^2 + q^2 < 2^128 for q < 2^60); beyond, R4 takes them below 4q first.
// FP: the target's prime is below 2^50 -- T holds the columns pass's doubles, the last
// layers run in fp64 and the sums are Acc26 of the transformed words' residues in [0, 4q).
// AHEAD, for groups of 4, and of 2 up to N = 2^14: the row's own twiddles are staged once for all
// steps, and a step's rows are requested while the step before runs its products, at three
// waves per SIMD instead of four.  Groups of 4: 20.0 -> 18.5 ms for 128 ciphertexts at N = 2^16,
// L = 24; 547 -> 434 us for 16 at N = 2^15, L = 15 in fp64.  Groups of 2 at N = 2^15 and 2^16 are
// better off with the fourth wave, which the registers of both cost them (relinearizations of
// two without / with, us: N = 2^16, L = 24 731 / 773, L = 8 124 / 129, N = 2^15, L = 15 169 / 184 and
// in fp64 157 / 163; N = 2^14, L = 8 64.0 / 60.8 and 57.3 / 57.1), and a single ciphertext's short
// launch too (274 -> 288 us with them).
constexpr bool keyprod_ahead(int logn, int cg) { return cg == 4 || (cg == 2 && logn <= 14); }

template <int LOGN, int K, int E, int SUBS, int CG, int RW, bool R4, bool FP>
__device__ __forceinline__ void rows_keyprod_core(
    uint64_t *tile, ulonglong2 *tws, uint32_t i, int g0, uint32_t grp, const uint64_t *__restrict__ T, const uint64_t *__restrict__ key,
    uint64_t *__restrict__ Pout, uint64_t *__restrict__ Sout, const DevPrime *__restrict__ primes,
    const uint64_t *__restrict__ diag, size_t diag_stride, uint32_t count, uint32_t L, uint32_t K_key, uint32_t ct_base, const KsFold &fold) {
    constexpr int TT = 1 << (K - E);  // threads per row
    constexpr int SZ = 1 << K;        // row length
    static_assert(SZ == SUBS * TT, "one coefficient per thread in the product phase");
    constexpr int NS = CG * RW;
    static_assert(SUBS % NS == 0, "whole digits per step");
    constexpr int RPL = LOGN - K;
    constexpr int DJ = SUBS / NS;  // digits per step
    static_assert(RW == 1 || DJ % (64 / TT) == 0, "slot-major: one slot per wave");
    using Acc = std::conditional_t<FP, Acc26, Acc3>;
    using Word = std::conditional_t<FP, Cut26, uint64_t>;  // an operand of the sums
    auto word = [](uint64_t x) -> Word {
        if constexpr (FP) return cut26(x);
        else return x;
    };
    const uint32_t ct0 = ct_base + grp * CG;
    const uint32_t gv = min<uint32_t>(CG, count - ct0);
    const bool short_row = diag && i < L;
    const uint32_t Lt = short_row ? L - 1 : L;
    const int tid = threadIdx.x;
    const int sub = tid / TT, t = tid % TT;
    // this thread's transform row: slot gg (ciphertext gg % CG, row gg / CG), digit dj;
    // tile row of (slot c, digit d): slot(c, d)
    const int gg = RW > 1 ? sub / DJ : sub % NS, dj = RW > 1 ? sub % DJ : sub / NS;
    auto slot = [](int c, int d) { return RW > 1 ? c * DJ + d : d * NS + c; };
    const size_t n = (size_t)1 << LOGN;
    auto row_off = [g0](int r) { return (size_t)(g0 + r) << K; };
    // the row index is uniform across a wave (one slot per wave when RW > 1)
    const int g_t = RW > 1 ? __builtin_amdgcn_readfirstlane(g0 + gg / CG) : g0;
    const DevPrime &P = primes[i];
    const BfConst bc = bf_const(P);
    const FpConst fc{P.q_fp, P.q_inv_fp};
    const double to_u52 = 4503599627370496.0 + 2 * P.q_fp;
    const uint32_t ki = i == L ? K_key - 1 : i;
    const size_t kstride = (size_t)K_key << LOGN;  // key[j][k] -> key[j][k+1]
    const uint64_t *kp = key + ((size_t)ki << LOGN) + row_off(0) + tid;  // row r: + r * SZ
    Acc a0[NS], a1[NS];
#pragma unroll
    for (int c = 0; c < NS; c++) a0[c] = a1[c] = Acc{0, 0, 0};
    const uint64_t *trow = T + (((size_t)i * count * L + (size_t)(ct0 + min<uint32_t>(gg % CG, gv - 1)) * Lt) << LOGN) +
                           row_off(gg / CG);
    const uint32_t steps = (Lt + DJ - 1) / DJ;
    constexpr bool AHEAD = keyprod_ahead(LOGN, CG);
    using W2 = std::conditional_t<FP, double2, ulonglong2>;
    const W2 *tab;
    if constexpr (FP) tab = P.fwd_fp;
    else tab = P.fwd;
    if constexpr (AHEAD) {
        static_assert(!AHEAD || RW == 1, "one row's twiddles are staged");
        stage_twiddles<K>((W2 *)tws, tab, g0, RPL, tid, SZ);
        __syncthreads();
    }
    uint64_t nx[1 << E];
    auto request = [&](uint32_t s) {
        const uint64_t *row = trow + ((size_t)min<uint32_t>(s * DJ + dj, Lt - 1) << LOGN);
#pragma unroll
        for (int j = 0; j < (1 << E); j++) nx[j] = row[phase_index<K, E, 0, E>(t, j)];
    };
    if (AHEAD && steps) request(0);  // (a one-digit level leaves no rows but the own-prime one)
    for (uint32_t s = 0; s < steps; s++) {
        if (s) __syncthreads();  // the previous step's products have read the tile
        // the first phase's twiddles are the same in every step; reloading them (cache hits)
        // keeps them from being held in registers across steps
        const void *tw = uniform_ptr(tab);
        asm volatile("" : "+s"(tw));
        auto twiddles = [&] {
            if constexpr (AHEAD) return TileTw<LOGN, W2>{(const W2 *)tw, g_t, RPL, (const W2 *)tws};
            else return GlobalTw<LOGN, false, W2>{(const W2 *)tw, g_t, RPL};
        };
        const auto twa = twiddles();
        if constexpr (!AHEAD) request(s);
        // small groups (short, latency-bound launches) also recompute their LDS addresses
        // each step, for fewer registers and more waves; a group of 4 keeps them (fewer
        // instructions; measured faster)
        int sub_s = sub, t_s = t;
        if constexpr (CG < 4) asm volatile("" : "+v"(sub_s), "+v"(t_s));
        auto addr_s = [sub_s](int idx) { return sub_s * row_words(K) + row_slot(idx); };
        // rows past the last digit (the last step of a short target) are not transformed:
        // with a group of 4 that is a whole wave, which leaves the SIMD to other waves
        const bool active = s * DJ + dj < Lt;
        if constexpr (FP) {
            auto load = [&](int, int j) { return __longlong_as_double((long long)nx[j]); };
            auto stage = [&](int idx, double x) { tile[addr_s(idx)] = fp_to_u52(x, to_u52); };
            run_phases_fp<K, E, true>(tile, addr_s, load, stage, t_s, twa, fc, active);
        } else {
            auto load = [&](int, int j) { return nx[j]; };
            auto stage = [&](int idx, uint64_t x) { tile[addr_s(idx)] = x; };
            run_phases<K, E, false, true>(tile, addr_s, load, stage, t_s, twa, bc, active);
        }
        // the key words of a digit are requested one digit ahead (the first before the
        // barrier), at clamped indices rather than behind a branch
        auto key_j = [&](uint32_t jt) {
            jt = min<uint32_t>(jt, Lt - 1);
            return short_row && jt >= i ? jt + 1 : jt;
        };
        uint64_t kn0[RW], kn1[RW];
        auto fetch_keys = [&](uint32_t j) {
#pragma unroll
            for (int r = 0; r < RW; r++) {
                kn0[r] = kp[(2 * j) * kstride + r * SZ];
                kn1[r] = kp[(2 * j + 1) * kstride + r * SZ];
            }
        };
        fetch_keys(key_j(s * DJ));
        __syncthreads();
        if (AHEAD && s + 1 < steps) request(s + 1);
#pragma unroll 1
        for (int d = 0; d < DJ; d++) {
            const uint32_t jt = s * DJ + d;
            if (jt >= Lt) break;  // uniform
            Word k0[RW], k1[RW];
#pragma unroll
            for (int r = 0; r < RW; r++) {
                k0[r] = word(kn0[r]);
                k1[r] = word(kn1[r]);
            }
            fetch_keys(key_j(jt + 1));
#pragma unroll
            for (int c = 0; c < NS; c++) {
                uint64_t x = tile[slot(c, d) * row_words(K) + row_slot(tid)];
                if (R4 && !FP) x = sub_if_ge_neg(x, bc.neg_four_q);
                const Word w = word(x);
                mac(a0[c], w, k0[c / CG]);
                mac(a1[c], w, k1[c / CG]);
            }
        }
    }
    if (short_row) {
#pragma unroll
        for (int c = 0; c < NS; c++) {
            const Word k0 = word(kp[(2 * i) * kstride + (c / CG) * SZ]);
            const Word k1 = word(kp[(2 * i + 1) * kstride + (c / CG) * SZ]);
            const size_t off = row_off(c / CG) + tid;
            const Word x = word(diag[(ct0 + min<uint32_t>(c % CG, gv - 1)) * diag_stride + ((size_t)i << LOGN) +
                                     (fold.diag_elt ? galois_slot((uint32_t)off, fold.diag_elt, LOGN) : off)]);
            mac(a0[c], x, k0);
            mac(a1[c], x, k1);
        }
    }
    // the ciphertext the switch adds into, times p (CKKS, i < L): one more term per sum,
    // and the ModDown reads no ciphertext
    if (fold.ct && i < L) {
        const uint64_t pm = fold.dc[i].p_mod;
#pragma unroll
        for (int c = 0; c < NS; c++) {
            const uint64_t *cw = fold.ct + (size_t)(ct0 + min<uint32_t>(c % CG, gv - 1)) * fold.ct_stride +
                                 ((size_t)i << LOGN) + row_off(c / CG) + tid;
            if constexpr (FP) {
                mac(a0[c], word(cw[0]), word(pm));
                if (!fold.c1_zero) mac(a1[c], word(cw[(size_t)L << LOGN]), word(pm));
            } else {
                mac<true>(a0[c], cw[0], pm);
                if (!fold.c1_zero) mac<true>(a1[c], cw[(size_t)L << LOGN], pm);
            }
        }
    }
#pragma unroll
    for (int c = 0; c < NS; c++) {
        if ((uint32_t)(c % CG) >= gv) continue;
        const size_t ct = ct0 + c % CG;
        const size_t off = row_off(c / CG) + tid;
        const uint64_t r0 = acc_reduce(a0[c], P), r1 = acc_reduce(a1[c], P);
        if (i == L) {
            Sout[(ct * 2 + 0) * n + off] = r0;
            Sout[(ct * 2 + 1) * n + off] = r1;
        } else {
            Pout[((ct * 2 + 0) * L + i) * n + off] = r0;
            Pout[((ct * 2 + 1) * L + i) * n + off] = r1;
        }
    }
}

// MIXED: some target primes are below 2^50 (the branch is uniform over the block).
template <int LOGN, int K, int E, int SUBS, int CG, int RW, bool R4, bool MIXED>
__device__ __forceinline__ void rows_keyprod_body(
    uint32_t bid, const uint64_t *__restrict__ T, const uint64_t *__restrict__ key, uint64_t *__restrict__ Pout,
    uint64_t *__restrict__ Sout, const DevPrime *__restrict__ primes, const uint64_t *__restrict__ diag,
    size_t diag_stride, uint32_t count, uint32_t L, uint32_t K_key, uint32_t ct_base, uint32_t groups,
    uint32_t tiles, const KsFold &fold) {
    constexpr int GPL = (1 << (LOGN - K)) / RW;  // row groups per limb
    static_assert(GPL * RW == (1 << (LOGN - K)), "whole row groups");
    __shared__ uint64_t tile[SUBS * row_words(K)];
    __shared__ ulonglong2 tws[keyprod_ahead(LOGN, CG) ? 1 << K : 1];
    // bid & 7 is the XCD (launches, and groups of a grouped launch, start at multiples of 8)
    const uint32_t xcd = bid & 7, kk = bid >> 3;
    const uint32_t tl = (kk / groups) * 8 + xcd;
    if (tl >= tiles) return;  // uniform: the whole block
    const uint32_t grp = kk % groups;
    const uint32_t i = tl / GPL;
    const int g0 = (int)(tl % GPL) * RW;  // first row of the group
    if constexpr (MIXED) {
        if (primes[i].fwd_fp) {
            rows_keyprod_core<LOGN, K, E, SUBS, CG, RW, R4, true>(tile, tws, i, g0, grp, T, key, Pout, Sout, primes, diag,
                                                                  diag_stride, count, L, K_key, ct_base, fold);
            return;
        }
    }
    rows_keyprod_core<LOGN, K, E, SUBS, CG, RW, R4, false>(tile, tws, i, g0, grp, T, key, Pout, Sout, primes, diag,
                                                           diag_stride, count, L, K_key, ct_base, fold);
}

template <int LOGN, int K, int E, int SUBS, int CG, int RW, bool R4, bool MIXED>
__global__ __launch_bounds__(SUBS << (K - E), keyprod_ahead(LOGN, CG) ? 3 : 4) void ntt_rows_keyprod_kernel(
    const uint64_t *__restrict__ T, const uint64_t *__restrict__ key, uint64_t *__restrict__ Pout,
    uint64_t *__restrict__ Sout, const DevPrime *__restrict__ primes, const uint64_t *__restrict__ diag,
    size_t diag_stride, uint32_t count, uint32_t L, uint32_t K_key, uint32_t ct_base, uint32_t groups,
    uint32_t tiles, KsFold fold) {
    rows_keyprod_body<LOGN, K, E, SUBS, CG, RW, R4, MIXED>(blockIdx.x, T, key, Pout, Sout, primes, diag, diag_stride, count,
                                                    L, K_key, ct_base, groups, tiles, fold);
}

// ---- grouped launches: ciphertexts at several levels in one launch per stage.  Group
// g owns blocks [start[g], start[g+1]) and runs the one-level body with its own
// arguments on block (blockIdx.x - start[g]); the argument tables travel by value (in
// the kernel-argument segment; the group index is uniform, so they are scalar loads).
struct KeyprodGroup {
    const uint64_t *T;
    uint64_t *P, *S;
    const DevPrime *primes;
    const uint64_t *diag;
    size_t diag_stride;
    uint32_t count, L, ct_base, groups, tiles;
    KsFold fold;
};
struct KeyprodGroups {
    uint32_t n;
    uint32_t start[MAX_GROUPS + 1];
    const uint64_t *key;
    uint32_t K_key;
    KeyprodGroup g[MAX_GROUPS];
};
template <int LOGN, int K, int E, int SUBS, int CG, int RW, bool R4, bool MIXED>
__global__ __launch_bounds__(SUBS << (K - E), keyprod_ahead(LOGN, CG) ? 3 : 4) void ntt_rows_keyprod_grouped_kernel(KeyprodGroups kg) {
    const uint32_t gi = group_of(kg.start, kg.n, blockIdx.x);
    const KeyprodGroup &a = kg.g[gi];
    rows_keyprod_body<LOGN, K, E, SUBS, CG, RW, R4, MIXED>(blockIdx.x - kg.start[gi], a.T, kg.key, a.P, a.S, a.primes,
                                                    a.diag, a.diag_stride, a.count, a.L, kg.K_key, a.ct_base,
                                                    a.groups, a.tiles, a.fold);
}

// The key switch's ModUp rows pass: the same code as a kernel of its own, so that
// profiles tell it apart from the other forward transforms.  Wide schedule; outputs
// left in [0, 4q) (FIN) or [0, 8q), ranges the key products' 128-bit sums absorb.
// jn_short: see rows_body (targets without their own digit's limb).
// MIXED: limbs of primes below 2^50 hold the columns pass's doubles, transformed in fp64
// and stored as words in [0, 4q).
template <int LOGN, int K, int E, int SUBS, bool FIN, bool MIXED>
__global__ __launch_bounds__(SUBS << (K - E)) void ntt_rows_modup_kernel(uint64_t *__restrict__ data,
                                                                        const DevPrime *__restrict__ primes,
                                                                        LimbGrid lg, uint32_t jn_short) {
    __shared__ uint64_t tile[SUBS * row_words(K)];
    const GridAccess g{data, lg, LOGN};
    if constexpr (MIXED) {
        constexpr int T = 1 << (K - E), SZ = 1 << K;
        // rows_body's block order: limb group fastest, then row, then prime
        const uint32_t jc_count = (lg.J + SUBS - 1) / SUBS;
        const uint32_t r = blockIdx.x / jc_count, j0 = blockIdx.x % jc_count * SUBS;
        const uint32_t row = r & ((1u << (LOGN - K)) - 1), i = r >> (LOGN - K);
        const DevPrime &P = primes[i];
        if (P.fwd_fp) {
            const uint32_t jend = jn_short && i + 1 < lg.I ? jn_short : lg.J;
            if (j0 >= jend) return;  // uniform: a whole block past a short row
            const uint32_t nsub = min<uint32_t>(SUBS, jend - j0);
            const int sub = threadIdx.x / T, t = threadIdx.x % T;
            const bool active = (uint32_t)sub < nsub;
            const uint64_t *in = g.at(i, j0 + (active ? sub : 0), (size_t)row << K);
            const double to_u52 = 4503599627370496.0 + 2 * P.q_fp;
            auto addr = [sub](int idx) { return sub * row_words(K) + row_slot(idx); };
            auto load = [in](int idx, int) { return __longlong_as_double((long long)in[idx]); };
            auto stage = [&](int idx, double x) { tile[addr(idx)] = fp_to_u52(x, to_u52); };
            run_phases_fp<K, E, true>(tile, addr, load, stage, t,
                                      GlobalTw<LOGN, false, double2>{P.fwd_fp, (int)row, LOGN - K},
                                      FpConst{P.q_fp, P.q_inv_fp}, active);
            __syncthreads();
            for (uint32_t e = threadIdx.x; e < nsub * SZ; e += SUBS * T)
                *g.at(i, j0 + e / SZ, ((size_t)row << K) + e % SZ) = tile[(e / SZ) * row_words(K) + row_slot(e % SZ)];
            return;
        }
    }
    rows_body_t<LOGN, K, E, SUBS, false, true>(
        tile, blockIdx.x, primes, lg.I, 0, lg.J, [&](uint32_t i, uint32_t j, size_t off) { return *g.at(i, j, off); },
        [&](uint32_t i, uint32_t j, size_t off, uint64_t x) {
            *g.at(i, j, off) = FIN ? finish<false, false>(x, primes[i]) : x;
        },
        jn_short);
}

// ModUp columns pass into T[i][ct][j] (target-major, so that the rows pass walks one
// prime's limbs at a time): a block takes one tile of 16 columns of digit j of
// ciphertext ct (read from d[ct][j]), keeps it in registers, and for each of tc target
// primes i in turn reduces it modulo q_i when the digit's prime exceeds 8 q_i (the
// forward butterflies take inputs < 8q) and runs the first K layers -- one LDS round
// trip and two barriers per target -- so the loads' latency is paid once per tile and
// chunk of targets, not once per target.  Large batches take all L + 1 targets per block
// (measured 0.6 ms faster per 128 ciphertexts than one block per target); small ones
// split the targets into chunks so that the grid still fills the GPU, down to one target
// per block (ONE: no words held across targets, 97 VGPRs instead of 128).
// skip_diag: limb (i, i) is not produced (its NTT is the NTT-form input limb) and the
// targets i < L keep L - 1 limbs per ciphertext, T[i][ct][j - (j > i)].
// MIXED: targets below 2^50 take the fp64 butterflies and leave doubles in T (their digits
// enter below 2 q_i, by Barrett when the digit's prime is above that).
template <int LOGN, int K, int E, int SUBS, bool ONE, bool MIXED>
__device__ __forceinline__ void cols_modup_body(uint32_t bid, const uint64_t *__restrict__ d, size_t d_ct_stride,
                                                uint64_t *__restrict__ T, const DevPrime *__restrict__ targets,
                                                const DevPrime *__restrict__ digits, uint32_t count, uint32_t L,
                                                bool skip_diag, uint32_t tc) {
    static_assert(K >= E, "the first phase fills all 2^E registers");
    constexpr int C = 1 << (LOGN - K);
    constexpr int TILES = C / SUBS;
    __shared__ uint64_t tile[SUBS * (1 << K)];
    const int tid = threadIdx.x;
    const int col = tid % SUBS, t = tid / SUBS;
    const uint32_t chunks = (L + tc) / tc;  // ceil((L + 1) / tc)
    const uint32_t rc = bid / TILES;  // (ct * L + j) * chunks + chunk
    const uint32_t r = rc / chunks;          // ct * L + j
    const uint32_t i0 = (rc % chunks) * tc, i1 = min<uint32_t>(i0 + tc, L + 1);
    const int c0 = (int)(bid % TILES) * SUBS;
    const uint32_t j = r % L;
    const size_t ct = r / L;
    const uint64_t *in = d + ct * d_ct_stride + ((size_t)j << LOGN) + c0 + col;
    const uint64_t qj = digits[j].q;
    auto addr = [col](int idx) { return idx * SUBS + col; };
    // the second phase's twiddles (the first 2^K entries of the target's table) go through
    // LDS, each thread bringing one, requested a target ahead
    __shared__ ulonglong2 tws[1 << K];
    static_assert(SUBS << (K - E) >= 1 << K, "one twiddle per thread");
    const bool brings = tid < 1 << K;
    auto table = [&](uint32_t i) {
        return MIXED && targets[i].fwd_fp ? (const ulonglong2 *)targets[i].fwd_fp : targets[i].fwd;
    };
    // target i of the digit's words (word(idx, k)), the twiddles in tws
    auto transform = [&](uint32_t i, const auto &word) {
        const bool short_row = skip_diag && i < L;
        const size_t limb = (size_t)i * count * L + ct * (short_row ? L - 1 : L) + (short_row && j > i ? j - 1 : j);
        uint64_t *out = T + (limb << LOGN) + c0 + col;
        const DevPrime &P = targets[i];
        if constexpr (MIXED) {
            if (P.fwd_fp) {
                const bool reduce = qj > 2 * P.q;
                auto load = [&](int idx, int k) {
                    const uint64_t x = word(idx, k);
                    return fp_from_u52(reduce ? barrett64(x, P.q, P.ratio_hi) : x);
                };
                auto store = [out](int idx, double x) { out[(size_t)idx * C] = (uint64_t)__double_as_longlong(x); };
                run_phases_fp<K, E, false>(tile, addr, load, store, t,
                                           TileTw<LOGN, double2>{P.fwd_fp, 0, 0, (const double2 *)tws},
                                           FpConst{P.q_fp, P.q_inv_fp}, true);
                return;
            }
        }
        const bool reduce = qj > 8 * P.q;
        auto load = [&](int idx, int k) {
            const uint64_t x = word(idx, k);
            return reduce ? barrett64(x, P.q, P.ratio_hi) : x;
        };
        auto store = [out](int idx, uint64_t x) { out[(size_t)idx * C] = x; };
        run_phases<K, E, false, true>(tile, addr, load, store, t, TileTw<LOGN, ulonglong2>{P.fwd, 0, 0, tws},
                                      bf_const(P), true);
    };
    if constexpr (ONE) {
        // one target per block (small batches): the first phase loads straight from the
        // digit, nothing held across targets (fewer registers, more waves)
        if (skip_diag && i0 == j) return;  // uniform: the whole block
        if (brings) tws[tid] = load_tw(table(i0), tid);
        transform(i0, [&](int idx, int) { return in[(size_t)idx * C]; });
        return;
    }
    ulonglong2 tw = load_tw(table(i0), brings ? tid : 0);
    uint64_t dv[1 << E];
#pragma unroll
    for (int k = 0; k < (1 << E); k++) dv[k] = in[(size_t)phase_index<K, E, 0, E>(t, k) * C];
    for (uint32_t i = i0; i < i1; i++) {
        __syncthreads();  // the previous target's second phase has read the tile
        if (brings) tws[tid] = tw;
        if (i + 1 < i1) tw = load_tw(table(i + 1), brings ? tid : 0);
        if (skip_diag && i == j) continue;  // uniform
        transform(i, [&](int, int k) { return dv[k]; });
    }
}

// (held to 128 VGPRs: four waves per SIMD)
template <int LOGN, int K, int E, int SUBS, bool ONE, bool MIXED>
__global__ __launch_bounds__(SUBS << (K - E), 4) void ntt_cols_modup_kernel(const uint64_t *__restrict__ d,
                                                                        size_t d_ct_stride,
                                                                        uint64_t *__restrict__ T,
                                                                        const DevPrime *__restrict__ targets,
                                                                        const DevPrime *__restrict__ digits,
                                                                        uint32_t count, uint32_t L, bool skip_diag,
                                                                        uint32_t tc) {
    cols_modup_body<LOGN, K, E, SUBS, ONE, MIXED>(blockIdx.x, d, d_ct_stride, T, targets, digits, count, L, skip_diag, tc);
}

struct ModupGroup {
    const uint64_t *d;
    size_t d_ct_stride;
    uint64_t *T;
    const DevPrime *targets;
    uint32_t count, L, tc;
    bool skip_diag;
};
struct ModupGroups {
    uint32_t n;
    uint32_t start[MAX_GROUPS + 1];
    const DevPrime *digits;
    ModupGroup g[MAX_GROUPS];
};

// (held to 128 VGPRs, four waves per SIMD; the integer form over several targets, whose
// groups' arguments would spill there, to three: 407 us spilled, 395 with its twiddles from
// the table, for two groups of 2 at N = 2^16, L = 24 and 20; relinearizations of groups of 4
// and 8 3,483 -> 3,425 us)
template <int LOGN, int K, int E, int SUBS, bool ONE, bool MIXED>
__global__ __launch_bounds__(SUBS << (K - E), ONE || MIXED ? 4 : 3) void ntt_cols_modup_grouped_kernel(ModupGroups mg) {
    const uint32_t gi = group_of(mg.start, mg.n, blockIdx.x);
    const ModupGroup &a = mg.g[gi];
    cols_modup_body<LOGN, K, E, SUBS, ONE, MIXED>(blockIdx.x - mg.start[gi], a.d, a.d_ct_stride, a.T, a.targets, mg.digits,
                                           a.count, a.L, a.skip_diag, a.tc);
}

// Targets per block of the ModUp columns pass: all L + 1 when the (digit, tile) blocks
// alone fill the GPU, fewer (chunks of them) so that a small batch still has about
// 16384 blocks.
inline uint32_t modup_targets_per_block(uint32_t tile_blocks, uint32_t L, uint32_t forced = 0) {
    if (forced) return forced < L + 1 ? forced : L + 1;
    const uint32_t want = (16384 + tile_blocks - 1) / tile_blocks;
    const uint32_t chunks = want < 1 ? 1 : (want > L + 1 ? L + 1 : want);
    return (L + chunks) / chunks;  // ceil((L + 1) / chunks)
}

// log2 of the values per thread of the ModUp columns pass: 8 where targets take the fp64
// butterflies, whose pass waits more than it issues (289 -> 271 us for 16 ciphertexts at
// N = 2^15, L = 15 against 16 values), 16 for integer ones (13.5 ms for 128 at N = 2^16,
// L = 24 against 13.9 with 8, 16.6 with 4).
constexpr int modup_cols_log(bool mixed) { return mixed ? 3 : 4; }

template <int LOGN, bool SMALL>
void launch_modup_as(const uint64_t *d, size_t d_stride, uint64_t *T, uint32_t cts, uint32_t L, const DevPrime *targets,
                  const DevPrime *digits, bool skip_diag, bool reduce_4q, bool mixed, const KernelProbe *probe,
                  hipStream_t st, KsShape shape) {
    using S = PassShape<LOGN, SMALL>;
    constexpr int K1 = S::K1, K2 = S::K2, E = S::E, CS = S::CS, RS = S::RS;
    const uint32_t tc = modup_targets_per_block(cts * L * ((1u << K2) / CS), L, shape.cols_targets);
    const uint32_t col_grid = cts * L * ((L + tc) / tc) * ((1u << K2) / CS);
    with_bool(mixed, [&](auto mx) {
        constexpr bool MIXED = decltype(mx)::value;
        // (at N = 2^16 16 values win here although they spill: 1,230 against 1,280 us for 16
        // ciphertexts at L = 24; 8 at N = 2^15 for 16 at L = 15 save 19 us of 1,266)
        constexpr int EC = SMALL ? E : LOGN == 16 ? 4 : modup_cols_log(MIXED);
        if (tc == 1)
            ntt_cols_modup_kernel<LOGN, K1, EC, CS, true, MIXED><<<col_grid, CS << (K1 - EC), 0, st>>>(
                d, d_stride, T, targets, digits, cts, L, skip_diag, tc);
        else
            ntt_cols_modup_kernel<LOGN, K1, EC, CS, false, MIXED><<<col_grid, CS << (K1 - EC), 0, st>>>(
                d, d_stride, T, targets, digits, cts, L, skip_diag, tc);
    });
    const LimbGrid lg{cts * L, 1, L + 1, cts * L};
    const uint32_t row_blocks = ((L + 1) << K1) * ((lg.J + RS - 1) / RS);
    if (probe) SHC_HIP(hipEventRecord(probe->begin, st));
    const uint32_t jn_short = skip_diag ? cts * (L - 1) : 0;
    with_bool(mixed, [&](auto mx) {
        constexpr bool MIXED = decltype(mx)::value;
        if (reduce_4q)
            ntt_rows_modup_kernel<LOGN, K2, E, RS, true, MIXED>
                <<<row_blocks, RS << (K2 - E), 0, st>>>(T, targets, lg, jn_short);
        else
            ntt_rows_modup_kernel<LOGN, K2, E, RS, false, MIXED>
                <<<row_blocks, RS << (K2 - E), 0, st>>>(T, targets, lg, jn_short);
    });
    if (probe) SHC_HIP(hipEventRecord(probe->end, st));
}

template <int LOGN>
void launch_modup(const uint64_t *d, size_t d_stride, uint64_t *T, uint32_t cts, uint32_t L, const DevPrime *targets,
                  const DevPrime *digits, bool skip_diag, bool reduce_4q, bool mixed, const KernelProbe *probe,
                  hipStream_t st, KsShape shape) {
    with_shape<LOGN>((uint64_t)cts * L * (L + 1), [&](auto s) {
        launch_modup_as<LOGN, decltype(s)::value>(d, d_stride, T, cts, L, targets, digits, skip_diag, reduce_4q, mixed,
                                                  probe, st, shape);
    });
}

// The fused rows pass + key products over a batch's groups.
template <int LOGN, bool R4, bool MIXED>
void launch_keyprod_groups(const uint64_t *T, const uint64_t *key, uint64_t *P, uint64_t *S, const uint64_t *diag,
                           size_t diag_stride, uint32_t cts, uint32_t L, uint32_t K_key, const DevPrime *targets,
                           uint32_t tiles, uint64_t tile_slots, uint32_t group, const KsFold &fold, hipStream_t st) {
    constexpr int K2 = LOGN - LOGN / 2;
    constexpr int E = 4;
    constexpr int RS = 16;
    // groups of `group` ciphertexts (4 by default), then what is left
    const uint32_t g = group == 1 || group == 2 ? group : 4;
    const auto [g4, g2, singles] = split_groups(LOGN, cts, g);
    if (g4)
        ntt_rows_keyprod_kernel<LOGN, K2, E, RS, 4, 1, R4, MIXED><<<(uint32_t)(tile_slots * g4), RS << (K2 - E), 0, st>>>(
            T, key, P, S, targets, diag, diag_stride, cts, L, K_key, 0, g4, tiles, fold);
    if (g2)
        ntt_rows_keyprod_kernel<LOGN, K2, E, RS, 2, 1, R4, MIXED><<<(uint32_t)(tile_slots * g2), RS << (K2 - E), 0, st>>>(
            T, key, P, S, targets, diag, diag_stride, cts, L, K_key, cts - 2 * g2 - singles, g2, tiles, fold);
    if (singles) {
        // single ciphertexts: two rows per block
        const uint32_t tiles2 = tiles / 2;
        const uint32_t slots2 = (uint32_t)keyprod_slots(LOGN, L, true);
        ntt_rows_keyprod_kernel<LOGN, K2, E, RS, 1, 2, R4, MIXED><<<slots2 * singles, RS << (K2 - E), 0, st>>>(
            T, key, P, S, targets, diag, diag_stride, cts, L, K_key, cts - singles, singles, tiles2, fold);
    }
}

template <int LOGN>
void launch_modup_keyprod(const uint64_t *d, size_t d_stride, uint64_t *T, const uint64_t *key, uint64_t *P,
                          uint64_t *S, const uint64_t *diag, size_t diag_stride, uint32_t cts, uint32_t L,
                          uint32_t K_key, const DevPrime *targets, const DevPrime *digits, bool mixed,
                          const KernelProbe *probe, hipStream_t st, KsShape shape, const KsFold &fold) {
    constexpr int K1 = LOGN / 2;
    constexpr int K2 = LOGN - K1;
    constexpr int CS = 16;
    const uint32_t tc = modup_targets_per_block(cts * L * ((1u << K2) / CS), L, shape.cols_targets);
    const uint32_t col_grid = cts * L * ((L + tc) / tc) * ((1u << K2) / CS);
    auto cols = [&](auto e, auto mx, auto one) {
        constexpr int E = decltype(e)::value;
        ntt_cols_modup_kernel<LOGN, K1, E, CS, decltype(one)::value, decltype(mx)::value>
            <<<col_grid, CS << (K1 - E), 0, st>>>(d, d_stride, T, targets, digits, cts, L, diag != nullptr, tc);
    };
    with_bool(mixed, [&](auto mx) {
        with_bool(tc == 1, [&](auto one) {
            constexpr int E = modup_cols_log(decltype(mx)::value);
            // (up to N = 2^14 a small launch takes 4 values, as the other small passes do)
            if constexpr (LOGN <= 14)
                with_shape<LOGN>((uint64_t)cts * L * (L + 1), [&](auto s) {
                    cols(std::integral_constant<int, decltype(s)::value ? 2 : E>{}, mx, one);
                });
            else
                cols(std::integral_constant<int, E>{}, mx, one);
        });
    });
    const uint32_t tiles = (L + 1) << K1;
    const uint64_t tile_slots = keyprod_slots(LOGN, L, false);
    if (tile_slots * cts >= (uint64_t(1) << 32))
        fail(ERR_INVALID_ARGUMENT, "key-switch batch too large for one launch");
    if (probe) SHC_HIP(hipEventRecord(probe->begin, st));
    // up to 31 digits the transformed words (< 8q) enter the sums unreduced
    // (contexts with fp64 primes have few integer targets: always reduced there)
    auto groups = [&](auto r4, auto mx) {
        launch_keyprod_groups<LOGN, decltype(r4)::value, decltype(mx)::value>(
            T, key, P, S, diag, diag_stride, cts, L, K_key, targets, tiles, tile_slots, shape.rows_group, fold, st);
    };
    if (mixed) groups(std::true_type{}, std::true_type{});
    else if (L > 31) groups(std::true_type{}, std::false_type{});
    else groups(std::false_type{}, std::false_type{});
    if (probe) SHC_HIP(hipEventRecord(probe->end, st));
}

template <int LOGN>
void launch_modup_keyprod_groups(const KsGroup *gs, uint32_t n, const uint64_t *key, uint32_t K_key,
                                 const DevPrime *digits, bool mixed, hipStream_t st) {
    constexpr int K1 = LOGN / 2;
    constexpr int K2 = LOGN - K1;
    constexpr int E = 4;
    constexpr int CS = 16;
    constexpr int RS = 16;
    // columns pass: targets per block chosen for the whole launch's tile blocks
    uint64_t tile_blocks = 0;
    uint32_t maxL = 0;
    for (uint32_t g = 0; g < n; g++) {
        tile_blocks += (uint64_t)gs[g].count * gs[g].L * ((1u << K2) / CS);
        maxL = gs[g].L > maxL ? gs[g].L : maxL;
    }
    const uint64_t want = (16384 + tile_blocks - 1) / tile_blocks;
    ModupGroups mg{};
    mg.digits = digits;
    std::vector<uint64_t> msz;
    bool all_one = true;
    for (uint32_t g = 0; g < n; g++) {
        const KsGroup &a = gs[g];
        const uint32_t chunks = (uint32_t)(want < 1 ? 1 : (want > a.L + 1 ? a.L + 1 : want));
        const uint32_t tc = (a.L + chunks) / chunks;
        all_one = all_one && tc == 1;
        mg.g[g] = ModupGroup{a.d, a.d_ct_stride, a.T, a.targets, a.count, a.L, tc, a.diag != nullptr};
        msz.push_back((uint64_t)a.count * a.L * ((a.L + tc) / tc) * ((1u << K2) / CS));
    }
    const uint32_t cb = fill_starts(mg, msz);
    with_bool(all_one, [&](auto one) {
        with_bool(mixed, [&](auto mx) {
            constexpr int EC = modup_cols_log(decltype(mx)::value);
            ntt_cols_modup_grouped_kernel<LOGN, K1, EC, CS, decltype(one)::value, decltype(mx)::value>
                <<<cb, CS << (K1 - EC), 0, st>>>(mg);
        });
    });
    // fused rows pass + key products: groups of 4, then of 2, then single ciphertexts
    KeyprodGroups t4{}, t2{}, t1{};
    t4.key = t2.key = t1.key = key;
    t4.K_key = t2.K_key = t1.K_key = K_key;
    std::vector<uint64_t> s4, s2, s1;
    for (uint32_t g = 0; g < n; g++) {
        const KsGroup &a = gs[g];
        const uint32_t tiles = (a.L + 1) << K1;
        const uint64_t tile_slots = keyprod_slots(LOGN, a.L, false);
        const auto [g4, g2, singles] = split_groups(LOGN, a.count, 4);
        if (g4) {
            t4.g[s4.size()] =
                KeyprodGroup{a.T, a.P, a.S, a.targets, a.diag, a.diag_stride, a.count, a.L, 0, g4, tiles, a.fold};
            s4.push_back(tile_slots * g4);
        }
        if (g2) {
            t2.g[s2.size()] =
                KeyprodGroup{a.T, a.P, a.S, a.targets, a.diag, a.diag_stride, a.count, a.L, a.count - 2 * g2 - singles,
                                           g2, tiles, a.fold};
            s2.push_back(tile_slots * g2);
        }
        if (singles) {
            const uint32_t tiles2 = tiles / 2;
            const uint64_t slots2 = keyprod_slots(LOGN, a.L, true);
            t1.g[s1.size()] = KeyprodGroup{a.T, a.P, a.S, a.targets, a.diag, a.diag_stride, a.count, a.L,
                                           a.count - singles, singles, tiles2, a.fold};
            s1.push_back(slots2 * singles);
        }
    }
    const bool r4 = maxL > 31;
    if (!s4.empty()) {
        const uint32_t b = fill_starts(t4, s4);
        if (mixed)
            ntt_rows_keyprod_grouped_kernel<LOGN, K2, E, RS, 4, 1, true, true><<<b, RS << (K2 - E), 0, st>>>(t4);
        else if (r4)
            ntt_rows_keyprod_grouped_kernel<LOGN, K2, E, RS, 4, 1, true, false><<<b, RS << (K2 - E), 0, st>>>(t4);
        else
            ntt_rows_keyprod_grouped_kernel<LOGN, K2, E, RS, 4, 1, false, false><<<b, RS << (K2 - E), 0, st>>>(t4);
    }
    if (!s2.empty()) {
        const uint32_t b = fill_starts(t2, s2);
        if (mixed)
            ntt_rows_keyprod_grouped_kernel<LOGN, K2, E, RS, 2, 1, true, true><<<b, RS << (K2 - E), 0, st>>>(t2);
        else if (r4)
            ntt_rows_keyprod_grouped_kernel<LOGN, K2, E, RS, 2, 1, true, false><<<b, RS << (K2 - E), 0, st>>>(t2);
        else
            ntt_rows_keyprod_grouped_kernel<LOGN, K2, E, RS, 2, 1, false, false><<<b, RS << (K2 - E), 0, st>>>(t2);
    }
    if (!s1.empty()) {
        const uint32_t b = fill_starts(t1, s1);
        if (mixed)
            ntt_rows_keyprod_grouped_kernel<LOGN, K2, E, RS, 1, 2, true, true><<<b, RS << (K2 - E), 0, st>>>(t1);
        else if (r4)
            ntt_rows_keyprod_grouped_kernel<LOGN, K2, E, RS, 1, 2, true, false><<<b, RS << (K2 - E), 0, st>>>(t1);
        else
            ntt_rows_keyprod_grouped_kernel<LOGN, K2, E, RS, 1, 2, false, false><<<b, RS << (K2 - E), 0, st>>>(t1);
    }
}

}  // namespace

bool ntt_forward_modup(const uint64_t *d, size_t d_ct_stride, uint64_t *T, uint32_t count, uint32_t L,
                       const DevPrime *targets, const DevPrime *digits, int logn, bool skip_diag, bool reduce_4q,
                       bool mixed, hipStream_t st, const KernelProbe *probe, KsShape shape) {
    if (logn < 13 || logn > 17 || count == 0) return false;
    if ((uint64_t)count * L * (L + 1) > ((uint64_t(1) << 34) >> logn))
        fail(ERR_INVALID_ARGUMENT, "key-switch batch too large for one launch");
    switch (logn) {
        case 13: launch_modup<13>(d, d_ct_stride, T, count, L, targets, digits, skip_diag, reduce_4q, mixed, probe, st, shape); break;
        case 14: launch_modup<14>(d, d_ct_stride, T, count, L, targets, digits, skip_diag, reduce_4q, mixed, probe, st, shape); break;
        case 15: launch_modup<15>(d, d_ct_stride, T, count, L, targets, digits, skip_diag, reduce_4q, mixed, probe, st, shape); break;
        case 16: launch_modup<16>(d, d_ct_stride, T, count, L, targets, digits, skip_diag, reduce_4q, mixed, probe, st, shape); break;
        case 17: launch_modup<17>(d, d_ct_stride, T, count, L, targets, digits, skip_diag, reduce_4q, mixed, probe, st, shape); break;
    }
    launch_check("ntt modup launch");
    return true;
}

bool ntt_modup_keyprod(const uint64_t *d, size_t d_ct_stride, uint64_t *T, const uint64_t *key, uint64_t *P,
                       uint64_t *S, const uint64_t *diag, size_t diag_stride, uint32_t count, uint32_t L,
                       uint32_t key_count, const DevPrime *targets, const DevPrime *digits, int logn, bool mixed,
                       hipStream_t st, const KernelProbe *probe, KsShape shape, KsFold fold) {
    if (logn < 13 || logn > 16 || count == 0) return false;
    if ((uint64_t)count * L * (L + 1) > ((uint64_t(1) << 34) >> logn))
        fail(ERR_INVALID_ARGUMENT, "key-switch batch too large for one launch");
    auto go = [&](auto n) {
        launch_modup_keyprod<decltype(n)::value>(d, d_ct_stride, T, key, P, S, diag, diag_stride, count, L, key_count,
                                                 targets, digits, mixed, probe, st, shape, fold);
    };
    switch (logn) {
        case 13: go(std::integral_constant<int, 13>{}); break;
        case 14: go(std::integral_constant<int, 14>{}); break;
        case 15: go(std::integral_constant<int, 15>{}); break;
        default: go(std::integral_constant<int, 16>{}); break;
    }
    launch_check("ntt modup keyprod launch");
    return true;
}

bool ntt_modup_keyprod_groups(const KsGroup *gs, uint32_t n, const uint64_t *key, uint32_t key_count,
                              const DevPrime *digits, int logn, bool mixed, hipStream_t st) {
    if (logn < 13 || logn > 16) return false;
    if (n > MAX_GROUPS) fail(ERR_INVALID_ARGUMENT, "too many groups for one launch");
    if (n == 0) return true;
    switch (logn) {
        case 13: launch_modup_keyprod_groups<13>(gs, n, key, key_count, digits, mixed, st); break;
        case 14: launch_modup_keyprod_groups<14>(gs, n, key, key_count, digits, mixed, st); break;
        case 15: launch_modup_keyprod_groups<15>(gs, n, key, key_count, digits, mixed, st); break;
        default: launch_modup_keyprod_groups<16>(gs, n, key, key_count, digits, mixed, st); break;
    }
    launch_check("grouped modup keyprod launch");
    return true;
}

}  // namespace shc

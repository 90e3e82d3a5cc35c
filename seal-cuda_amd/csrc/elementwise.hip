// elementwise.hip -- coefficient-wise evaluator operations.
//
// Evaluator::negateInplace / addInplace / subInplace (src/evaluator.cpp:149-357; GPU
// src/evaluator_cuda.cu:145-281), addPlainInplace / subPlainInplace (evaluator.cpp:
// 1603-1764, GPU :1544-1690; BFV through src/utils/scalingvariant.cpp:53-131),
// multiplyPlainNtt (evaluator.cpp:1932, GPU :1811) and the GPU multiplyPlainNormal
// (src/evaluator_cuda.cu:1726-1807: the plaintext is always lifted, m >= ceil(t/2) ->
// m + q_i - t, then NTT, dyadic product, inverse NTT).  The CPU multiplyPlainNormal
// multiplies by a monomial plaintext without lifting it (evaluator.cpp:1818-1866), so
// for a monomial with m >= ceil(t/2) the two reference paths give different words;
// this build follows the GPU path it replaces.
#include "elementwise.h"
#include "accum.h"
#include <type_traits>
#include "behz.h"
#include "crypto.h"
#include "modarith.h"
#include "ntt.h"

namespace shc {
namespace {

constexpr int TPB = 256;

inline uint32_t blocks_for(size_t n) {
    const size_t b = (n + TPB - 1) / TPB;
    return (uint32_t)(b < (size_t(1) << 20) ? b : (size_t(1) << 20));
}

enum BinOp { BIN_ADD, BIN_SUB, BIN_MUL_PLAIN };

template <int OP>
__global__ void binary_kernel(const uint64_t *__restrict__ a, const uint64_t *__restrict__ b, uint64_t *out,
                              const DevPrime *__restrict__ primes, uint32_t L, int logn, size_t total) {
    const size_t limb_words = (size_t)L << logn;
    for (size_t idx = (size_t)blockIdx.x * TPB + threadIdx.x; idx < total; idx += (size_t)gridDim.x * TPB) {
        const size_t r = idx % limb_words;
        const DevPrime &P = primes[r >> logn];
        const uint64_t x = a[idx];
        uint64_t o;
        if (OP == BIN_ADD) o = addmod(x, b[idx], P.q);
        else if (OP == BIN_SUB) o = submod(x, b[idx], P.q);
        else o = mulmod(x, b[r], P.q, P.ratio_lo, P.ratio_hi);
        out[idx] = o;
    }
}

// The same two words per thread with 16-byte accesses (all pointers 16-byte aligned;
// N is even, so a pair never straddles two limbs).  From N = 128 a wave's 128 words lie
// in one limb, and the limb index is wave-uniform.
__device__ __forceinline__ uint32_t pair_limb(size_t w, int logn, uint32_t L) {
    uint32_t r = (uint32_t)(w >> logn);
    if (logn >= 7) r = __builtin_amdgcn_readfirstlane(r);
    return r % L;
}

template <int OP>
__global__ void binary_pairs_kernel(const ulonglong2 *__restrict__ a, const uint64_t *__restrict__ b, ulonglong2 *out,
                                    const DevPrime *__restrict__ primes, uint32_t L, int logn, size_t pairs) {
    const size_t n = (size_t)1 << logn;
    for (size_t p = (size_t)blockIdx.x * TPB + threadIdx.x; p < pairs; p += (size_t)gridDim.x * TPB) {
        const size_t w = 2 * p;
        const uint32_t l = pair_limb(w, logn, L);
        const DevPrime &P = primes[l];
        const ulonglong2 x = a[p];
        const ulonglong2 y = OP == BIN_MUL_PLAIN ? *reinterpret_cast<const ulonglong2 *>(b + ((size_t)l << logn) + (w & (n - 1)))
                                                 : reinterpret_cast<const ulonglong2 *>(b)[p];
        ulonglong2 o;
        if (OP == BIN_ADD) {
            o.x = addmod(x.x, y.x, P.q);
            o.y = addmod(x.y, y.y, P.q);
        } else if (OP == BIN_SUB) {
            o.x = submod(x.x, y.x, P.q);
            o.y = submod(x.y, y.y, P.q);
        } else {
            o.x = mulmod(x.x, y.x, P.q, P.ratio_lo, P.ratio_hi);
            o.y = mulmod(x.y, y.y, P.q, P.ratio_lo, P.ratio_hi);
        }
        out[p] = o;
    }
}

__global__ void negate_pairs_kernel(const ulonglong2 *__restrict__ a, ulonglong2 *out,
                                    const DevPrime *__restrict__ primes, uint32_t L, int logn, size_t pairs) {
    for (size_t p = (size_t)blockIdx.x * TPB + threadIdx.x; p < pairs; p += (size_t)gridDim.x * TPB) {
        const uint64_t q = primes[pair_limb(2 * p, logn, L)].q;
        const ulonglong2 x = a[p];
        out[p] = make_ulonglong2(negmod(x.x, q), negmod(x.y, q));
    }
}

inline bool aligned16(const void *p) { return ((uintptr_t)p & 15) == 0; }

template <int OP>
void launch_binary(const uint64_t *a, const uint64_t *b, uint64_t *out, const DevPrime *primes, uint32_t L, int logn,
                   size_t total, hipStream_t st) {
    if (logn >= 1 && aligned16(a) && aligned16(b) && aligned16(out)) {
        const size_t pairs = total / 2;
        binary_pairs_kernel<OP><<<blocks_for(pairs), TPB, 0, st>>>(reinterpret_cast<const ulonglong2 *>(a), b,
                                                                    reinterpret_cast<ulonglong2 *>(out), primes, L,
                                                                    logn, pairs);
    } else {
        binary_kernel<OP><<<blocks_for(total), TPB, 0, st>>>(a, b, out, primes, L, logn, total);
    }
}

__global__ void negate_kernel(const uint64_t *__restrict__ a, uint64_t *out, const DevPrime *__restrict__ primes,
                              uint32_t L, int logn, size_t total) {
    for (size_t idx = (size_t)blockIdx.x * TPB + threadIdx.x; idx < total; idx += (size_t)gridDim.x * TPB)
        out[idx] = negmod(a[idx], primes[(idx >> logn) % L].q);
}

__global__ void add_plain_poly0_kernel(const uint64_t *ct, const uint64_t *__restrict__ plain, uint64_t *out,
                                       const DevPrime *__restrict__ primes, uint32_t size, uint32_t L, int logn,
                                       bool subtract, size_t total) {
    const size_t limb_words = (size_t)L << logn;
    for (size_t idx = (size_t)blockIdx.x * TPB + threadIdx.x; idx < total; idx += (size_t)gridDim.x * TPB) {
        const size_t r = idx % limb_words;
        const uint64_t x = ct[idx];
        if ((idx / limb_words) % size == 0) {
            const uint64_t q = primes[r >> logn].q;
            out[idx] = subtract ? submod(x, plain[r], q) : addmod(x, plain[r], q);
        } else {
            out[idx] = x;
        }
    }
}

// lifted[l][c] = (m - t [m >= ceil(t/2)]) mod q_l for m = plain[c] < t.
__global__ void plain_lift_kernel(const uint64_t *__restrict__ plain, uint64_t *__restrict__ lifted, uint64_t t,
                                  const DevPrime *__restrict__ primes, uint32_t L, int logn, size_t total) {
    const uint64_t thr = (t + 1) >> 1;
    for (size_t idx = (size_t)blockIdx.x * TPB + threadIdx.x; idx < total; idx += (size_t)gridDim.x * TPB) {
        const size_t c = idx & (((size_t)1 << logn) - 1);
        const DevPrime &P = primes[idx >> logn];
        const uint64_t m = plain[c];
        const uint64_t mq = m >= P.q ? barrett64(m, P.q, P.ratio_hi) : m;
        lifted[idx] = m >= thr ? submod(mq, t >= P.q ? barrett64(t, P.q, P.ratio_hi) : t, P.q) : mq;
    }
}

// out[h][ct][p][l][c] = sum_j plains[h][j][l][c] * cts[j][ct][p][l][c] mod q_l for the
// H outputs h0 .. h0 + H - 1 (hn of them valid; the rest repeat the last, unstored).
// A thread owns one word position (l, c) of G consecutive polynomials (ct, p): each
// ciphertext word it loads serves H outputs (the diagonal matrix-vector products' giant
// steps) and each plaintext word G polynomials, so the plaintexts -- shared by every
// ciphertext of the batch -- are loaded polys / G times instead of polys times (and the
// block order below serves the repeats from L2).  Sums in three words (Acc3), folded mod
// q every 64 terms.  With G = 2 and H = 8 the sums fit three waves per SIMD (the launch
// bound), which measured faster than G = 4 at two waves.
//
// xcd: the grid is exactly groups x (lw / TPB) blocks with lw / TPB a multiple of 8, and
// block B (dispatched to XCD B % 8) takes position block 8 (B / 8 / groups) + B % 8 of
// polynomial group (B / 8) % groups: consecutive blocks of one XCD share their plaintext
// words, which then come from that XCD's L2 after the first.
template <int H, int G>
__global__ __launch_bounds__(TPB, 3) void plain_dot_many_kernel(const uint64_t *__restrict__ cts, const uint64_t *__restrict__ plains,
                                      uint64_t *__restrict__ out, const DevPrime *__restrict__ primes, uint32_t terms,
                                      uint32_t h0, uint32_t hn, uint32_t polys, uint32_t L, int logn, size_t total,
                                      bool xcd) {
    const size_t lw = (size_t)L << logn, pw = (size_t)polys * lw;
    size_t first = (size_t)blockIdx.x * TPB + threadIdx.x;
    if (xcd) {
        const uint32_t groups = (polys + G - 1) / G, k = blockIdx.x >> 3;
        first = (size_t)(k % groups) * lw + ((size_t)(k / groups) * 8 + (blockIdx.x & 7)) * TPB + threadIdx.x;
    }
    for (size_t idx = first; idx < total; idx += (size_t)gridDim.x * TPB) {
        const uint32_t row = uniform_row(idx, logn), grp = row / L;  // idx = grp * lw + r
        const size_t r = idx - (size_t)grp * lw;
        const uint32_t p0 = grp * G, gn = min<uint32_t>(G, polys - p0);
        const DevPrime &P = primes[row - grp * L];
        const uint64_t *pp[H];
#pragma unroll
        for (int h = 0; h < H; h++) pp[h] = plains + (size_t)(h0 + min<uint32_t>(h, hn - 1)) * terms * lw + r;
        const uint64_t *cp = cts + (size_t)p0 * lw + r;
        Acc3 acc[G][H];
#pragma unroll
        for (int g = 0; g < G; g++)
#pragma unroll
            for (int h = 0; h < H; h++) acc[g][h] = Acc3{0, 0, 0};
        for (uint32_t j = 0; j < terms; j++) {
            uint64_t pv[H];
#pragma unroll
            for (int h = 0; h < H; h++) pv[h] = pp[h][(size_t)j * lw];
#pragma unroll
            for (int g = 0; g < G; g++) {
                if ((uint32_t)g < gn) {  // uniform: a wave shares its polynomial group
                    const uint64_t t = cp[(size_t)j * pw + (size_t)g * lw];
#pragma unroll
                    for (int h = 0; h < H; h++) mac(acc[g][h], t, pv[h]);
                }
            }
            if ((j & 63) == 63) {
#pragma unroll
                for (int g = 0; g < G; g++)
#pragma unroll
                    for (int h = 0; h < H; h++) acc_fold(acc[g][h], P);
            }
        }
#pragma unroll
        for (int g = 0; g < G; g++)
            if ((uint32_t)g < gn)
#pragma unroll
                for (int h = 0; h < H; h++)
                    if ((uint32_t)h < hn) out[(size_t)(h0 + h) * pw + (size_t)(p0 + g) * lw + r] = acc_reduce(acc[g][h], P);
    }
}

// The same sums where both outputs and polynomials are many (a batch of diagonal matrix-vector
// products): a product of small matrices per word position.  A block owns PT positions x
// 16 outputs x 16 polynomials and stages JC terms at a time in LDS, so that a word is loaded
// polys / 16 or outputs / 16 times instead of once per 2 or 8 sums: the per-thread form moved
// 80 GB through L2 for 12 GB of operands (32 terms x 32 outputs x 32 polynomials, N = 2^15,
// L = 15) and waited for it.  A thread keeps 4 x 4 sums of its position (8 LDS words for 16
// products); the words of the next JC terms are requested while these are summed.  Primes
// below 2^50 stage the words cut at 26 bits and sum in Acc26.  That product takes 4.6 ms (12 GB
// at 2.6 TB/s; 148 VGPRs, three blocks per CU), 10.0 per thread.  32 positions per block (512
// threads) measured 5.2 ms held to 128 VGPRs (13 spilled) and 5.7 ms without.
constexpr int PT = 16;           // positions per block (128-byte rows)
constexpr int DT = 16;           // outputs, and polynomials, per block
constexpr int JC = 2;            // terms per stage
constexpr int DB = PT * 16;      // threads: 4 x 4 tiles of 4 x 4 sums per position

struct DotArgs {
    const uint64_t *cts, *plains;
    uint64_t *out;
    const DevPrime *primes;
    uint32_t terms, outputs, polys, L;
    int logn;
    uint32_t tiles, hb, gb;      // position tiles, output and polynomial blocks
};

template <bool FP>
__device__ __forceinline__ void plain_dot_tile(uint2 (*lds)[JC][2 * DT][PT], const DotArgs &a, size_t r0,
                                               const DevPrime &P, uint32_t h0, uint32_t g0) {
    using Acc = std::conditional_t<FP, Acc26, Acc3>;
    using Word = std::conditional_t<FP, Cut26, uint64_t>;
    const size_t lw = (size_t)a.L << a.logn, pw = (size_t)a.polys * lw;
    const int tid = threadIdx.x, pos = tid % PT, tl = tid / PT;
    const int th = (tl / 4) * 4, tg = (tl % 4) * 4;  // this thread's 4 x 4 sums
    // loads: row tl (< 16) of the outputs' plaintexts and of the polynomials, per term
    const uint64_t *pp = a.plains + (size_t)min(h0 + tl, a.outputs - 1) * a.terms * lw + r0 + pos;
    const uint64_t *cp = a.cts + (size_t)min(g0 + tl, a.polys - 1) * lw + r0 + pos;
    uint64_t nx[2 * JC];
    auto request = [&](uint32_t j0) {
#pragma unroll
        for (int k = 0; k < JC; k++) {
            const size_t j = min<uint32_t>(j0 + k, a.terms - 1);
            nx[2 * k] = pp[j * lw];
            nx[2 * k + 1] = cp[j * pw];
        }
    };
    auto cut = [](uint64_t x) -> uint2 {
        if constexpr (FP) {
            const Cut26 c = cut26(x);
            return uint2{c.lo, c.hi};
        }
        return uint2{(uint32_t)x, (uint32_t)(x >> 32)};
    };
    auto word = [](uint2 w) -> Word {
        if constexpr (FP) return Cut26{w.x, w.y};
        else return (uint64_t)w.y << 32 | w.x;
    };
    Acc acc[4][4];
#pragma unroll
    for (int h = 0; h < 4; h++)
#pragma unroll
        for (int g = 0; g < 4; g++) acc[h][g] = Acc{0, 0, 0};
    request(0);
    for (uint32_t j0 = 0, b = 0; j0 < a.terms; j0 += JC, b ^= 1) {
        // two buffers: the barrier of the stage before has passed its readers of this one
#pragma unroll
        for (int k = 0; k < JC; k++) {
            lds[b][k][tl][pos] = cut(nx[2 * k]);
            lds[b][k][DT + tl][pos] = cut(nx[2 * k + 1]);
        }
        __syncthreads();
        if (j0 + JC < a.terms) request(j0 + JC);
#pragma unroll 1
        for (int k = 0; k < JC; k++) {
            if (j0 + k >= a.terms) break;  // uniform
            Word w[4], t[4];
#pragma unroll
            for (int x = 0; x < 4; x++) w[x] = word(lds[b][k][th + x][pos]), t[x] = word(lds[b][k][DT + tg + x][pos]);
#pragma unroll
            for (int h = 0; h < 4; h++)
#pragma unroll
                for (int g = 0; g < 4; g++) mac(acc[h][g], t[g], w[h]);
        }
        if ((j0 & 63) + JC == 64) {
#pragma unroll
            for (int h = 0; h < 4; h++)
#pragma unroll
                for (int g = 0; g < 4; g++) acc_fold(acc[h][g], P);
        }
    }
#pragma unroll
    for (int h = 0; h < 4; h++)
#pragma unroll
        for (int g = 0; g < 4; g++)
            if (h0 + th + h < a.outputs && g0 + tg + g < a.polys)
                a.out[(size_t)(h0 + th + h) * pw + (size_t)(g0 + tg + g) * lw + r0 + pos] = acc_reduce(acc[h][g], P);
}

__global__ __launch_bounds__(DB, 3) void plain_dot_tiles_kernel(DotArgs a) {
    __shared__ uint2 lds[2][JC][2 * DT][PT];
    // the blocks of one position tile run one after another on one XCD (block % 8), whose L2
    // serves the words they share
    const uint32_t subs = a.hb * a.gb, k = blockIdx.x >> 3;
    const uint32_t tile = k / subs * 8 + (blockIdx.x & 7), sub = k % subs;
    if (tile >= a.tiles) return;  // uniform
    const size_t r0 = (size_t)tile * PT;
    const DevPrime &P = a.primes[r0 >> a.logn];
    const uint32_t h0 = sub / a.gb * DT, g0 = sub % a.gb * DT;
    if (P.fwd_fp) plain_dot_tile<true>(lds, a, r0, P, h0, g0);
    else plain_dot_tile<false>(lds, a, r0, P, h0, g0);
}

// Where the tiles beat the per-thread form: a tile costs the same however many of its 16 x 16
// sums are asked for, and its set-up weighs more the fewer terms there are, so the line is a
// share of the tiles' sums, in sixteenths, for terms >= 16, >= 8, >= 2 and 1, one lower for Acc26
// sums of 8 terms and more, and for 16 terms of fewer polynomials than outputs.  Measured,
// per-thread / tiles in us, N = 2^15 (60-bit primes, L = 12 and 15; 40-bit): 32 terms 8x16
// (outputs x polynomials) 1,291 / 1,325 and 1,290 / 1,051 (a half), 16x8 1,376 / 1,315, 12x12
// 1,555 / 1,337 (9/16), 20x20 4,082 / 5,026 and 4,080 / 3,979 (6/16); ratios at 8 terms 12x12 1.01, 16x10
// 1.06 (10/16), 40-bit 1.02; at 2 terms 16x10 0.88, 11x16 1.09 (11/16), 40-bit 0.98 and 1.19; at
// 1 term 24x16 679 / 757 (12/16), 16x16 458 / 395, 40-bit 679 / 698.
bool plain_dot_takes_tiles(uint32_t terms, uint32_t outputs, uint32_t polys, bool fp) {
    const uint64_t slots = (uint64_t)((outputs + DT - 1) / DT) * ((polys + DT - 1) / DT) * DT * DT;
    const uint32_t line = terms >= 16 ? 9 - (fp || polys < outputs) : terms >= 8 ? 10 - fp : terms >= 2 ? 11 : 14 - 2 * fp;
    return 16 * (uint64_t)outputs * polys >= line * slots;
}

template <int H>
void launch_plain_dot(uint32_t G, const uint64_t *cts, const uint64_t *plains, uint64_t *out, const DevPrime *primes,
                      uint32_t terms, uint32_t h0, uint32_t hn, uint32_t polys, uint32_t L, int logn, hipStream_t st) {
    const size_t groups = (polys + G - 1) / G, lw = (size_t)L << logn, total = groups * lw;
    const size_t rblocks = lw / TPB;
    // the XCD-aware order where the grid is one block per (group, position block)
    const bool xcd = groups > 1 && lw % TPB == 0 && rblocks % 8 == 0 && groups * rblocks < (size_t(1) << 20);
    if (G == 2)
        plain_dot_many_kernel<H, 2><<<blocks_for(total), TPB, 0, st>>>(cts, plains, out, primes, terms, h0, hn, polys, L,
                                                                        logn, total, xcd);
    else
        plain_dot_many_kernel<H, 1><<<blocks_for(total), TPB, 0, st>>>(cts, plains, out, primes, terms, h0, hn, polys, L,
                                                                        logn, total, xcd);
}

void check_level(const Context &c, uint32_t L) {
    if (L < 1 || L > c.key_count()) fail(ERR_INVALID_ARGUMENT, "limb count out of range");
}

}  // namespace

void poly_add(const Context &c, const uint64_t *a, const uint64_t *b, uint64_t *out, uint32_t polys, uint32_t L,
              hipStream_t st) {
    check_level(c, L);
    const size_t total = ((size_t)polys * L) << c.logn;
    if (!total) return;
    launch_binary<BIN_ADD>(a, b, out, c.primes(), L, c.logn, total, st);
    launch_check("add");
}

void poly_sub(const Context &c, const uint64_t *a, const uint64_t *b, uint64_t *out, uint32_t polys, uint32_t L,
              hipStream_t st) {
    check_level(c, L);
    const size_t total = ((size_t)polys * L) << c.logn;
    if (!total) return;
    launch_binary<BIN_SUB>(a, b, out, c.primes(), L, c.logn, total, st);
    launch_check("sub");
}

void poly_negate(const Context &c, const uint64_t *a, uint64_t *out, uint32_t polys, uint32_t L, hipStream_t st) {
    check_level(c, L);
    const size_t total = ((size_t)polys * L) << c.logn;
    if (!total) return;
    if (c.logn >= 1 && aligned16(a) && aligned16(out))
        negate_pairs_kernel<<<blocks_for(total / 2), TPB, 0, st>>>(reinterpret_cast<const ulonglong2 *>(a),
                                                                   reinterpret_cast<ulonglong2 *>(out), c.primes(), L,
                                                                   c.logn, total / 2);
    else
        negate_kernel<<<blocks_for(total), TPB, 0, st>>>(a, out, c.primes(), L, c.logn, total);
    launch_check("negate");
}

void multiply_plain_ntt(const Context &c, const uint64_t *a, const uint64_t *plain, uint64_t *out, uint32_t polys,
                        uint32_t L, hipStream_t st) {
    check_level(c, L);
    const size_t total = ((size_t)polys * L) << c.logn;
    if (!total) return;
    launch_binary<BIN_MUL_PLAIN>(a, plain, out, c.primes(), L, c.logn, total, st);
    launch_check("multiply_plain");
}

void add_plain_poly0(const Context &c, const uint64_t *ct, const uint64_t *plain, uint64_t *out, uint32_t count,
                     uint32_t size, uint32_t L, bool subtract, hipStream_t st) {
    check_level(c, L);
    if (size < 1) fail(ERR_INVALID_ARGUMENT, "ciphertext size must be at least 1");
    const size_t total = (((size_t)count * size) * L) << c.logn;
    if (!total) return;
    add_plain_poly0_kernel<<<blocks_for(total), TPB, 0, st>>>(ct, plain, out, c.primes(), size, L, c.logn, subtract,
                                                              total);
    launch_check("add_plain");
}

void bfv_add_plain(const Context &c, const uint64_t *ct, const uint64_t *plain, uint64_t *out, uint32_t count,
                   uint32_t size, uint32_t L, bool subtract, hipStream_t st) {
    if (c.scheme != SCHEME_BFV) fail(ERR_LOGIC, "scaled plaintext addition is for BFV");
    if (L < 1 || L >= c.key_count()) fail(ERR_INVALID_ARGUMENT, "level out of range");
    if (size < 1) fail(ERR_INVALID_ARGUMENT, "ciphertext size must be at least 1");
    const size_t ct_words = ((size_t)size * L) << c.logn;
    if (out != ct) SHC_HIP(hipMemcpyAsync(out, ct, (size_t)count * ct_words * 8, hipMemcpyDeviceToDevice, st));
    for (uint32_t i = 0; i < count; i++) bfv_scale_add(c, out + i * ct_words, plain, L, subtract, st);
}

void bfv_plain_to_ntt(const Context &c, const uint64_t *plain, uint32_t L, uint64_t *out, hipStream_t st) {
    if (c.scheme != SCHEME_BFV || !c.plain) fail(ERR_LOGIC, "plaintext lift is for BFV");
    check_level(c, L);
    const size_t lw = (size_t)L << c.logn;
    plain_lift_kernel<<<blocks_for(lw), TPB, 0, st>>>(plain, out, c.plain, c.primes(), L, c.logn, lw);
    launch_check("plain_lift");
    ntt_forward(out, L, L, c.primes(), c.logn, NTT_FULL, st);
}

void multiply_plain_accumulate(const Context &c, const uint64_t *cts, const uint64_t *plains, uint32_t terms,
                               uint32_t polys, uint32_t L, uint64_t *out, hipStream_t st) {
    multiply_plain_accumulate_many(c, cts, plains, terms, 1, polys, L, out, st);
}

void multiply_plain_accumulate_many(const Context &c, const uint64_t *cts, const uint64_t *plains, uint32_t terms,
                                    uint32_t outputs, uint32_t polys, uint32_t L, uint64_t *out, hipStream_t st) {
    check_level(c, L);
    if (!terms) fail(ERR_INVALID_ARGUMENT, "no terms to accumulate");
    if (!outputs) fail(ERR_INVALID_ARGUMENT, "no outputs to accumulate");
    if (!polys) return;
    // two polynomials per thread (the plaintexts' reuse) -- a ciphertext's pair -- one
    // for a lone polynomial
    const uint32_t G = polys >= 2 ? 2 : 1;
    const DevPrime *primes = c.primes();
    const int logn = c.logn;
    const uint64_t tiles = ((uint64_t)L << logn) / PT;
    const uint64_t tile_blocks = (tiles + 7) / 8 * 8 * ((outputs + DT - 1) / DT) * ((polys + DT - 1) / DT);
    uint32_t fp = 0;
    for (uint32_t i = 0; i < L; i++) fp += c.host_primes[i].fwd_fp != nullptr;
    if (plain_dot_takes_tiles(terms, outputs, polys, 2 * fp > L) && logn >= 5 && tile_blocks < (uint64_t(1) << 32) / DB) {
        const DotArgs a{cts, plains, out, primes, terms, outputs, polys, L, logn, (uint32_t)tiles,
                        (outputs + DT - 1) / DT, (polys + DT - 1) / DT};
        plain_dot_tiles_kernel<<<(uint32_t)tile_blocks, DB, 0, st>>>(a);
        launch_check("plain_dot_tiles");
        return;
    }
    for (uint32_t h0 = 0; h0 < outputs;) {
        const uint32_t left = outputs - h0;
        const uint32_t hn = left >= 8 ? 8 : left;
        if (hn > 4) launch_plain_dot<8>(G, cts, plains, out, primes, terms, h0, hn, polys, L, logn, st);
        else if (hn > 2) launch_plain_dot<4>(G, cts, plains, out, primes, terms, h0, hn, polys, L, logn, st);
        else if (hn == 2) launch_plain_dot<2>(G, cts, plains, out, primes, terms, h0, hn, polys, L, logn, st);
        else launch_plain_dot<1>(G, cts, plains, out, primes, terms, h0, hn, polys, L, logn, st);
        launch_check("plain_dot");
        h0 += hn;
    }
}

size_t bfv_multiply_plain_workspace(const Context &c, uint32_t L) { return ((size_t)L << c.logn) * 8; }

void bfv_multiply_plain(const Context &c, const uint64_t *a, const uint64_t *plain, uint64_t *out, uint32_t polys,
                        uint32_t L, void *ws, size_t ws_bytes, hipStream_t st) {
    if (c.scheme != SCHEME_BFV || !c.plain) fail(ERR_LOGIC, "coefficient-form plain multiply is for BFV");
    check_level(c, L);
    if (!ws || ws_bytes < bfv_multiply_plain_workspace(c, L))
        fail(ERR_INVALID_ARGUMENT, "workspace too small for plain multiply");
    const size_t words = ((size_t)polys * L) << c.logn;
    if (!words) return;
    uint64_t *lifted = static_cast<uint64_t *>(ws);
    bfv_plain_to_ntt(c, plain, L, lifted, st);
    if (out != a) SHC_HIP(hipMemcpyAsync(out, a, words * 8, hipMemcpyDeviceToDevice, st));
    ntt_forward(out, polys * L, L, c.primes(), c.logn, NTT_FULL, st);
    multiply_plain_ntt(c, out, lifted, out, polys, L, st);
    ntt_inverse(out, polys * L, L, c.primes(), c.logn, NTT_FULL, st);
}

}  // namespace shc

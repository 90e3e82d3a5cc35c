// ntt_device.h -- device code shared by the transform kernels (ntt.hip, modup.hip,
// moddown.hip): register phases, the rows and columns passes, grouped-launch tables.
#pragma once
#include "ntt.h"
#include "butterfly.h"
#include "butterfly_fp.h"
#include "launch_limits.h"
#include "modarith.h"
#include <type_traits>
#include <vector>

namespace shc {
namespace {

// Twiddle tables are global memory; saying so lets the compiler use global loads
// (flat loads would also hold up the LDS waits).
__device__ __forceinline__ ulonglong2 load_tw(const ulonglong2 *tw, int i) {
    typedef uint64_t g2 __attribute__((ext_vector_type(2)));
    const g2 v = ((const __attribute__((address_space(1))) g2 *)tw)[i];
    return ulonglong2{v.x, v.y};
}

__device__ __forceinline__ double2 load_tw(const double2 *tw, int i) {
    typedef double g2 __attribute__((ext_vector_type(2)));
    const g2 v = ((const __attribute__((address_space(1))) g2 *)tw)[i];
    return double2{v.x, v.y};
}

// Position inside a 2^K-point sub-transform of register j of thread t, for the phase
// that runs local layers [S0, S0+EP): the EP butterfly bits sit at bit positions
// [K-S0-EP, K-S0) of the index and come from the low EP bits of j.
template <int K, int E, int S0, int EP>
__device__ __forceinline__ int phase_index(int t, int j) {
    constexpr int LOWB = K - S0 - EP;
    const int jl = j & ((1 << EP) - 1);
    const int jh = j >> EP;
    const int other = (t << (E - EP)) | jh;
    return ((other >> LOWB) << (K - S0)) | (jl << LOWB) | (other & ((1 << LOWB) - 1));
}

// A prime's butterfly constants: 4q, 2^64 - q, 2^64 - 4q, 2^64 - 8q.
struct BfConst {
    uint64_t four_q, neg_q, neg_four_q, neg_eight_q;
};
__device__ __forceinline__ BfConst bf_const(const DevPrime &P) {
    return BfConst{P.q << 2, 0 - P.q, P.neg_four_q, P.neg_eight_q};
}

// Where a phase finds the twiddle of local layer s, local group lg (of the 2^s groups of a
// sub-transform).  GlobalTw: the prime's table, for sub-transform g of the 2^L0 at layer L0.
// TileTw: the first phase from there (scalar loads), later phases from the sub-transform's
// own 2^K entries in LDS (entry 2^s + lg, see stage_twiddles), whose latency is a few dozen
// cycles where a table load in the middle of a pass takes hundreds.
// UNIFORM: g is the same in every lane, and so are the first phase's twiddles.
template <int LOGN, bool INV, class W2, bool UNIFORM = true>
struct GlobalTw {
    static constexpr bool uniform = UNIFORM;
    const W2 *tw;
    int g, L0;
    template <bool FIRST>
    __device__ __forceinline__ W2 at(int s, int lg) const {
        const int l = L0 + s, grp = (g << s) + lg;
        return load_tw(tw, INV ? (1 << LOGN) - (2 << l) + 1 + grp : (1 << l) + grp);
    }
};
template <int LOGN, class W2>
struct TileTw {
    static constexpr bool uniform = true;
    const W2 *tw;
    int g, L0;
    const W2 *lds;
    template <bool FIRST>
    __device__ __forceinline__ W2 at(int s, int lg) const {
        if constexpr (FIRST) return load_tw(tw, (1 << (L0 + s)) + (g << s) + lg);
        else return lds[(1 << s) + lg];
    }
};
// Entry 2^s + lg of lds (2^K entries) = the forward twiddle of local layer s, group lg of
// sub-transform g at layer L0 (entry 0 unused).  No barrier.
template <int K, class W2>
__device__ __forceinline__ void stage_twiddles(W2 *lds, const W2 *tw, int g, int L0, int tid, int threads) {
    for (int e = tid; e < (1 << K); e += threads) {
        const int s = e ? 31 - __clz(e) : 0;
        lds[e] = load_tw(tw, e ? (1 << (L0 + s)) + (g << s) + (e - (1 << s)) : 1);
    }
}

// One phase on the thread's registers.  W selects the wide forward schedule (q < 2^60).
template <int K, int E, int S0, int EP, bool INV, bool W, class Tw>
__device__ __forceinline__ void phase_compute(uint64_t (&r)[1 << E], int t, const Tw &tw, const BfConst &bc) {
#pragma unroll
    for (int ss = 0; ss < EP; ss++) {
        const int s = INV ? (S0 + EP - 1 - ss) : (S0 + ss);
        const int b = S0 + EP - 1 - s;
#pragma unroll
        for (int j = 0; j < (1 << E); j++) {
            if (j & (1 << b)) continue;
            // in the first phase a register's group does not depend on the thread (its
            // index bits above K - s all come from j): with t = 0 it is a constant, so
            // the twiddle address is uniform and the load scalar
            const int idx = phase_index<K, E, S0, EP>(S0 == 0 ? 0 : t, j);
            const ulonglong2 w = tw.template at<S0 == 0>(s, idx >> (K - s));
            const bool red = !W || (s >= 2 && !(s & 1));
            butterfly<INV, S0 == 0 && Tw::uniform>(r[j], r[j | (1 << b)], w, bc.four_q, bc.neg_q, red, W ? bc.neg_eight_q : bc.neg_four_q);
        }
    }
}

// Runs all phases of a sub-transform.  The first phase reads its registers straight
// from global memory through `load(idx, j)` (j: the register) and the last writes them
// back through
// `store(idx, value)` or `store(idx, value, j)`; in between, values cross threads through LDS at `addr(idx)`,
// so a pass makes one LDS round trip per phase boundary and one barrier each.
template <int K, int E, bool INV, bool W, int P = 0, class Addr, class Load, class Store, class Tw>
__device__ __forceinline__ void run_phases(uint64_t *tile, const Addr &addr, const Load &load, const Store &store,
                                           int t, const Tw &tw, const BfConst &bc, bool active) {
    constexpr int NP = (K + E - 1) / E;
    if constexpr (P < NP) {
        // forward runs phases from layer 0 upwards, inverse from the top layer down
        constexpr int PI = INV ? (NP - 1 - P) : P;
        constexpr int S0 = PI * E;
        constexpr int EP = (S0 + E <= K) ? E : (K - S0);
        uint64_t r[1 << E];
        if (active) {
#pragma unroll
            for (int j = 0; j < (1 << E); j++) {
                const int idx = phase_index<K, E, S0, EP>(t, j);
                r[j] = P == 0 ? load(idx, j) : tile[addr(idx)];
            }
            phase_compute<K, E, S0, EP, INV, W>(r, t, tw, bc);
#pragma unroll
            for (int j = 0; j < (1 << E); j++) {
                const int idx = phase_index<K, E, S0, EP>(t, j);
                if constexpr (P == NP - 1) {
                    const uint64_t v = W ? sub_if_ge_neg(r[j], bc.neg_eight_q) : r[j];  // wide: [0,16q) -> [0,8q)
                    if constexpr (std::is_invocable_v<Store, int, uint64_t, int>) store(idx, v, j);
                    else store(idx, v);
                } else {
                    tile[addr(idx)] = r[j];
                }
            }
        }
        if constexpr (P + 1 < NP) {
            __syncthreads();
            run_phases<K, E, INV, W, P + 1>(tile, addr, load, store, t, tw, bc, active);
        }
    }
}

// ---- the same phases in fp64, forward, for primes below 2^50 (butterfly_fp.h) --------
// The tile holds the doubles' bits.  ROWS picks the layers that reduce x first.
struct FpConst {
    double q, qinv;
};

template <int K, int E, int S0, int EP, bool ROWS, class Tw>
__device__ __forceinline__ void phase_compute_fp(double (&r)[1 << E], int t, const Tw &tw, const FpConst &fc) {
#pragma unroll
    for (int ss = 0; ss < EP; ss++) {
        const int s = S0 + ss;
        const int b = S0 + EP - 1 - s;
#pragma unroll
        for (int j = 0; j < (1 << E); j++) {
            if (j & (1 << b)) continue;
            const int idx = phase_index<K, E, S0, EP>(S0 == 0 ? 0 : t, j);
            fp_butterfly(r[j], r[j | (1 << b)], tw.template at<S0 == 0>(s, idx >> (K - s)), fc.q, fc.qinv,
                         fp_centers(ROWS, K, s));
        }
    }
}

// load(idx, j) and store(idx, value) take doubles.
template <int K, int E, bool ROWS, int P = 0, class Addr, class Load, class Store, class Tw>
__device__ __forceinline__ void run_phases_fp(uint64_t *tile, const Addr &addr, const Load &load, const Store &store,
                                              int t, const Tw &tw, const FpConst &fc, bool active) {
    constexpr int NP = (K + E - 1) / E;
    if constexpr (P < NP) {
        constexpr int S0 = P * E;
        constexpr int EP = (S0 + E <= K) ? E : (K - S0);
        double r[1 << E];
        if (active) {
#pragma unroll
            for (int j = 0; j < (1 << E); j++) {
                const int idx = phase_index<K, E, S0, EP>(t, j);
                r[j] = P == 0 ? load(idx, j) : __longlong_as_double((long long)tile[addr(idx)]);
            }
            phase_compute_fp<K, E, S0, EP, ROWS>(r, t, tw, fc);
#pragma unroll
            for (int j = 0; j < (1 << E); j++) {
                const int idx = phase_index<K, E, S0, EP>(t, j);
                if (P == NP - 1) store(idx, r[j]);
                else tile[addr(idx)] = (uint64_t)__double_as_longlong(r[j]);
            }
        }
        if constexpr (P + 1 < NP) {
            __syncthreads();
            run_phases_fp<K, E, ROWS, P + 1>(tile, addr, load, store, t, tw, fc, active);
        }
    }
}

// LDS slot of element idx of a row of 2^K words: one pad word after every 16, so that both
// the "stride 16" and the "16 consecutive" phase patterns hit distinct banks, and a
// register's address is a per-thread base plus a constant (an XOR swizzle, which needs no
// pad, costs an address register per element: 32 of the fused key-product kernel's).
__host__ __device__ constexpr int row_slot(int idx) { return idx + (idx >> 4); }
__host__ __device__ constexpr int row_words(int K) { return (1 << K) + (1 << K >> 4); }

// Final touch of a value leaving the last pass: forward [0, 8q) -> [0, 4q) (lazy) or
// [0, q); inverse [0, 4q) times N^-1 (exact Shoup) -> [0, 2q) (lazy) or [0, q).
template <bool INV, bool FULL>
__device__ __forceinline__ uint64_t finish(uint64_t x, const DevPrime &P) {
    if (!INV) {
        const uint64_t four_q = P.q << 2;
        x = x >= four_q ? x - four_q : x;
        if (FULL) {
            x = x >= P.two_q ? x - P.two_q : x;
            x = x >= P.q ? x - P.q : x;
        }
    } else {
        x = shoup_lazy(x, P.inv_n, P.inv_n_shoup, P.q);
        if (FULL) x = x >= P.q ? x - P.q : x;
    }
    return x;
}

// Rows pass: one block takes row g (the last K layers; the whole limb when K == LOGN)
// of SUBS limbs that share prime i -- limbs (i, j) for SUBS consecutive j -- so every
// row in the block uses the same twiddles (broadcast loads, L1/L2 hits).  Blocks run
// with the limb group fastest, so consecutive blocks also share them.  jn_short != 0:
// primes i < I - 1 have only jn_short limbs (the grid is sized for jn).
// MX (fewer than SUBS limbs per prime, e.g. one ciphertext, or 5 for blocks of 4): a block
// takes SUBS (limb, row) pairs of prime i instead, limb fastest, so that its threads are not
// idle; the rows of a block then differ and so do their twiddles, which costs more than a
// second block with two rows or more of its four (forward transforms of 5 and 7 polynomials at
// N = 2^16, L = 12: 42.9 -> 38.6 us and 2% more; 5 at N = 2^15, L = 15 30.5 -> 27.7; 9 for blocks of
// 8 at N = 2^13, L = 4 2% more).
template <int LOGN, int K, int E, int SUBS>
__host__ __device__ constexpr uint32_t rows_blocks_per_prime(uint32_t jn, bool mx) {
    return mx ? ((jn << (LOGN - K)) + SUBS - 1) / SUBS : (1u << (LOGN - K)) * ((jn + SUBS - 1) / SUBS);
}
template <int LOGN, int K, int SUBS>
__host__ __device__ constexpr bool rows_mixed(uint32_t jn) {
    return LOGN > K && (jn < (uint32_t)SUBS || (SUBS == 4 && jn == 5));
}

// (tile: SUBS * row_words(K) words of LDS, the caller's)
template <int LOGN, int K, int E, int SUBS, bool INV, bool W = false, bool MX = false, class Load, class Store>
__device__ __forceinline__ void rows_body_t(uint64_t *tile, uint32_t bid, const DevPrime *__restrict__ primes,
                                            uint32_t I, uint32_t j0, uint32_t jn, const Load &load_elem,
                                            const Store &store_elem, uint32_t jn_short = 0) {
    constexpr int T = 1 << (K - E);
    constexpr int SZ = 1 << K;
    constexpr int RPL = LOGN - K;  // log2(rows per limb)
    constexpr int NP = (K + E - 1) / E;
    static_assert(!MX || (NP > 1 && RPL > 0), "pairs of (limb, row) need rows and a staged store");
    const int tid = threadIdx.x;
    const int sub = tid / T, t = tid % T;
    uint32_t i, jfirst = 0, q0 = 0;
    int g, nsub;
    bool active;
    uint32_t j;
    if constexpr (MX) {
        const uint32_t per = rows_blocks_per_prime<LOGN, K, E, SUBS>(jn, true);
        i = bid / per;
        q0 = (bid % per) * SUBS;
        nsub = (int)min<uint32_t>(SUBS, (jn << RPL) - q0);
        active = sub < nsub;
        const uint32_t q = q0 + (uint32_t)(active ? sub : 0);
        j = j0 + q % jn;
        g = (int)(q / jn);
    } else {
        const uint32_t jc_count = (jn + SUBS - 1) / SUBS;
        const uint32_t jc = bid % jc_count;
        const uint32_t r = bid / jc_count;
        g = (int)(r & ((1u << RPL) - 1));
        i = r >> RPL;
        jfirst = j0 + jc * SUBS;
        const uint32_t jend = j0 + (jn_short && i + 1 < I ? jn_short : jn);
        if (jfirst >= jend) return;  // uniform: a whole block past a short row
        nsub = (int)min<uint32_t>(SUBS, jend - jfirst);
        active = sub < nsub;
        j = jfirst + (uint32_t)(active ? sub : 0);
    }
    const size_t row_off = (size_t)g << K;
    const DevPrime &P = primes[i];
    const GlobalTw<LOGN, INV, ulonglong2, !MX> tw{INV ? P.inv : P.fwd, g, RPL};
    auto addr = [sub](int idx) { return sub * row_words(K) + row_slot(idx); };
    auto load = [&](int idx, int) { return load_elem(i, j, row_off + idx); };
    if constexpr (NP == 1) {
        auto store = [&](int idx, uint64_t x) { store_elem(i, j, row_off + idx, x); };
        run_phases<K, E, INV, W>(tile, addr, load, store, t, tw, bf_const(P), active);
    } else {
        // the last phase leaves 16 consecutive values per thread; stage them in LDS so
        // that the block writes whole rows with consecutive lanes on consecutive words
        auto stage = [&](int idx, uint64_t x) { tile[addr(idx)] = x; };
        run_phases<K, E, INV, W>(tile, addr, load, stage, t, tw, bf_const(P), active);
        __syncthreads();
        if constexpr (MX) {
            for (int e = tid; e < nsub * SZ; e += SUBS * T) {
                const int sb = e / SZ, off = e % SZ;
                const uint32_t q = q0 + (uint32_t)sb;
                store_elem(i, j0 + q % jn, ((size_t)(q / jn) << K) + off, tile[sb * row_words(K) + row_slot(off)]);
            }
        } else if (nsub == SUBS) {
            // a full block: a fixed number of elements per thread, unrolled so that every
            // row's base address is uniform (scalar) and only the offset varies by lane
            constexpr int PER = SUBS * SZ / (SUBS * T);
#pragma unroll
            for (int k = 0; k < PER; k++) {
                const int e = tid + k * SUBS * T;
                const int sb = e / SZ, off = e % SZ;
                store_elem(i, jfirst + (uint32_t)sb, row_off + off, tile[sb * row_words(K) + row_slot(off)]);
            }
        } else {
            for (int e = tid; e < nsub * SZ; e += SUBS * T) {
                const int sb = e / SZ, off = e % SZ;
                store_elem(i, jfirst + (uint32_t)sb, row_off + off, tile[sb * row_words(K) + row_slot(off)]);
            }
        }
    }
}

template <int LOGN, int K, int E, int SUBS, bool INV, bool W = false, bool MX = false, class Load, class Store>
__device__ __forceinline__ void rows_body(uint32_t bid, const DevPrime *__restrict__ primes, uint32_t I, uint32_t j0,
                                          uint32_t jn, const Load &load_elem, const Store &store_elem,
                                          uint32_t jn_short = 0) {
    constexpr int NP = (K + E - 1) / E;
    __shared__ uint64_t tile[NP > 1 ? SUBS * row_words(K) : 1];
    rows_body_t<LOGN, K, E, SUBS, INV, W, MX>(tile, bid, primes, I, j0, jn, load_elem, store_elem, jn_short);
}

// Columns pass: SUBS adjacent columns of one limb per block; a column is the first
// K layers of the limb (stride 2^(LOGN-K) between its values).
// Blocks run limb (i, j) by limb with j fastest, or with i fastest when I_FAST (then I
// is the prime count) -- the order for loads shared by all primes of one j.
template <int LOGN, int K, int E, int SUBS, bool INV, bool I_FAST = false, class Load, class Store>
__device__ __forceinline__ void cols_body_t(uint64_t *tile, uint32_t bid, const DevPrime *__restrict__ primes,
                                            uint32_t j0, uint32_t jn, const Load &load_elem, const Store &store_elem,
                                            uint32_t I = 1) {
    constexpr int C = 1 << (LOGN - K);
    constexpr int TILES = C / SUBS;
    const int tid = threadIdx.x;
    const int col = tid % SUBS, t = tid / SUBS;
    const uint32_t r = bid / TILES;
    const size_t c = (size_t)(bid % TILES) * SUBS + col;
    const uint32_t i = I_FAST ? r % I : r / jn, j = j0 + (I_FAST ? r / I : r % jn);
    const DevPrime &P = primes[i];
    const GlobalTw<LOGN, INV, ulonglong2> tw{INV ? P.inv : P.fwd, 0, 0};
    auto addr = [col](int idx) { return idx * SUBS + col; };
    auto load = [&](int idx, int) { return load_elem(i, j, (size_t)idx * C + c); };
    auto store = [&](int idx, uint64_t x) { store_elem(i, j, (size_t)idx * C + c, x); };
    run_phases<K, E, INV, false>(tile, addr, load, store, t, tw, bf_const(P), true);
}

template <int LOGN, int K, int E, int SUBS, bool INV, bool I_FAST = false, class Load, class Store>
__device__ __forceinline__ void cols_body(uint32_t bid, const DevPrime *__restrict__ primes, uint32_t j0, uint32_t jn,
                                          const Load &load_elem, const Store &store_elem, uint32_t I = 1) {
    __shared__ uint64_t tile[SUBS << K];
    cols_body_t<LOGN, K, E, SUBS, INV, I_FAST>(tile, bid, primes, j0, jn, load_elem, store_elem, I);
}

__device__ __forceinline__ uint32_t group_of(const uint32_t *start, uint32_t n, uint32_t b) {
    uint32_t g = 0;
#pragma unroll 1
    while (g + 1 < n && b >= start[g + 1]) g++;
    return g;
}

// Plain in-place passes over a LimbGrid buffer.
struct GridAccess {
    uint64_t *data;
    LimbGrid lg;
    int logn;
    __device__ uint64_t *at(uint32_t i, uint32_t j, size_t off) const {
        return data + ((size_t)(i * lg.A + j * lg.B) << logn) + off;
    }
};

template <int LOGN, int K, int E, int SUBS, bool INV, bool LAST, bool FULL, bool MX = false>
__global__ __launch_bounds__(SUBS << (K - E)) void ntt_rows_kernel(uint64_t *__restrict__ data,
                                                                  const DevPrime *__restrict__ primes, LimbGrid lg,
                                                                  uint32_t j0, uint32_t jn) {
    const GridAccess g{data, lg, LOGN};
    rows_body<LOGN, K, E, SUBS, INV, false, MX>(
        blockIdx.x, primes, lg.I, j0, jn, [&](uint32_t i, uint32_t j, size_t off) { return *g.at(i, j, off); },
        [&](uint32_t i, uint32_t j, size_t off, uint64_t x) {
            *g.at(i, j, off) = LAST ? finish<INV, FULL>(x, primes[i]) : x;
        });
}

template <int LOGN, int K, int E, int SUBS, bool INV, bool LAST, bool FULL>
__global__ __launch_bounds__(SUBS << (K - E)) void ntt_cols_kernel(uint64_t *__restrict__ data,
                                                                  const DevPrime *__restrict__ primes, LimbGrid lg,
                                                                  uint32_t j0, uint32_t jn) {
    const GridAccess g{data, lg, LOGN};
    cols_body<LOGN, K, E, SUBS, INV>(
        blockIdx.x, primes, j0, jn, [&](uint32_t i, uint32_t j, size_t off) { return *g.at(i, j, off); },
        [&](uint32_t i, uint32_t j, size_t off, uint64_t x) {
            *g.at(i, j, off) = LAST ? finish<INV, FULL>(x, primes[i]) : x;
        });
}

// Rows pass of a transform whose input lies elsewhere: reads limb (i, j) from `src`
// (grid slg) and writes it to `data` (grid lg), same shape.
template <int LOGN, int K, int E, int SUBS, bool INV, bool LAST, bool FULL, bool MX = false>
__global__ __launch_bounds__(SUBS << (K - E)) void ntt_rows_from_kernel(const uint64_t *__restrict__ src,
                                                                       LimbGrid slg, uint64_t *__restrict__ data,
                                                                       const DevPrime *__restrict__ primes,
                                                                       LimbGrid lg, uint32_t j0, uint32_t jn) {
    const GridAccess g{data, lg, LOGN};
    const GridAccess s{const_cast<uint64_t *>(src), slg, LOGN};
    rows_body<LOGN, K, E, SUBS, INV, false, MX>(
        blockIdx.x, primes, lg.I, j0, jn, [&](uint32_t i, uint32_t j, size_t off) { return *s.at(i, j, off); },
        [&](uint32_t i, uint32_t j, size_t off, uint64_t x) {
            *g.at(i, j, off) = LAST ? finish<INV, FULL>(x, primes[i]) : x;
        });
}

// Block prefix table of a grouped launch; sizes[g] blocks for group g.
template <class Table>
uint32_t fill_starts(Table &t, const std::vector<uint64_t> &sizes) {
    uint64_t acc = 0;
    t.n = (uint32_t)sizes.size();
    for (size_t g = 0; g < sizes.size(); g++) {
        t.start[g] = (uint32_t)acc;
        acc += sizes[g];
    }
    t.start[sizes.size()] = (uint32_t)acc;
    if (acc >= GROUPED_BLOCKS) fail(ERR_INVALID_ARGUMENT, "grouped launch too large");
    return (uint32_t)acc;
}

// The passes' shape at one degree: the first K1 layers along columns (CS columns per block),
// the last K2 inside rows (RS rows per block), 2^E values per thread.  Large launches take 16
// values per thread (fewest LDS round trips and twiddle loads).  SMALL ones take 4: with few
// waves per SIMD a pass is one wave's latency, of which a quarter is left.  A product, its
// relinearization and rescale of one ciphertext at N = 2^13, L = 3 took 102.6 us with 16
// values and takes 54.4 with 4; 37 of them at N = 2^14, L = 7 645 and 581 us; a chain round
// over 64 at N = 2^15 7.41 and 6.82 ms.  The line lies at 2^26 words (1,024 limbs of 2^16):
// beyond it the forms differ by under 1% (encryption) or 16 values win (decryption of 128
// ciphertexts at N = 2^16, L = 24: 3.13 against 3.26 ms).  (The transforms in place have lines
// of their own, ntt.hip.)  N = 2^17 and the launches of several degrees are not compiled in the
// small form; measured there, it would win for one or two ciphertexts (relinearization of one
// at L = 2 93 -> 61 us, L = 8 213 -> 183, L = 24 1,132 -> 1,100) and is even at four.
constexpr uint64_t SMALL_WORDS = uint64_t(1) << 26;
template <int LOGN, bool SMALL>
struct PassShape {
    static constexpr int K1 = LOGN / 2;
    static constexpr int K2 = LOGN - K1;
    static constexpr int E = SMALL ? 2 : 4;
    static constexpr int CS = 16;
    static constexpr int RS = SMALL ? 256 >> (K2 - E) : (4096 >> K2) < 1 ? 1 : 4096 >> K2;
};
// f(std::true_type) for a small launch over `limbs` limbs, else f(std::false_type).
template <int LOGN, class F>
void with_shape(uint64_t limbs, F &&f, uint64_t line = SMALL_WORDS) {
    if constexpr (LOGN <= 16) {
        if (limbs << LOGN <= line) {
            f(std::true_type{});
            return;
        }
    }
    f(std::false_type{});
}

// f(std::true_type / std::false_type) for a run-time flag.
template <class F>
void with_bool(bool b, F &&f) {
    if (b) f(std::true_type{});
    else f(std::false_type{});
}

}  // namespace
}  // namespace shc

// ntt.hip -- batched negacyclic NTT / inverse NTT for gfx950.
//
// Same transform as the reference's nttNegacyclicHarvey / inverseNttNegacyclicHarvey
// (src/utils/ntt.cpp:158-213, src/utils/dwthandler.h:88-372; GPU launchers
// src/kernelutils.cu:330-476), scheduled for CDNA4 instead of one launch per layer:
//
//   * A length-2^logn limb is viewed as a 2^K1 x 2^K2 matrix.  The first K1 layers
//     act along columns, the last K2 layers inside contiguous rows, so a forward
//     transform is two kernels (columns pass, rows pass) and each reads and writes
//     the limb once.  Up to 2^12 points the whole limb is one tile (one kernel).
//   * A tile lives in LDS; each thread pulls 2^E values into VGPRs and runs E
//     butterfly layers there before writing them back, so one LDS round trip
//     covers E layers.
//   * Harvey-style lazy butterflies with Shoup twiddles keep values in [0,8q)
//     (forward) or [0,4q) (inverse); the twiddle product uses a quotient estimate
//     that may be low by up to 2 (9 32-bit multiplies instead of 10), which those
//     wider ranges absorb.  The full reduction and the N^-1 scaling are folded into
//     the store of the last pass.
//   * The key switch's ModUp transforms take the wide schedule, which needs q < 2^60
//     (contexts hold only such primes): values may grow to 16q inside a pass (local
//     layers 0, 1 and odd layers skip the conditional subtraction, even layers >= 2
//     subtract 8q) and one subtraction of 8q at the end of the pass brings them back
//     below 8q, so passes still hand each other [0, 8q).
//
// Twiddle indexing: forward layer l (m = 2^l groups) uses root_powers[m + group];
// inverse layer l uses inv_root_powers[N - 2m + 1 + group], group = x >> (logn - l).
#include "ntt_device.h"

namespace shc {
namespace {

template <int LOGN, bool INV, bool FULL, bool SMALL>
void launch_ntt_as(uint64_t *data, LimbGrid lg, uint32_t j0, uint32_t jn, const DevPrime *primes, hipStream_t st) {
    if constexpr (LOGN <= 12) {
        constexpr int K = LOGN;
        constexpr int E = K < 4 ? K : 4;
        constexpr int T = 1 << (K - E);
        constexpr int SUBS = (T >= 256) ? 1 : (256 / T);
        const uint32_t blocks = lg.I * ((jn + SUBS - 1) / SUBS);
        ntt_rows_kernel<LOGN, K, E, SUBS, INV, true, FULL><<<blocks, SUBS * T, 0, st>>>(data, primes, lg, j0, jn);
    } else {
        using S = PassShape<LOGN, SMALL>;
        constexpr int K1 = S::K1, K2 = S::K2, E = S::E, CS = S::CS, RS = S::RS;
        const uint32_t col_blocks = lg.I * jn * ((1u << K2) / CS);
        const bool mx = rows_mixed<LOGN, K2, RS>(jn);
        const uint32_t row_blocks = lg.I * rows_blocks_per_prime<LOGN, K2, E, RS>(jn, mx);
        if (!INV) {
            ntt_cols_kernel<LOGN, K1, E, CS, false, false, FULL>
                <<<col_blocks, CS << (K1 - E), 0, st>>>(data, primes, lg, j0, jn);
            if (mx)
                ntt_rows_kernel<LOGN, K2, E, RS, false, true, FULL, true>
                    <<<row_blocks, RS << (K2 - E), 0, st>>>(data, primes, lg, j0, jn);
            else
                ntt_rows_kernel<LOGN, K2, E, RS, false, true, FULL, false>
                    <<<row_blocks, RS << (K2 - E), 0, st>>>(data, primes, lg, j0, jn);
        } else {
            if (mx)
                ntt_rows_kernel<LOGN, K2, E, RS, true, false, FULL, true>
                    <<<row_blocks, RS << (K2 - E), 0, st>>>(data, primes, lg, j0, jn);
            else
                ntt_rows_kernel<LOGN, K2, E, RS, true, false, FULL, false>
                    <<<row_blocks, RS << (K2 - E), 0, st>>>(data, primes, lg, j0, jn);
            ntt_cols_kernel<LOGN, K1, E, CS, true, true, FULL>
                <<<col_blocks, CS << (K1 - E), 0, st>>>(data, primes, lg, j0, jn);
        }
    }
}

// The line of the transforms in place, which do nothing beside their butterflies: forward ones
// wait less on memory, and 16 values per thread win earlier.  16 / 4 values in us: forward, one
// prime at N = 2^16: 2^22 words 38.0 / 36.9, 2^23 63.0 / 64.8, 2^24 113 / 123, 2^26 (62.5 M) 464 /
// 552; N = 2^13, L = 4: 2^23 58.9 / 57.3, 2^24 102.7 / 107.3.  Inverse, N = 2^16: 2^23 69.4 /
// 65.7, 2^24 121.6 / 126.6, 62.5 M 512 / 554; N = 2^13: 2^24 111.5 / 107.7, 2^25 220 / 224.
// (Polynomials count in fours, a block's rows: 5 at N = 2^16, L = 24 68.7 / 74.3.)  Where 16 values'
// blocks of rows (16 of them at N = 2^15 and 2^16, 32 below) would idle for too many rows that are
// not there, 4 values go on to SMALL_WORDS: N = 2^16, L = 24, forward 17 polynomials 218 / 204, 20
// 242 / 238, 24 301 / 312; inverse 17 250 / 208, 20 278 / 245, 24 363 / 316, 26 377 / 347, 28 387 / 370.
constexpr uint64_t NTT_SMALL_WORDS = (uint64_t(1) << 23) - 1;
constexpr uint64_t INTT_SMALL_WORDS = (uint64_t(1) << 24) - 1;

template <int LOGN, bool INV>
uint64_t in_place_line(uint32_t jn) {
    constexpr uint32_t RS = PassShape<LOGN, false>::RS;
    const uint64_t rows = (uint64_t)((jn + RS - 1) / RS) * RS;
    const bool ragged = jn >= RS && 16 * (uint64_t)jn <= (INV ? 13 : 10) * rows;
    return ragged ? SMALL_WORDS : INV ? INTT_SMALL_WORDS : NTT_SMALL_WORDS;
}

template <int LOGN, bool INV, bool FULL>
void launch_ntt(uint64_t *data, LimbGrid lg, uint32_t j0, uint32_t jn, const DevPrime *primes, hipStream_t st) {
    if constexpr (LOGN <= 12)
        launch_ntt_as<LOGN, INV, FULL, false>(data, lg, j0, jn, primes, st);
    else
        with_shape<LOGN>((uint64_t)lg.I * (jn < 4 ? jn : (jn + 3) & ~3u), [&](auto s) {
            launch_ntt_as<LOGN, INV, FULL, decltype(s)::value>(data, lg, j0, jn, primes, st);
        }, in_place_line<LOGN, INV>(jn));
}

// Inverse transform of src's limbs into data (rows pass from src, columns pass in place).
template <int LOGN, bool FULL, bool SMALL>
void launch_inverse_from_as(const uint64_t *src, LimbGrid slg, uint64_t *data, LimbGrid lg, uint32_t j0, uint32_t jn,
                         const DevPrime *primes, hipStream_t st) {
    if constexpr (LOGN <= 12) {
        constexpr int K = LOGN;
        constexpr int E = K < 4 ? K : 4;
        constexpr int T = 1 << (K - E);
        constexpr int SUBS = (T >= 256) ? 1 : (256 / T);
        const uint32_t blocks = lg.I * ((jn + SUBS - 1) / SUBS);
        ntt_rows_from_kernel<LOGN, K, E, SUBS, true, true, FULL>
            <<<blocks, SUBS * T, 0, st>>>(src, slg, data, primes, lg, j0, jn);
    } else {
        using S = PassShape<LOGN, SMALL>;
        constexpr int K1 = S::K1, K2 = S::K2, E = S::E, CS = S::CS, RS = S::RS;
        const uint32_t col_blocks = lg.I * jn * ((1u << K2) / CS);
        const bool mx = rows_mixed<LOGN, K2, RS>(jn);
        const uint32_t row_blocks = lg.I * rows_blocks_per_prime<LOGN, K2, E, RS>(jn, mx);
        if (mx)
            ntt_rows_from_kernel<LOGN, K2, E, RS, true, false, FULL, true>
                <<<row_blocks, RS << (K2 - E), 0, st>>>(src, slg, data, primes, lg, j0, jn);
        else
            ntt_rows_from_kernel<LOGN, K2, E, RS, true, false, FULL, false>
                <<<row_blocks, RS << (K2 - E), 0, st>>>(src, slg, data, primes, lg, j0, jn);
        ntt_cols_kernel<LOGN, K1, E, CS, true, true, FULL>
            <<<col_blocks, CS << (K1 - E), 0, st>>>(data, primes, lg, j0, jn);
    }
}

template <int LOGN, bool FULL>
void launch_inverse_from(const uint64_t *src, LimbGrid slg, uint64_t *data, LimbGrid lg, uint32_t j0, uint32_t jn,
                         const DevPrime *primes, hipStream_t st) {
    if constexpr (LOGN <= 12)
        launch_inverse_from_as<LOGN, FULL, false>(src, slg, data, lg, j0, jn, primes, st);
    else
        with_shape<LOGN>((uint64_t)lg.I * jn, [&](auto s) {
            launch_inverse_from_as<LOGN, FULL, decltype(s)::value>(src, slg, data, lg, j0, jn, primes, st);
        });
}

template <bool FULL>
void dispatch_inverse_from(const uint64_t *src, LimbGrid slg, uint64_t *data, LimbGrid lg, const DevPrime *primes,
                           int logn, hipStream_t st) {
    if (logn < 1 || logn > 17) fail(ERR_INVALID_ARGUMENT, "poly_modulus_degree must be 2^1 .. 2^17");
    if (slg.I != lg.I || slg.J != lg.J) fail(ERR_LOGIC, "transform source and destination shapes differ");
    if ((uint64_t)lg.I * lg.J == 0) return;
    for (const LimbGrid &g : {slg, lg})
        if ((uint64_t)(g.I - 1) * g.A + (uint64_t)(g.J - 1) * g.B > UINT32_MAX)
            fail(ERR_INVALID_ARGUMENT, "too many limbs for one transform call");
    const uint64_t max_limbs = (uint64_t(1) << 34) >> logn;
    if (lg.I > max_limbs) fail(ERR_INVALID_ARGUMENT, "too many primes for one transform call");
    const uint32_t step = (uint32_t)(max_limbs / lg.I < lg.J ? max_limbs / lg.I : lg.J);
    for (uint32_t j0 = 0; j0 < lg.J; j0 += step) {
        const uint32_t jn = lg.J - j0 < step ? lg.J - j0 : step;
        switch (logn) {
#define SHC_NTT_CASE(L) \
    case L: launch_inverse_from<L, FULL>(src, slg, data, lg, j0, jn, primes, st); break;
            SHC_NTT_CASE(1) SHC_NTT_CASE(2) SHC_NTT_CASE(3) SHC_NTT_CASE(4) SHC_NTT_CASE(5) SHC_NTT_CASE(6)
            SHC_NTT_CASE(7) SHC_NTT_CASE(8) SHC_NTT_CASE(9) SHC_NTT_CASE(10) SHC_NTT_CASE(11) SHC_NTT_CASE(12)
            SHC_NTT_CASE(13) SHC_NTT_CASE(14) SHC_NTT_CASE(15) SHC_NTT_CASE(16) SHC_NTT_CASE(17)
#undef SHC_NTT_CASE
        }
        launch_check("ntt launch");
    }
}

template <bool INV, bool FULL>
void dispatch_chunk(uint64_t *data, LimbGrid lg, uint32_t j0, uint32_t jn, const DevPrime *primes, int logn,
                    hipStream_t st) {
    switch (logn) {
#define SHC_NTT_CASE(L) \
    case L: launch_ntt<L, INV, FULL>(data, lg, j0, jn, primes, st); break;
        SHC_NTT_CASE(1) SHC_NTT_CASE(2) SHC_NTT_CASE(3) SHC_NTT_CASE(4) SHC_NTT_CASE(5) SHC_NTT_CASE(6)
        SHC_NTT_CASE(7) SHC_NTT_CASE(8) SHC_NTT_CASE(9) SHC_NTT_CASE(10) SHC_NTT_CASE(11) SHC_NTT_CASE(12)
        SHC_NTT_CASE(13) SHC_NTT_CASE(14) SHC_NTT_CASE(15) SHC_NTT_CASE(16) SHC_NTT_CASE(17)
#undef SHC_NTT_CASE
        default: fail(ERR_INVALID_ARGUMENT, "poly_modulus_degree must be 2^1 .. 2^17");
    }
    launch_check("ntt launch");
}

// Splits very large batches over j so that one launch covers at most 2^34 / N limbs
// (every pass runs N/16 work-items per limb, so a launch stays below 2^30).
template <bool INV, bool FULL>
void dispatch(uint64_t *data, LimbGrid lg, const DevPrime *primes, int logn, hipStream_t st) {
    if (logn < 1 || logn > 17) fail(ERR_INVALID_ARGUMENT, "poly_modulus_degree must be 2^1 .. 2^17");
    if ((uint64_t)lg.I * lg.J == 0) return;
    if ((uint64_t)(lg.I - 1) * lg.A + (uint64_t)(lg.J - 1) * lg.B > UINT32_MAX)
        fail(ERR_INVALID_ARGUMENT, "too many limbs for one transform call");
    const uint64_t max_limbs = (uint64_t(1) << 34) >> logn;
    if (lg.I > max_limbs) fail(ERR_INVALID_ARGUMENT, "too many primes for one transform call");
    const uint32_t step = (uint32_t)(max_limbs / lg.I < lg.J ? max_limbs / lg.I : lg.J);
    for (uint32_t j0 = 0; j0 < lg.J; j0 += step) {
        const uint32_t jn = lg.J - j0 < step ? lg.J - j0 : step;
        dispatch_chunk<INV, FULL>(data, lg, j0, jn, primes, logn, st);
    }
}

LimbGrid poly_grid(uint32_t count, uint32_t lpp) {
    if (lpp == 0 || count % lpp) fail(ERR_INVALID_ARGUMENT, "limb count must be a multiple of limbs per polynomial");
    return LimbGrid{1, lpp, lpp, count / lpp};
}
}  // namespace

namespace {
__global__ void fp_tables_kernel(const DevPrime *__restrict__ primes, uint32_t n) {
    const DevPrime &P = primes[blockIdx.y];
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (!P.fwd_fp || i >= n) return;
    const int64_t w = (int64_t)P.fwd[i].x;
    const double c = (double)(2 * (uint64_t)w > P.q ? w - (int64_t)P.q : w);
    const_cast<double2 *>(P.fwd_fp)[i] = double2{c, c / (double)P.q};
}
}  // namespace

void build_fp_tables(const DevPrime *primes, uint32_t count, int logn, hipStream_t st) {
    const uint32_t n = 1u << logn;
    fp_tables_kernel<<<dim3((n + 255) / 256, count), 256, 0, st>>>(primes, n);
    launch_check("fp tables");
}

void ntt_forward(uint64_t *data, uint32_t count, uint32_t lpp, const DevPrime *primes, int logn, NttOut out,
                 hipStream_t st) {
    if (count == 0) return;
    ntt_forward_grid(data, poly_grid(count, lpp), primes, logn, out, st);
}

void ntt_forward_grid(uint64_t *data, LimbGrid lg, const DevPrime *primes, int logn, NttOut out, hipStream_t st) {
    if (out == NTT_FULL) dispatch<false, true>(data, lg, primes, logn, st);
    else dispatch<false, false>(data, lg, primes, logn, st);
}

void ntt_inverse(uint64_t *data, uint32_t count, uint32_t lpp, const DevPrime *primes, int logn, NttOut out,
                 hipStream_t st) {
    if (count == 0) return;
    ntt_inverse_grid(data, poly_grid(count, lpp), primes, logn, out, st);
}

void ntt_inverse_grid(uint64_t *data, LimbGrid lg, const DevPrime *primes, int logn, NttOut out, hipStream_t st) {
    if (out == NTT_FULL) dispatch<true, true>(data, lg, primes, logn, st);
    else dispatch<true, false>(data, lg, primes, logn, st);
}

void ntt_inverse_from(const uint64_t *src, LimbGrid src_grid, uint64_t *data, LimbGrid grid, const DevPrime *primes,
                      int logn, NttOut out, hipStream_t st) {
    if (out == NTT_FULL) dispatch_inverse_from<true>(src, src_grid, data, grid, primes, logn, st);
    else dispatch_inverse_from<false>(src, src_grid, data, grid, primes, logn, st);
}

}  // namespace shc

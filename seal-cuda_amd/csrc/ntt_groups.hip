// ntt_groups.hip -- transforms of several limb groups, levels and ring degrees in one launch
// per pass (the passes are those of ntt_device.h, the schedules ntt.hip's).
#include "ntt_device.h"

namespace shc {
namespace {

// Grouped transform passes: group g's limbs (i, j) of its grid, j < lg.J, all primes of
// its grid; the first pass of an inverse reads from src when the group has one.
struct NttGroupDev {
    uint64_t *data;
    const uint64_t *src;
    LimbGrid lg, slg;
    const DevPrime *primes;
};
struct NttGroups {
    uint32_t n;
    uint32_t start[MAX_GROUPS + 1];
    NttGroupDev g[MAX_GROUPS];
};

template <int LOGN, int K, int E, int SUBS, bool INV, bool LAST, bool FULL, bool MX>
__global__ __launch_bounds__(SUBS << (K - E)) void ntt_rows_grouped_kernel(NttGroups ng) {
    const uint32_t gi = group_of(ng.start, ng.n, blockIdx.x);
    const NttGroupDev &a = ng.g[gi];
    const GridAccess g{a.data, a.lg, LOGN};
    const GridAccess s{const_cast<uint64_t *>(a.src ? a.src : a.data), a.src ? a.slg : a.lg, LOGN};
    const DevPrime *primes = a.primes;
    rows_body<LOGN, K, E, SUBS, INV, false, MX>(
        blockIdx.x - ng.start[gi], primes, a.lg.I, 0, a.lg.J,
        [&](uint32_t i, uint32_t j, size_t off) { return *s.at(i, j, off); },
        [&](uint32_t i, uint32_t j, size_t off, uint64_t x) {
            *g.at(i, j, off) = LAST ? finish<INV, FULL>(x, primes[i]) : x;
        });
}

template <int LOGN, int K, int E, int SUBS, bool INV, bool LAST, bool FULL>
__global__ __launch_bounds__(SUBS << (K - E)) void ntt_cols_grouped_kernel(NttGroups ng) {
    const uint32_t gi = group_of(ng.start, ng.n, blockIdx.x);
    const NttGroupDev &a = ng.g[gi];
    const GridAccess g{a.data, a.lg, LOGN};
    const GridAccess s{const_cast<uint64_t *>(a.src ? a.src : a.data), a.src ? a.slg : a.lg, LOGN};
    const DevPrime *primes = a.primes;
    cols_body<LOGN, K, E, SUBS, INV>(
        blockIdx.x - ng.start[gi], primes, 0, a.lg.J, [&](uint32_t i, uint32_t j, size_t off) { return *s.at(i, j, off); },
        [&](uint32_t i, uint32_t j, size_t off, uint64_t x) {
            *g.at(i, j, off) = LAST ? finish<INV, FULL>(x, primes[i]) : x;
        });
}

// ---- Transforms over several ring degrees (N = 2^13 .. 2^17) in one launch per pass.
// Every degree runs 256-thread blocks over a 32 KB LDS tile -- the rows pass 4096 >> K2
// rows per block, the columns pass 4096 >> K1 columns -- so blocks of every degree share
// one kernel; a group's degree is uniform over its blocks.
struct NttMultiDev {
    NttGroupDev d;
    int32_t logn;
};
struct NttMulti {
    uint32_t n;
    uint32_t start[MAX_GROUPS + 1];
    NttMultiDev g[MAX_GROUPS];
};

template <int LOGN, bool INV, bool LAST, bool FULL>
__device__ __forceinline__ void rows_multi(uint64_t *tile, uint32_t bid, const NttGroupDev &a) {
    constexpr int K2 = LOGN - LOGN / 2;
    constexpr int RS = 4096 >> K2;
    const GridAccess g{a.data, a.lg, LOGN};
    const GridAccess s{const_cast<uint64_t *>(a.src ? a.src : a.data), a.src ? a.slg : a.lg, LOGN};
    const DevPrime *primes = a.primes;
    rows_body_t<LOGN, K2, 4, RS, INV>(
        tile, bid, primes, a.lg.I, 0, a.lg.J, [&](uint32_t i, uint32_t j, size_t off) { return *s.at(i, j, off); },
        [&](uint32_t i, uint32_t j, size_t off, uint64_t x) {
            *g.at(i, j, off) = LAST ? finish<INV, FULL>(x, primes[i]) : x;
        });
}

template <int LOGN, bool INV, bool LAST, bool FULL>
__device__ __forceinline__ void cols_multi(uint64_t *tile, uint32_t bid, const NttGroupDev &a) {
    constexpr int K1 = LOGN / 2;
    constexpr int CS = 4096 >> K1;
    const GridAccess g{a.data, a.lg, LOGN};
    const GridAccess s{const_cast<uint64_t *>(a.src ? a.src : a.data), a.src ? a.slg : a.lg, LOGN};
    const DevPrime *primes = a.primes;
    cols_body_t<LOGN, K1, 4, CS, INV>(
        tile, bid, primes, 0, a.lg.J, [&](uint32_t i, uint32_t j, size_t off) { return *s.at(i, j, off); },
        [&](uint32_t i, uint32_t j, size_t off, uint64_t x) {
            *g.at(i, j, off) = LAST ? finish<INV, FULL>(x, primes[i]) : x;
        });
}

template <bool INV, bool LAST, bool FULL>
__global__ __launch_bounds__(256) void ntt_rows_multi_kernel(NttMulti ng) {
    __shared__ uint64_t tile[4096 + 256];  // 4096 >> K2 rows of row_words(K2)
    const uint32_t gi = group_of(ng.start, ng.n, blockIdx.x);
    const NttMultiDev &m = ng.g[gi];
    const uint32_t bid = blockIdx.x - ng.start[gi];
    switch (m.logn) {  // uniform: the whole block
    case 13: rows_multi<13, INV, LAST, FULL>(tile, bid, m.d); break;
    case 14: rows_multi<14, INV, LAST, FULL>(tile, bid, m.d); break;
    case 15: rows_multi<15, INV, LAST, FULL>(tile, bid, m.d); break;
    case 16: rows_multi<16, INV, LAST, FULL>(tile, bid, m.d); break;
    default: rows_multi<17, INV, LAST, FULL>(tile, bid, m.d); break;
    }
}

template <bool INV, bool LAST, bool FULL>
__global__ __launch_bounds__(256) void ntt_cols_multi_kernel(NttMulti ng) {
    __shared__ uint64_t tile[4096];
    const uint32_t gi = group_of(ng.start, ng.n, blockIdx.x);
    const NttMultiDev &m = ng.g[gi];
    const uint32_t bid = blockIdx.x - ng.start[gi];
    switch (m.logn) {
    case 13: cols_multi<13, INV, LAST, FULL>(tile, bid, m.d); break;
    case 14: cols_multi<14, INV, LAST, FULL>(tile, bid, m.d); break;
    case 15: cols_multi<15, INV, LAST, FULL>(tile, bid, m.d); break;
    case 16: cols_multi<16, INV, LAST, FULL>(tile, bid, m.d); break;
    default: cols_multi<17, INV, LAST, FULL>(tile, bid, m.d); break;
    }
}

template <int LOGN, bool INV, bool FULL, bool SMALL>
void launch_ntt_groups_as(const NttGroup *gs, uint32_t n, hipStream_t st) {
    static_assert(LOGN > 12, "grouped transforms run the two-pass schedule");
    using S = PassShape<LOGN, SMALL>;
    constexpr int K1 = S::K1, K2 = S::K2, E = S::E, CS = S::CS, RS = S::RS;
    // the first pass reads src where a group has one; the second runs in place
    NttGroups cols{}, rows_mx{}, rows_full{};
    std::vector<uint64_t> csz, msz, fsz;
    for (uint32_t g = 0; g < n; g++) {
        const NttGroup &a = gs[g];
        const bool first_is_cols = !INV;
        NttGroupDev d{a.data, nullptr, a.lg, a.lg, a.primes};
        NttGroupDev d_first{a.data, a.src, a.lg, a.src ? a.slg : a.lg, a.primes};
        cols.g[csz.size()] = first_is_cols ? d_first : d;
        csz.push_back((uint64_t)a.lg.I * a.lg.J * ((1u << K2) / CS));
        const bool mx = rows_mixed<LOGN, K2, RS>(a.lg.J);
        const uint64_t rb = (uint64_t)a.lg.I * rows_blocks_per_prime<LOGN, K2, E, RS>(a.lg.J, mx);
        if (mx) {
            rows_mx.g[msz.size()] = first_is_cols ? d : d_first;
            msz.push_back(rb);
        } else {
            rows_full.g[fsz.size()] = first_is_cols ? d : d_first;
            fsz.push_back(rb);
        }
    }
    const uint32_t cb = fill_starts(cols, csz);
    auto rows = [&](bool last) {
        if (!msz.empty()) {
            const uint32_t b = fill_starts(rows_mx, msz);
            if (last) ntt_rows_grouped_kernel<LOGN, K2, E, RS, INV, true, FULL, true><<<b, RS << (K2 - E), 0, st>>>(rows_mx);
            else ntt_rows_grouped_kernel<LOGN, K2, E, RS, INV, false, FULL, true><<<b, RS << (K2 - E), 0, st>>>(rows_mx);
        }
        if (!fsz.empty()) {
            const uint32_t b = fill_starts(rows_full, fsz);
            if (last) ntt_rows_grouped_kernel<LOGN, K2, E, RS, INV, true, FULL, false><<<b, RS << (K2 - E), 0, st>>>(rows_full);
            else ntt_rows_grouped_kernel<LOGN, K2, E, RS, INV, false, FULL, false><<<b, RS << (K2 - E), 0, st>>>(rows_full);
        }
    };
    if (!INV) {
        ntt_cols_grouped_kernel<LOGN, K1, E, CS, false, false, FULL><<<cb, CS << (K1 - E), 0, st>>>(cols);
        rows(true);
    } else {
        rows(false);
        ntt_cols_grouped_kernel<LOGN, K1, E, CS, true, true, FULL><<<cb, CS << (K1 - E), 0, st>>>(cols);
    }
    launch_check("grouped ntt launch");
}

template <int LOGN, bool INV, bool FULL>
void launch_ntt_groups(const NttGroup *gs, uint32_t n, hipStream_t st) {
    uint64_t limbs = 0;
    for (uint32_t g = 0; g < n; g++) limbs += (uint64_t)gs[g].lg.I * gs[g].lg.J;
    with_shape<LOGN>(limbs, [&](auto s) { launch_ntt_groups_as<LOGN, INV, FULL, decltype(s)::value>(gs, n, st); });
}

template <bool INV, bool FULL>
void launch_ntt_multi(const NttGroup *gs, const int *logns, uint32_t n, hipStream_t st) {
    NttMulti cols{}, rows{};
    std::vector<uint64_t> csz, rsz;
    for (uint32_t g = 0; g < n; g++) {
        const NttGroup &a = gs[g];
        const int L = logns[g];
        const int K1 = L / 2, K2 = L - K1;
        const uint32_t CS = 4096u >> K1, RS = 4096u >> K2;
        const NttGroupDev d{a.data, nullptr, a.lg, a.lg, a.primes};
        const NttGroupDev d_first{a.data, a.src, a.lg, a.src ? a.slg : a.lg, a.primes};
        // the first pass reads src where a group has one; the second runs in place
        cols.g[g] = NttMultiDev{INV ? d : d_first, L};
        rows.g[g] = NttMultiDev{INV ? d_first : d, L};
        csz.push_back((uint64_t)a.lg.I * a.lg.J * ((1u << (L - K1)) / CS));
        rsz.push_back((uint64_t)a.lg.I * (1u << (L - K2)) * ((a.lg.J + RS - 1) / RS));
    }
    const uint32_t cb = fill_starts(cols, csz), rb = fill_starts(rows, rsz);
    if (!INV) {
        ntt_cols_multi_kernel<false, false, FULL><<<cb, 256, 0, st>>>(cols);
        ntt_rows_multi_kernel<false, true, FULL><<<rb, 256, 0, st>>>(rows);
    } else {
        ntt_rows_multi_kernel<true, false, FULL><<<rb, 256, 0, st>>>(rows);
        ntt_cols_multi_kernel<true, true, FULL><<<cb, 256, 0, st>>>(cols);
    }
    launch_check("multi-degree ntt launch");
}

}  // namespace

void ntt_forward_groups(const NttGroup *gs, uint32_t n, int logn, NttOut out, hipStream_t st) {
    if (n > MAX_GROUPS) fail(ERR_INVALID_ARGUMENT, "too many groups for one launch");
    if (n == 0) return;
    if (logn <= 12) {
        // one-tile transforms: a group with a source is copied first, then transformed
        for (uint32_t g = 0; g < n; g++) {
            if (gs[g].src) {
                const LimbGrid &d = gs[g].lg, &s = gs[g].slg;
                if (d.A == 1 && s.A == 1 && d.B == d.I && s.B == s.I) {  // both dense: one copy
                    SHC_HIP(hipMemcpyAsync(gs[g].data, gs[g].src, ((size_t)d.I * d.J * 8) << logn,
                                           hipMemcpyDeviceToDevice, st));
                    ntt_forward_grid(gs[g].data, gs[g].lg, gs[g].primes, logn, out, st);
                    continue;
                }
                for (uint32_t j = 0; j < d.J; j++)
                    for (uint32_t i = 0; i < d.I; i++)
                        SHC_HIP(hipMemcpyAsync(gs[g].data + ((size_t)(i * d.A + j * d.B) << logn),
                                               gs[g].src + ((size_t)(i * s.A + j * s.B) << logn), (size_t)8 << logn,
                                               hipMemcpyDeviceToDevice, st));
            }
            ntt_forward_grid(gs[g].data, gs[g].lg, gs[g].primes, logn, out, st);
        }
        return;
    }
    switch (logn) {
#define SHC_NTT_CASE(L)                                                          \
    case L:                                                                      \
        if (out == NTT_FULL) launch_ntt_groups<L, false, true>(gs, n, st);       \
        else launch_ntt_groups<L, false, false>(gs, n, st);                      \
        break;
        SHC_NTT_CASE(13) SHC_NTT_CASE(14) SHC_NTT_CASE(15) SHC_NTT_CASE(16) SHC_NTT_CASE(17)
#undef SHC_NTT_CASE
        default: fail(ERR_INVALID_ARGUMENT, "poly_modulus_degree must be 2^1 .. 2^17");
    }
}

void ntt_inverse_groups(const NttGroup *gs, uint32_t n, int logn, NttOut out, hipStream_t st) {
    if (n > MAX_GROUPS) fail(ERR_INVALID_ARGUMENT, "too many groups for one launch");
    if (n == 0) return;
    if (logn <= 12) {
        for (uint32_t g = 0; g < n; g++) {
            if (gs[g].src) ntt_inverse_from(gs[g].src, gs[g].slg, gs[g].data, gs[g].lg, gs[g].primes, logn, out, st);
            else ntt_inverse_grid(gs[g].data, gs[g].lg, gs[g].primes, logn, out, st);
        }
        return;
    }
    switch (logn) {
#define SHC_NTT_CASE(L)                                                          \
    case L:                                                                      \
        if (out == NTT_FULL) launch_ntt_groups<L, true, true>(gs, n, st);        \
        else launch_ntt_groups<L, true, false>(gs, n, st);                       \
        break;
        SHC_NTT_CASE(13) SHC_NTT_CASE(14) SHC_NTT_CASE(15) SHC_NTT_CASE(16) SHC_NTT_CASE(17)
#undef SHC_NTT_CASE
        default: fail(ERR_INVALID_ARGUMENT, "poly_modulus_degree must be 2^1 .. 2^17");
    }
}

namespace {
void check_multi(const NttGroup *gs, const int *logns, uint32_t n) {
    if (n > MAX_GROUPS) fail(ERR_INVALID_ARGUMENT, "too many groups for one launch");
    uint64_t cols = 0, rows = 0;
    for (uint32_t g = 0; g < n; g++) {
        const int L = logns[g];
        if (L < 13 || L > 17) fail(ERR_INVALID_ARGUMENT, "multi-degree transforms take N = 2^13 .. 2^17");
        const LimbGrid &lg = gs[g].lg;
        if (!lg.I || !lg.J) fail(ERR_INVALID_ARGUMENT, "empty transform group");
        const int K1 = L / 2, K2 = L - K1;
        cols += (uint64_t)lg.I * lg.J * ((1u << (L - K1)) / (4096u >> K1));
        rows += (uint64_t)lg.I * (1u << (L - K2)) * ((lg.J + (4096u >> K2) - 1) / (4096u >> K2));
    }
    if (cols >= (uint64_t(1) << 32) || rows >= (uint64_t(1) << 32))
        fail(ERR_INVALID_ARGUMENT, "transform batch too large for one launch");
}
}  // namespace

void ntt_forward_multi(const NttGroup *gs, const int *logns, uint32_t n, NttOut out, hipStream_t st) {
    check_multi(gs, logns, n);
    if (!n) return;
    if (out == NTT_FULL) launch_ntt_multi<false, true>(gs, logns, n, st);
    else launch_ntt_multi<false, false>(gs, logns, n, st);
}

void ntt_inverse_multi(const NttGroup *gs, const int *logns, uint32_t n, NttOut out, hipStream_t st) {
    check_multi(gs, logns, n);
    if (!n) return;
    if (out == NTT_FULL) launch_ntt_multi<true, true>(gs, logns, n, st);
    else launch_ntt_multi<true, false>(gs, logns, n, st);
}

}  // namespace shc

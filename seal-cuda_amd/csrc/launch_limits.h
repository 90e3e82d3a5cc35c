// launch_limits.h -- how the key switch splits a batch into blocks, and which grouped calls
// one launch per stage holds.  Host code free of HIP, so host tests build it alone.
#pragma once
#include <cstdint>
#include <initializer_list>

namespace shc {

// A grouped launch has fewer blocks than this (of at most 1024 threads: below 2^32 threads).
constexpr uint64_t GROUPED_BLOCKS = uint64_t(1) << 22;

// A batch's groups of ciphertexts.  N = 2^15 up: groups of 4, then the rest as a group of 2
// and/or 1, so that no row is transformed for a ciphertext that is not there.  Up to
// N = 2^14 a launch of its own for the rest costs more than its idle slots: the last group
// of 4 is a short one (products at N = 2^14, L = 7: 101 against 110 us for 3 ciphertexts, 546
// against 551 for 37; in two kernels 101 and 575).
struct GroupSplit {
    uint32_t g4, g2, singles;
};
inline GroupSplit split_groups(int logn, uint32_t cts, uint32_t group) {
    uint32_t g4 = group == 4 ? cts / 4 : 0;
    uint32_t rest = cts - 4 * g4;
    if (logn <= 14 && group == 4 && (g4 ? rest : rest == 3)) g4++, rest = 0;
    const uint32_t g2 = group == 1 ? 0 : rest / 2;
    return GroupSplit{g4, g2, rest - 2 * g2};
}

// The group sizes among 4, 2 and 1 that split cts ciphertexts differently, the largest first;
// returns how many (out: room for 3).
inline uint32_t distinct_groups(int logn, uint32_t cts, uint32_t *out) {
    uint32_t n = 0;
    for (uint32_t g : {4u, 2u, 1u}) {
        const GroupSplit s = split_groups(logn, cts, g);
        bool known = false;
        for (uint32_t k = 0; k < n; k++) {
            const GroupSplit o = split_groups(logn, cts, out[k]);
            known |= o.g4 == s.g4 && o.g2 == s.g2 && o.singles == s.singles;
        }
        if (!known) out[n++] = g;
    }
    return n;
}

// Blocks per group of the fused key products at level L: one per row of every target prime (a
// single ciphertext's blocks take two rows), a multiple of the 8 XCDs.
inline uint64_t keyprod_slots(int logn, uint32_t L, bool single) {
    const uint64_t tiles = ((uint64_t)L + 1) << (logn / 2);
    return ((single ? tiles / 2 : tiles) + 7) / 8 * 8;
}

// Whether a grouped relinearization (CKKS, N = 2^13 .. 2^16) of n groups, count[g] ciphertexts at
// L[g] limbs, stays below GROUPED_BLOCKS in every launch: the key products' of 4, 2 and 1, and
// the ModDown's passes, which have the most blocks of the transforms (2 L limbs per ciphertext;
// the ModUp's columns pass has as many per digit limb once its tiles fill the chip, and at most
// 32,768 before).
inline bool relinearize_groups_fit(int logn, const uint32_t *count, const uint32_t *L, uint32_t n) {
    const int K1 = logn / 2, K2 = logn - K1;
    uint64_t s4 = 0, s2 = 0, s1 = 0, cols = 0, rows = 0;
    for (uint32_t g = 0; g < n; g++) {
        const GroupSplit s = split_groups(logn, count[g], 4);
        s4 += keyprod_slots(logn, L[g], false) * s.g4;
        s2 += keyprod_slots(logn, L[g], false) * s.g2;
        s1 += keyprod_slots(logn, L[g], true) * s.singles;
        const uint64_t j = 2 * (uint64_t)count[g], per = 4096u >> K2;
        cols += L[g] * j << (K2 - 4);
        rows += (uint64_t)L[g] * ((j + per - 1) / per) << K1;
    }
    for (uint64_t blocks : {s4, s2, s1, cols, rows})
        if (blocks >= GROUPED_BLOCKS) return false;
    return true;
}

}  // namespace shc

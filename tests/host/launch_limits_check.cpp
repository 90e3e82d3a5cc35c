// Host check of seal-cuda_amd/csrc/launch_limits.h: a batch's groups cover its ciphertexts once
// and in order of size, the autotuner's group sizes all split it differently, and a grouped
// relinearization is taken exactly when the blocks of
// each launch, counted here from the kernels' grids, stay below the limit of a grouped launch.
// Prints "ok <cases>" and exits 0, or prints the first failing case and exits 1.
#include "launch_limits.h"
#include <cstdio>
#include <vector>

using u64 = uint64_t;

static bool fits(int logn, const std::vector<uint32_t> &count, const std::vector<uint32_t> &L) {
    const int K1 = logn / 2, K2 = logn - K1;
    u64 most = 0, launch[5] = {};
    for (size_t g = 0; g < count.size(); g++) {
        const shc::GroupSplit s = shc::split_groups(logn, count[g], 4);
        const u64 rows = (u64)(L[g] + 1) << K1;  // multiples of 8 for every degree
        launch[0] += rows * s.g4;
        launch[1] += rows * s.g2;
        launch[2] += (rows / 2 + 7) / 8 * 8 * s.singles;
        // ModDown: limbs 2 L count, 16 columns a block; rows of one row index, 4096 words a block
        launch[3] += 2 * (u64)L[g] * count[g] * ((1u << K2) / 16);
        const u64 per = (4096 >> K2);
        launch[4] += L[g] * ((2 * (u64)count[g] + per - 1) / per) * (1u << K1);
    }
    for (u64 b : launch) most = b > most ? b : most;
    return most < (u64(1) << 32) / 1024;
}

int main() {
    long cases = 0, taken = 0;
    for (int logn = 13; logn <= 16; logn++) {
        for (uint32_t group : {1u, 2u, 4u})
            for (uint32_t cts = 1; cts < 70; cts++, cases++) {
                const shc::GroupSplit s = shc::split_groups(logn, cts, group);
                const u64 slots = 4 * (u64)s.g4 + 2 * s.g2 + s.singles;
                if (slots < cts || slots > cts + 3 || (logn >= 15 && slots != cts))
                    return std::printf("split of %u at 2^%d by %u\n", cts, logn, group), 1;
            }
        // one ciphertext splits one way, two two ways (4 splits like 2), others by all three
        for (uint32_t cts = 1; cts < 70; cts++, cases++) {
            uint32_t g[3] = {};
            const uint32_t ways = shc::distinct_groups(logn, cts, g);
            const uint32_t want = cts == 1 ? 1 : cts == 2 || (cts == 3 && logn >= 15) ? 2 : 3;
            if (ways != want || g[0] != 4 || (ways > 1 && g[ways - 1] != 1))
                return std::printf("splits of %u at 2^%d\n", cts, logn), 1;
        }
        for (uint32_t L : {1u, 2u, 3u, 7u, 24u})
            for (uint32_t groups : {1u, 2u, 16u})
                for (uint32_t base = 1; base < (1u << 20); base = base * 3 / 2 + 1)
                    for (uint32_t d = 0; d < 5; d++, cases++) {
                        std::vector<uint32_t> count, lv;
                        for (uint32_t g = 0; g < groups; g++) count.push_back(base + d * g), lv.push_back(L);
                        const bool want = fits(logn, count, lv);
                        taken += want;
                        if (shc::relinearize_groups_fit(logn, count.data(), lv.data(), groups) != want)
                            return std::printf("2^%d L=%u %u groups of %u\n", logn, L, groups, base), 1;
                    }
    }
    // 131,072 ciphertexts of one limb at N = 2^13 are 2^22 blocks of the groups of 4
    for (uint32_t c : {131068u, 131072u}) {
        const uint32_t L = 1;
        if (shc::relinearize_groups_fit(13, &c, &L, 1) != (c < 131072)) return std::printf("line at %u\n", c), 1;
        cases++;
    }
    if (!taken || taken == cases) return std::printf("one-sided\n"), 1;
    std::printf("ok %ld\n", cases);
    return 0;
}

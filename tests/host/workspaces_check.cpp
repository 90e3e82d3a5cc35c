// Host check of seal-cuda_amd/csrc/workspaces.h, over ring degrees, levels and batch sizes:
//   * the regions of a layout lie apart (but for the overlay that it states) and inside its
//     total;
//   * the sizes that are asked for never shrink as the batch grows, and a workspace asked for a
//     batch holds every smaller one;
//   * hoisted rotations ask for no more than 19 L + 12 + L (L + 1) limbs per ciphertext, and
//     rotation sums for no more than that, ACC_BYTES, or a Galois switch's need.
// Prints "ok <cases>" and exits 0, or prints the first failing case and exits 1.
#include "workspaces.h"
#include <cstdio>
#include <vector>

using namespace shc;

struct Region {
    size_t at, len;
};
static bool apart(const std::vector<Region> &rs, size_t total) {
    for (size_t i = 0; i < rs.size(); i++) {
        if (rs[i].at + rs[i].len > total || rs[i].at % 256) return false;
        for (size_t j = 0; j < i; j++)
            if (rs[i].at < rs[j].at + rs[j].len && rs[j].at < rs[i].at + rs[i].len) return false;
    }
    return true;
}

static bool check(int logn, uint32_t L, uint32_t count) {
    const size_t limb = ((size_t)8 << logn) * count, per = (size_t)L * (L + 1);
    const KsLayout k = ks_layout(logn, count, L);
    if (!apart({{k.d, L * limb}, {k.T, per * limb}, {k.P, 2 * L * limb}, {k.S, 2 * limb}, {k.U, 2 * L * limb}}, k.total))
        return false;
    const RotLayout r = rot_layout(logn, count, L);
    const std::vector<Region> shared{{r.flag, 8}, {r.zc, 8 * (2 + (size_t)count)}, {r.c, L * limb}, {r.T, per * limb},
                                     {r.list, L * limb}, {r.Pm, 8 * L * limb}};
    for (bool sum : {false, true}) {
        std::vector<Region> v = shared;
        if (r.batched) {
            // U over Sm
            const size_t u = (sum ? 2 : 8) * (size_t)L;
            if ((sum ? r.U_sum != r.Sm_sum : r.U != r.Sm)) return false;
            v.push_back({r.S2, 8 * limb});
            v.push_back({sum ? r.U_sum : r.U, (u > 8 ? u : 8) * limb});
            if (sum) v.push_back({r.V, 2 * limb}), v.push_back({r.Psum, 2 * L * limb});
        } else {
            for (Region x : {Region{r.Sm, 8 * limb}, Region{r.C0, L * limb}, Region{r.P2, 2 * L * limb},
                             Region{r.S2, 2 * limb}, Region{r.U, 2 * L * limb}})
                v.push_back(x);
            if (r.Sm != r.Sm_sum || r.U != r.U_sum) return false;
        }
        if (!apart(v, r.total)) return false;
    }
    auto up = [](size_t b) { return (b + 255) & ~size_t(255); };
    const size_t hoisted = up(L * limb) + k.total + 2 * up(2 * L * limb) + up(2 * limb) + up(L * limb) +
                           up(8 * L * limb) + up(8 * limb) + up(8) + up(8 * (2 + (size_t)count));
    if (r.total > hoisted) return std::printf("hoisted rotations ask for more\n"), false;
    for (uint32_t nb = 1; nb <= ROT_MAX; nb++) {
        const AccLayout a = acc_layout(logn, count, L, nb);
        if (!a.batched) {
            if (!apart({{a.d, L * limb}, {a.C0, L * limb}, {a.ks, k.total}}, a.total)) return false;
            continue;
        }
        if (!apart({{a.d, nb * L * limb}, {a.T, (acc_fused(logn) ? 1 : nb) * per * limb}, {a.P, nb * 2 * L * limb},
                    {a.S, nb * 2 * limb}, {a.Psum, 2 * L * limb}, {a.V, 2 * limb}, {a.U, 2 * L * limb}}, a.total))
            return false;
    }
    const size_t ask = acc_workspace(logn, count, L);
    const uint32_t nb = acc_rotations(logn, count, L, ask);
    if (!nb || acc_layout(logn, count, L, nb).total > ask) return std::printf("ask\n"), false;
    const size_t one = acc_layout(logn, count, L, 1).total;
    if (acc_rotations(logn, count, L, one) < 1 || acc_rotations(logn, count, L, one - 1)) return std::printf("need\n"), false;
    if (one > hoisted) return std::printf("one rotation needs more\n"), false;
    if (acc_batched(logn, count, L) && ask > hoisted && ask > ACC_BYTES) return std::printf("rotation sums ask for more\n"), false;
    return true;
}

int main() {
    long cases = 0;
    std::vector<uint32_t> counts;
    for (uint32_t c = 1; c < 70; c++) counts.push_back(c);
    for (uint32_t c = 70; c < 200000; c = c * 21 / 20 + 1) counts.push_back(c);
    for (uint32_t c = 100; c < 130; c++) counts.push_back(c);
    std::sort(counts.begin(), counts.end());
    for (int logn : {1, 3, 10, 12, 13, 14, 15, 16, 17})
        for (uint32_t L : {1u, 2u, 3u, 4u, 8u, 15u, 16u, 24u, 40u}) {
            size_t rot = 0, acc = 0, ks = 0;
            std::vector<uint32_t> cs = counts;
            const uint64_t line = launch_limbs(logn) / ((uint64_t)L * (L + 1));  // the last batched count
            for (uint64_t c = line > 2 ? line - 2 : 1; c < line + 3; c++)
                if (c && c < 2000000) cs.push_back((uint32_t)c);
            std::sort(cs.begin(), cs.end());
            uint32_t last = 0;
            for (uint32_t c : cs) {
                if (!check(logn, L, c)) return std::printf("2^%d L=%u count=%u\n", logn, L, c), 1;
                const size_t a = acc_workspace(logn, c, L);
                const size_t r = rot_layout(logn, c, L).total, k = ks_layout(logn, c, L).total;
                if (a < acc || r < rot || k < ks || (last && !acc_rotations(logn, last, L, a)))
                    return std::printf("shrinks: 2^%d L=%u count=%u\n", logn, L, c), 1;
                acc = a, rot = r, ks = k, last = c;
                cases++;
            }
        }
    std::printf("ok %ld\n", cases);
    return 0;
}

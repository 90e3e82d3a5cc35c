// workspaces.h -- what lies where in the workspaces of key switches, hoisted rotations and
// rotation sums, and how many rotations share a launch.  A workspace that was sized for a
// batch holds every smaller one: the sizes never shrink as the batch grows.  Host code free
// of HIP, so host tests build it alone.
#pragma once
#include <algorithm>
#include <cstddef>
#include <cstdint>

namespace shc {

constexpr uint32_t ROT_MAX = 4;    // rotations per launch
constexpr uint32_t SUM_MAX = 15;   // rotations per summed ModDown (15 words below 2^60)

// Regions of whole limbs (count ciphertexts of N words each), 256-byte aligned.
struct WorkspaceRegions {
    size_t limb, off = 0;
    WorkspaceRegions(int logn, uint32_t count) : limb(((size_t)8 << logn) * count) {}
    size_t bytes(size_t b) {
        const size_t o = off;
        off += (b + 255) & ~size_t(255);
        return o;
    }
    size_t limbs(size_t per_ct) { return bytes(per_ct * limb); }
};

// Most limbs that one launch's transforms cover.
inline uint64_t launch_limbs(int logn) { return (uint64_t(1) << 34) >> logn; }

// Key switch: digits [count][L], T[i][ct][j], products P [count][2][L] and S [count][2], and the
// ModDown's corrections.
struct KsLayout {
    size_t d, T, P, S, U, total;
};
inline KsLayout ks_layout(int logn, uint32_t count, uint32_t L) {
    WorkspaceRegions r(logn, count);
    KsLayout l;
    l.d = r.limbs(L);
    l.T = r.limbs((size_t)L * (L + 1));
    l.P = r.limbs(2 * (size_t)L);
    l.S = r.limbs(2);
    l.U = r.limbs(2 * (size_t)L);
    l.total = r.off;
    return l;
}

// Hoisted rotations.  c: the digits (CKKS) or c0's transforms (BFV); list: the zero digits; Pm,
// Sm: the products of up to ROT_MAX rotations; S2: their special limbs in coefficient form; U:
// the ModDown's corrections.
//   N >= 2^13: a pass's rotations share each launch.  U takes the place of Sm, which is dead once
//   S2 is there; sums (Psum, V: the sums over passes) hold one ModDown's corrections, separate
//   outputs (for which those two are not needed) a whole pass's.
//   N < 2^13: one rotation at a time -- its permuted products (P2, S2), and C0 = sigma(c0).
struct RotLayout {
    bool batched;
    size_t c, T, list, Pm, Sm, S2, U;
    size_t Psum, V, U_sum, Sm_sum;  // batched
    size_t C0, P2;                  // one at a time
    size_t flag, zc, total;
};
inline RotLayout rot_layout(int logn, uint32_t count, uint32_t L) {
    WorkspaceRegions r(logn, count);
    RotLayout l{};
    l.batched = logn >= 13;
    l.flag = r.bytes(8);
    l.zc = r.bytes(8 * (2 + (size_t)count));
    l.c = r.limbs(L);
    l.T = r.limbs((size_t)L * (L + 1));
    l.list = r.limbs(L);
    l.Pm = r.limbs(ROT_MAX * 2 * (size_t)L);
    if (l.batched) {
        l.S2 = r.limbs(ROT_MAX * 2);
        WorkspaceRegions many = r;
        l.Sm = l.U = many.limbs(ROT_MAX * 2 * (size_t)L);  // (no fewer than Sm's 2 ROT_MAX)
        l.V = r.limbs(2);
        l.Psum = r.limbs(2 * (size_t)L);
        l.Sm_sum = l.U_sum = r.limbs(std::max<size_t>(ROT_MAX * 2, 2 * (size_t)L));
        l.total = std::max(r.off, many.off);
        return l;
    }
    l.Sm = l.Sm_sum = r.limbs(ROT_MAX * 2);
    l.C0 = r.limbs(L);
    l.P2 = r.limbs(2 * (size_t)L);
    l.S2 = r.limbs(2);
    l.U = l.U_sum = r.limbs(2 * (size_t)L);
    l.total = r.off;
    return l;
}

// Sums of rotations of different ciphertexts (rotate_accumulate): batches of nb rotations, or one
// at a time (d: sigma(c1); C0: sigma(c0); a key switch's workspace) below N = 2^13 and where one
// rotation's T is more than a launch.  N = 2^15, 2^16: the fused key products take
// one rotation's T at a time; other degrees a batch's.
struct AccLayout {
    bool batched;
    size_t d, T, P, S, Psum, V, U;  // batched
    size_t C0, ks;                  // one at a time, beside d
    size_t total;
};
inline bool acc_fused(int logn) { return logn == 15 || logn == 16; }
inline bool acc_batched(int logn, uint32_t count, uint32_t L) {
    return logn >= 13 && (uint64_t)count * L * (L + 1) <= launch_limbs(logn);
}
inline AccLayout acc_layout(int logn, uint32_t count, uint32_t L, uint32_t nb) {
    WorkspaceRegions r(logn, count);
    AccLayout l{};
    l.batched = acc_batched(logn, count, L);
    l.d = r.limbs((size_t)(l.batched ? nb : 1) * L);
    if (l.batched) {
        l.T = r.limbs((acc_fused(logn) ? 1 : nb) * (size_t)L * (L + 1));
        l.P = r.limbs((size_t)nb * 2 * L);
        l.S = r.limbs((size_t)nb * 2);
        l.Psum = r.limbs(2 * (size_t)L);
        l.V = r.limbs(2);
        l.U = r.limbs(2 * (size_t)L);
    } else {
        l.C0 = r.limbs(L);
        l.ks = r.bytes(ks_layout(logn, count, L).total);
    }
    l.total = r.off;
    return l;
}
// Rotations per batch in a workspace of ws_bytes (0: too small for one).
inline uint32_t acc_rotations(int logn, uint32_t count, uint32_t L, size_t ws_bytes) {
    uint32_t nb = ROT_MAX;
    auto fits = [&] {
        const uint64_t limbs = (uint64_t)nb * count * (acc_fused(logn) ? 2 * L : L * (L + 1));
        return acc_layout(logn, count, L, nb).total <= ws_bytes &&
               (nb == 1 || !acc_batched(logn, count, L) || limbs <= launch_limbs(logn));
    };
    while (nb && !fits()) nb--;
    return nb;
}
// The workspace that is asked for.  Batches pay where launches are short, so where their T is
// shared they take no more than ACC_BYTES beyond one rotation's need: at N = 2^17, L = 16,
// 120 ciphertexts four rotations' T would be 137 GB.  Past the largest batched count: no less
// than for that one.
constexpr size_t ACC_BYTES = size_t(1) << 30;
inline size_t acc_workspace(int logn, uint32_t count, uint32_t L) {
    if (!acc_batched(logn, count, L)) {
        const size_t one = acc_layout(logn, count, L, 1).total;
        const uint32_t most = logn < 13 ? 0 : (uint32_t)(launch_limbs(logn) / ((uint64_t)L * (L + 1)));
        return most ? std::max(one, acc_workspace(logn, most, L)) : one;
    }
    const size_t full = acc_layout(logn, count, L, ROT_MAX).total;
    if (acc_fused(logn)) return full;
    return std::min(full, std::max(acc_layout(logn, count, L, 1).total, ACC_BYTES));
}

}  // namespace shc

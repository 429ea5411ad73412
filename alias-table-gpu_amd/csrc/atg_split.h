// Split search of SplitMethodBasic (SplitMethodBasic.cu:14-50, predicate
// SplitMethodBasic.cuh:9-41), shared by the bisection and learned kernels.
#pragma once

#include "atg_device.h"

namespace atg {

// 0 FOUND, 1 continue left, 2 continue right.
__device__ __forceinline__ int check_split(int64_t i, int64_t j, double target, const double* Lp, int64_t numL,
                                           const double* Hp, int64_t numH, double& sigma) {
    if (j + 1 >= numH || i - 1 < 0) return 1;  // LEFT
    if (i >= numL || j < 0) return 2;          // RIGHT
    const double s = Lp[i] + Hp[j];
    const double sn = Lp[i - 1] + Hp[j + 1];
    sigma = s;
    if (s <= target && sn > target) return 0;  // FOUND
    if (s <= target) return 2;
    return 1;
}

// The number of list items before split k, and the weight they should hold.
__device__ __forceinline__ int64_t split_items(int64_t k, int64_t p, int64_t nToSplit) {
    return (int64_t)ceil(((double)nToSplit * (double)k) / (double)p);
}
__device__ __forceinline__ double split_target(int64_t k, int64_t p, int64_t nToSplit, double wToSplit) {
    return (wToSplit * (double)split_items(k, p, nToSplit)) / (double)nToSplit;
}

// A split's spill, or, where the heavy weights come later, its prefix sum.
struct SpillLater {};
__device__ __forceinline__ double split_spill(double sigma, const double* Hw, int64_t j, double target) {
    return sigma + Hw[j] - target;
}
__device__ __forceinline__ double split_spill(double sigma, SpillLater, int64_t, double) { return sigma; }

// Bisection; 64 probes bound the loop (the reference spins forever when
// FOUND is unreachable), then a deterministic clamp is returned.
template <typename HW>
__device__ __forceinline__ bool bisect_split(int64_t k, int64_t p, int64_t nToSplit, double wToSplit,
                                             const double* Lp, int64_t numL, const double* Hp, HW Hw,
                                             int64_t numH, Split& out) {
    const int64_t n_ = split_items(k, p, nToSplit);
    const int64_t b0 = min(n_, numH) - 1;
    const double target = (wToSplit * (double)n_) / (double)nToSplit;
    int64_t lo = 0, hi = b0;
    double sigma = 0.0;
    for (int it = 0; it < 64; ++it) {
        const int64_t j = (lo + hi) / 2;
        const int64_t i = min(n_ - j, numL - 1);
        const int stt = check_split(i, j, target, Lp, numL, Hp, numH, sigma);
        if (stt == 0) {
            out.i = (int32_t)i; out.j = (int32_t)j; out.spill = split_spill(sigma, Hw, j, target);
            return true;
        }
        if (stt == 2) lo = j + 1; else hi = j;
    }
    int64_t j = min(max<int64_t>(lo, 0), max<int64_t>(b0, 0));
    int64_t i = min(n_ - j, numL - 1);
    if (i < 0) i = 0;
    out.i = (int32_t)i; out.j = (int32_t)j; out.spill = split_spill(Lp[i] + Hp[j], Hw, j, target);
    return false;
}

// bisect_split by a group of 2^LEVELS consecutive lanes, lane g of the group
// (all of them with the same k): a round probes the positions that the
// bisection's next LEVELS levels can reach, lane g > 0 the node g of their
// tree in heap order, and follows the statuses down, so the probes that
// decide are those of bisect_split, in LEVELS times fewer dependent reads.
// live: groups without a split take part in the ballots only.  The result
// and the return value are the same on every lane of the group.  Positions
// fit 30 bits (their sums are ints).
template <int LEVELS>
__device__ __forceinline__ bool bisect_split_wide(bool live, int g, int64_t k, int64_t p, int64_t nToSplit,
                                                  double wToSplit, const double* Lp, int64_t numL, const double* Hp,
                                                  const double* Hw, int64_t numH, Split& out) {
    constexpr int LANES = 1 << LEVELS;
    static_assert(64 % LEVELS == 0, "as many probes as bisect_split");
    constexpr uint32_t group = (uint32_t)((1ull << LANES) - 1);
    const int lane = lane_id(), base = lane & ~(LANES - 1);
    const int n_ = live ? (int)ceil(((double)nToSplit * (double)k) / (double)p) : 1;
    const int b0 = min(n_, (int)numH) - 1;
    const double target = (wToSplit * (double)n_) / (double)nToSplit;
    int lo = 0, hi = b0;
    bool open = live;
    int hit_j = 0;
    double hit = 0.0;
    for (int round = 0; round < 64 / LEVELS; ++round) {
        // Node g's range: the path of g's bits below the leading one.
        int l = lo, h = hi;
        const int depth = 31 - __builtin_clz(g | 1);
#pragma unroll
        for (int d = LEVELS - 2; d >= 0; --d) {
            if (d < depth) {
                const int m = (l + h) / 2;
                if ((g >> d) & 1) l = m + 1;
                else h = m;
            }
        }
        const int j = (l + h) / 2, i = min(n_ - j, (int)numL - 1);
        double sigma = 0.0;
        int stt = 1;
        if (open && g > 0) stt = check_split(i, j, target, Lp, numL, Hp, numH, sigma);
        const uint32_t fnd = (uint32_t)(__ballot(open && g > 0 && stt == 0) >> base) & group;
        const uint32_t rgt = (uint32_t)(__ballot(open && g > 0 && stt == 2) >> base) & group;
        int node = 1, at = 0;
#pragma unroll
        for (int d = 0; d < LEVELS; ++d) {
            if (at == 0 && ((fnd >> node) & 1)) at = node;
            if (at == 0) {
                const int m = (lo + hi) / 2;
                const int right = (int)(rgt >> node) & 1;
                if (right) lo = m + 1;
                else hi = m;
                node = 2 * node + right;
            }
        }
        const double sg = __shfl(sigma, base + at, 64);
        const int jg = __shfl(j, base + at, 64);
        if (open && at != 0) {
            hit_j = jg;
            hit = sg;
            open = false;
        }
        if (__ballot(open) == 0ull) break;
    }
    if (!live) return true;
    if (!open) {
        out.i = min(n_ - hit_j, (int)numL - 1);
        out.j = hit_j;
        out.spill = hit + Hw[hit_j] - target;
        return true;
    }
    const int64_t j = min(max<int64_t>(lo, 0), max<int64_t>(b0, 0));
    int64_t i = min<int64_t>(n_ - j, numL - 1);
    if (i < 0) i = 0;
    out.i = (int32_t)i; out.j = (int32_t)j; out.spill = (Lp[i] + Hp[j]) + Hw[j] - target;
    return false;
}

}  // namespace atg

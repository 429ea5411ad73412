// Split searches that use the split certificate, for gfx950: the learned index, the
// P-ary search and the bisection in groups.
// Learned split index: a piecewise-linear model of the split
// position j*(k) over K segments, fitted on the build's own prefix sums, with an
// exact bounded local search and the plain bisection as fallback and judge.
//
// Model: K + 1 knots k_m = floor(m p / K); the knot splits are computed exactly
// by bisection (they are splits of the table).  For k inside segment m the
// model predicts j by linear interpolation between the knot values and the
// search gallops outwards from the prediction inside [j_m, j_{m+1}].
//
// Bit identity with bisection: the partition certifies max dL < min dH over
// the stored prefix sums (dL, dH: consecutive increments, sentinels included).  Then the
// FOUND predicate of SplitMethodBasic (SplitMethodBasic.cuh:23-39) holds at
// exactly one j and bisection returns it, so any exact search returns the same
// (i, j, spill).  Without the certificate, or when the bracket check or the
// local search fails, the k is resolved by full bisection (and counted).
#include "atg_kernels.h"

namespace atg {

__global__ __launch_bounds__(256) void split_learned(BuildArgs a, int64_t blk0) {
    DevState* st = a.st;
    if (st->error || st->degenerate) return;
    const int64_t k = (blk0 + (int64_t)blockIdx.x) * blockDim.x + threadIdx.x + 1;
    if (k >= st->p) return;
    const uint32_t f = learned_split(a, k);
    if (f & 1u) atomicAdd((unsigned long long*)&st->split_fallbacks, 1ull);
    if (f & 2u) atomicAdd((unsigned long long*)&st->learned_fallbacks, 1ull);
}

// P-ary search for split k by a group of LANES lanes (lane g of it, shift its
// first lane in the wave): every step probes LANES positions of the bracket at
// once and keeps the part between the last RIGHT and the first LEFT probe
// (about LANES + 1 times smaller each step), then probes the last <= LANES
// positions together.  Under the split certificate the FOUND position is the
// only one and the statuses run RIGHT .. FOUND .. LEFT along j.  Returns the
// group's lane that found it, whose out is written, or -1.  live: groups
// without a search take part in the ballots only.
template <int LANES>
__device__ __forceinline__ int pary_search(const BuildArgs& a, bool live, int64_t k, int g, int shift, Split& out) {
    const DevState* st = a.st;
    const int64_t p = st->p, numL = st->numL, numH = st->numH;
    const int64_t n_ = live ? split_items(k, p, st->nToSplit) : 0;
    const double target = live ? split_target(k, p, st->nToSplit, st->wToSplit) : 0.0;
    constexpr uint64_t group = (1ull << LANES) - 1;
    int64_t lo = 0, hi = min(n_, numH) - 1;
    int found_lane = -1;  // the same on every lane of the group
    // Every lane of a wave runs the loop until all its groups are done (the
    // ballots are wave-wide); finished groups only idle.
    for (int level = 0; level < 64; ++level) {
        const bool wide = live && hi - lo + 1 > LANES;
        int64_t j = -1;
        if (live) j = wide ? lo + ((hi - lo) * (int64_t)(g + 1)) / (LANES + 1) : lo + g;
        int stt = 1;
        double sigma = 0.0;
        int64_t i = 0;
        if (live && j <= hi) {
            i = min(n_ - j, numL - 1);
            stt = check_split(i, j, target, a.Lp, numL, a.Hp, numH, sigma);
        }
        const uint64_t fnd = (__ballot(live && j <= hi && stt == 0) >> shift) & group;
        const uint64_t rgt = (__ballot(live && j <= hi && stt == 2) >> shift) & group;
        if (live && fnd) {
            found_lane = __ffsll((long long)fnd) - 1;
            if (g == found_lane) {
                out.i = (int32_t)i;
                out.j = (int32_t)j;
                out.spill = sigma + a.Hw[j] - target;
            }
            live = false;
        } else if (live) {
            if (!wide) {
                live = false;  // no FOUND among the last positions
            } else {
                // RIGHT probes are a prefix of the group: the answer lies
                // after the last of them and before the next probe.
                const int nr = __popcll(rgt);
                const int64_t jl = nr > 0 ? __shfl(j, shift + nr - 1, 64) + 1 : lo;
                const int64_t jh = nr < LANES ? __shfl(j, shift + nr, 64) - 1 : hi;
                lo = jl;
                hi = jh;
                if (lo > hi) live = false;
            }
        }
        if (__ballot(live) == 0ull) break;
    }
    return found_lane;
}

// P-ary split search (SplitMethodParySearch.cu:9-145), PARY_LANES lanes per
// split.  Without the certificate, or when no probe is FOUND, the split is
// resolved by bisection (and counted).
#define PARY_LANES 16
__global__ __launch_bounds__(256) void split_pary(BuildArgs a, int64_t blk0) {
    DevState* st = a.st;
    if (st->error || st->degenerate) return;
    const int g = threadIdx.x % PARY_LANES;
    const int shift = (threadIdx.x & 63) / PARY_LANES * PARY_LANES;  // the group's first lane in the wave
    const int64_t k = ((blk0 + (int64_t)blockIdx.x) * blockDim.x + threadIdx.x) / PARY_LANES + 1;
    const int64_t p = st->p, numL = st->numL, numH = st->numH;
    const bool active = k < p;  // whole groups
    if (k == 1 && g == 0) {
        a.splits[0] = Split{0, 0, 0.0};
        a.splits[p] = Split{(int32_t)(numL - 1), (int32_t)(numH - 1), 0.0};
    }
    const bool cert = u2d(st->cert_max_dL) < u2d(st->cert_min_dH);
    Split out{0, 0, 0.0};
    const int found_lane = pary_search<PARY_LANES>(a, active && cert, k, g, shift, out);
    if (!active) return;
    if (found_lane >= 0) {
        if (g == found_lane) a.splits[k] = out;
    } else if (g == 0) {
        Split sp;
        if (!bisect_split(k, p, st->nToSplit, st->wToSplit, a.Lp, numL, a.Hp, a.Hw, numH, sp))
            atomicAdd((unsigned long long*)&st->split_fallbacks, 1ull);
        a.splits[k] = sp;
        atomicAdd((unsigned long long*)&st->learned_fallbacks, 1ull);
    }
}

// Bisection where many splits are to be found (split_by_group): half a wave
// each searches, 32 positions at a time, for the split before the wave's 64
// (and the last wave for the one after them, too); between those every lane
// finds its own.  Lanes that ask for lines all over the lists one after the
// other are what bisecting the whole lists is bound by.  Under the certificate
// the position found is the bisection's; without it, and where the bracket
// holds none, the lists are bisected.
__global__ __launch_bounds__(256) void split_grouped(BuildArgs a, int64_t blk0) {
    __shared__ int32_t ends[5];  // the heavies of the waves' ends, -1: not found
    DevState* st = a.st;
    if (st->error || st->degenerate || st->p <= a.direct_splits) return;
    const int64_t p = st->p, numL = st->numL, numH = st->numH;
    const int lane = (int)(threadIdx.x & 63), wave = wave_in_block();
    const int64_t k0 = (blk0 + (int64_t)blockIdx.x) * 256 + 64 * wave, k = k0 + 1 + lane;
    if (k0 == 0 && lane == 0) {
        a.splits[0] = Split{0, 0, 0.0};
        a.splits[p] = Split{(int32_t)(numL - 1), (int32_t)(numH - 1), 0.0};
    }
    Split out{0, 0, 0.0};
    bool found = false;
    if (u2d(st->cert_max_dL) < u2d(st->cert_min_dH)) {  // the same in every thread
        const int half = lane >> 5;
        const int64_t ke = k0 + 64 * half;
        Split e{-1, -1, 0.0};
        const int at = pary_search<32>(a, (half == 0 || wave == 3) && ke > 0 && ke < p, ke, lane & 31, half << 5, e);
        if (half == 0 || wave == 3) {
            const bool inside = ke > 0 && ke < p;
            if (inside ? at == (lane & 31) : (lane & 31) == 0) ends[wave + half] = inside ? e.j : ke > 0 ? (int)(numH - 1) : 0;
            if (inside && at < 0 && (lane & 31) == 0) ends[wave + half] = -1;
        }
        __syncthreads();
        const int64_t lo = max(ends[wave], 0), hi = ends[wave + 1] < 0 ? numH - 1 : ends[wave + 1];
        found = k < p && bracket_split(a, k, k0, min(k0 + 64, p), lo, hi, out);
    }
    if (k >= p) return;
    if (!found && !bisect_split(k, p, st->nToSplit, st->wToSplit, a.Lp, numL, a.Hp, a.Hw, numH, out))
        atomicAdd((unsigned long long*)&st->split_fallbacks, 1ull);
    a.splits[k] = out;
}

hipError_t launch_split_grouped_blocks(const BuildArgs& a, hipStream_t s, int64_t b0, int64_t b1) {
    if (b1 > b0) hipLaunchKernelGGL(split_grouped, dim3((unsigned)(b1 - b0)), dim3(256), 0, s, a, b0);
    return hipGetLastError();
}

hipError_t launch_split_grouped(const BuildArgs& a, hipStream_t s) {
    hipError_t e = launch_split_prepare(a, false, s);
    if (e == hipSuccess) e = launch_split_grouped_blocks(a, s, 0, split_blocks(a));
    return e;
}

// Blocks of 256 splits as the other split kernels count them (blocks
// [b0, b1)), 256 / PARY_LANES splits per launched block.
hipError_t launch_split_pary_blocks(const BuildArgs& a, hipStream_t s, int64_t b0, int64_t b1) {
    constexpr int64_t per = 256 / PARY_LANES;
    if (b1 > b0) hipLaunchKernelGGL(split_pary, dim3((unsigned)((b1 - b0) * per)), dim3(256), 0, s, a, b0 * per);
    return hipGetLastError();
}

hipError_t launch_split_pary(const BuildArgs& a, hipStream_t s) {
    hipError_t e = launch_split_prepare(a, false, s);
    if (e == hipSuccess) e = launch_split_pary_blocks(a, s, 0, split_blocks(a));
    return e;
}

hipError_t launch_split_learned_blocks(const BuildArgs& a, hipStream_t s, int64_t b0, int64_t b1) {
    if (b1 > b0) hipLaunchKernelGGL(split_learned, dim3((unsigned)(b1 - b0)), dim3(256), 0, s, a, b0);
    return hipGetLastError();
}

hipError_t launch_split_learned(const BuildArgs& a, hipStream_t s) {
    hipError_t e = launch_split_prepare(a, true, s);
    if (e == hipSuccess) e = launch_split_learned_blocks(a, s, 0, split_blocks(a));
    return e;
}

}  // namespace atg

// The whole construction of a small table by one workgroup, its lists in LDS:
// one launch instead of eight or more, and no global round trip between the
// phases.  The same canonical association as the kernels of atg_build.hip,
// so the same rows, lists and splits.
//
// A section has a wave (so at most as many sections as waves), a split and a
// pack chain a thread.  Each phase ends at a barrier that every thread of the
// workgroup reaches; nothing waits for another workgroup.
// Bound by latency, much of it that of fetching instructions: each launch
// runs through the code about once, so loops stay loops (the classes of a
// list, the chunks of a section) and a kernel holds as few chunks of a
// section as its sections have.
#pragma once

#include "atg_kernels.h"

namespace atg {

// LDS of a table of n items and p_req requested splits.  The section weights
// and, later, the prefixes share one array; the list weights and items have
// their own unless the build is compact.
struct SmallLds {
    int64_t items;  // entries of a list array: n items and two sentinels, even
    int64_t splits;
    __host__ __device__ SmallLds(int64_t n, int64_t p_req) : items((n + 3) & ~(int64_t)1), splits(p_req + 1) {}
    __host__ __device__ size_t bytes() const { return (size_t)items * (8 + 8 + 2 + 2) + (size_t)splits * 16; }
    __host__ __device__ size_t compact_bytes() const { return (size_t)items * (8 + 2) + (size_t)splits * 16; }
};

// Tables built by seg_small, in classes by their sections' length (kSmallChunks
// chunks of 64 items a lane) and number (waves, a power of two) and by how
// many tables fit a CU (one, two, more).  A class has one launch, with the LDS
// of its largest table, so that small tables are not held to the occupancy of
// larger ones; finer classes lose more at the ends of their launches than
// occupancy gains (16,384 tables of 16 to 4,096 items 230 us, 238 with four
// more tiers of LDS below 32 KB).
constexpr int kSmallChunks[] = {2, 8, 16, 32};
constexpr size_t kSmallTiers[] = {52 * 1024, 79 * 1024, 154 * 1024};  // of 160 KB, static LDS aside
struct SmallClass {
    int xu;            // index into kSmallChunks
    int waves, tier;
    int threads = 64;  // of the table with the most sections
    size_t lds = 0;    // of the largest table
};
// The class of a table of n items in G sections of Ls, false: not small.  Small
// tables have a wave per section and fit a CU's LDS.
inline bool small_class_of(int64_t n, int64_t G, int64_t Ls, int64_t p_req, SmallClass& c) {
    if (G > (Ls <= kShortSectionMax ? kSmallMaxWaves : kSmallLongWaves)) return false;
    c.xu = 0;
    c.waves = 1;
    c.tier = 0;
    while (Ls > 64 * kSmallChunks[c.xu]) ++c.xu;
    while (G > c.waves) c.waves *= 2;
    c.lds = SmallLds(n, p_req).compact_bytes();
    while (c.tier < 2 && c.lds > kSmallTiers[c.tier]) ++c.tier;
    return c.lds <= kSmallTiers[2];
}

// Whether a group's small tables, so many sections of so many classes, pay for
// launches of their own beside the phases of its other tables: the fork, the
// launches and the join cost 15 to 20 us and each class some more, and the
// phases take a wave per section.  In the phases and so, us, with few larger
// tables beside: 64 tables of 11 sections, one class 57 and 73; 2,000 of one
// section 75 and 80, 10,000 255 and 112; 400 of 11 sections 93 and 73.  Sizes
// log-uniform over a hundredfold or more, sections by classes and two: 47 by 10
// 57 and 137, 459 by 9 67 and 152, 2,680 by 9 332 and 381, 5,593 by 7 267 and
// 261, 7,610 by 10 234 and 204, 22,595 by 7 311 and 206.
inline bool small_beside_ok(int64_t sections, int classes) { return sections >= 640 * (int64_t)(classes + 2); }

// The light list followed by the heavy list (from entry numL) in LDS.
struct SmallLists {
    const double* w;
    const uint16_t* item;
    int numL;
    __device__ int li(int i) const { return item[i]; }
    __device__ double lw(int i) const { return w[i]; }
    __device__ int hi(int j) const { return item[numL + j]; }
    __device__ double hw(int j) const { return w[numL + j]; }
};

// Chunks c0 .. c0 + U - 1 of a section's leftovers into registers: cL chunks of
// 64 lights, then the heavies.  lo, off: first position and rank of each
// chain's leftovers (chain_positions), the lights' in the low halves; the
// chunks' searches run interleaved.
template <int U>
__device__ __forceinline__ void list_chunks(SecLDS& L, int c0, int cL, int mL, int mH, int lane, bool chains,
                                            uint32_t lo, uint32_t off, int first, int64_t start, double* w,
                                            uint16_t* item) {
    int r[U], t[U], sh[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
        const bool hv = c0 + u >= cL;
        r[u] = ((hv ? c0 + u - cL : c0 + u) << 6) + lane;
        sh[u] = hv ? 16 : 0;
        t[u] = 0;
    }
    if (chains) {
        for (int step = first; step >= 1; step >>= 1) {
            int o[U];
#pragma unroll
            for (int u = 0; u < U; ++u) o[u] = __shfl((int)off, t[u] + step, 64);
#pragma unroll
            for (int u = 0; u < U; ++u) t[u] += (int)((uint32_t)o[u] >> sh[u] & 0xFFFFu) <= r[u] ? step : 0;
        }
    }
#pragma unroll
    for (int u = 0; u < U; ++u) {
        int pos = r[u];
        if (chains) {
            const uint32_t b = (uint32_t)__shfl((int)lo, t[u], 64), c = (uint32_t)__shfl((int)off, t[u], 64);
            pos = (int)(b >> sh[u] & 0xFFFFu) + r[u] - (int)(c >> sh[u] & 0xFFFFu);
        }
        if (r[u] < (sh[u] ? mH : mL)) {
            w[u] = sh[u] ? L.Hw(pos) : L.Lw(pos);
            item[u] = (uint16_t)(start + (sh[u] ? L.Hi(pos) : L.Li(pos)));
        }
    }
}

// XU: weights a lane holds (sections of up to 64 XU items).  LISTS: the lists
// and splits go to HBM as well (for the copy-out of a single table).
// W_out, error_out: nullable copies of the state's fields.
// COMPACT: for many tables at once, whose number in flight the LDS bounds.
// One array holds the section weights, then the prefixes, then the list
// weights, which wait in registers meanwhile.
template <typename T, bool AOS, int XU, bool LISTS, bool COMPACT>
__device__ __forceinline__ void small_build(const BuildArgs& a, double* W_out, uint32_t* error_out, double* lds) {
    __shared__ double ssum[kSmallMaxWaves], sagg[2][kSmallMaxWaves];
    __shared__ uint32_t scnt[2][kSmallMaxWaves];
    __shared__ uint32_t sfall;
    const SmallLds lay(a.n, a.p_req);
    double* A = lds;              // section weights, then prefixes (lights, then heavies)
    double* B = COMPACT ? A : A + lay.items;  // list weights
    Split* sp = reinterpret_cast<Split*>(B + lay.items);
    uint16_t* idx = reinterpret_cast<uint16_t*>(sp + lay.splits);  // section items, local to the section
    uint16_t* item = COMPACT ? idx : idx + lay.items;              // list items
    const int tid = (int)threadIdx.x, lane = tid & 63, wave = wave_in_block();
    const int G = (int)a.G, s = wave;
    const bool has = s < G;
    const int64_t start = min(a.n, s * a.Ls);
    const int len = has ? (int)(min(a.n, (s + 1) * a.Ls) - start) : 0;

    // 1. The section's weights and their sum (section_sum's order).
    T x[XU];
    if (has) section_load<T>(a, s, lane, x);
    {
        double acc = 0.0;
        bool bad = false;
#pragma unroll
        for (int u = 0; u < XU; ++u) {
            if ((u << 6) + lane < len) {
                const double v = (double)x[u];
                bad |= !(v >= 0.0) || (v == __builtin_inf());
                acc = acc + v;
            }
        }
        double sum = wave_tree_sum(acc);
        if (__ballot(bad) != 0ull) sum = __builtin_nan("");
        if (has && lane == 0) ssum[s] = sum;
        if (tid == 0) sfall = 0u;
    }
    __syncthreads();
    const double W = wave_tree_sum(lane < G ? ssum[lane] : 0.0);
    const double W_N = W / (double)a.n;
    const uint32_t err = sum_error(a, W);
    if (tid == 0) {
        sum_state(a, W);
        if (W_out) *W_out = W;
        if (error_out) *error_out = err;
    }
    if (err) return;  // the same in every thread

    // 2. Stable partition, chains, leftover counts (psa_section's).
    SecLDS L;
    L.w = A + start;
    L.idx = idx + start;
    L.len = len;
    int iLo = 0, iHi = 0, jLo = 0, jHi = 0, offL = 0, offH = 0, mL = 0, mH = 0;
    if (has) {
        const uint64_t lt = lanemask_lt();
        int nL = 0, nH = 0;
#pragma unroll
        for (int u = 0; u < XU; ++u) {
            if ((u << 6) < len) {
                const int k = (u << 6) + lane;
                const double xv = (double)x[u];
                const bool valid = k < len, light = valid && xv <= W_N;
                const uint64_t bl = __ballot(light), bh = __ballot(valid && !light);
                const int slot = light ? nL + __popcll(bl & lt) : len - 1 - (nH + __popcll(bh & lt));
                if (valid) {
                    L.w[slot] = xv;
                    L.idx[slot] = (uint16_t)k;
                }
                nL += __popcll(bl);
                nH += __popcll(bh);
            }
        }
        wave_lds_sync();
        if (a.psa_plus) {
            chain_ranges(a, nL, nH, lane, iLo, iHi, jLo, jHi);
            psa_chain_rows<AOS>(a, L, start, W_N, iHi - iLo > 0 && jHi - jLo > 0, iLo, iHi, jLo, jHi);
        } else if (lane == 0) {
            iHi = nL;
            jHi = nH;
        }
        const int cl = iHi - iLo, ch = jHi - jLo;
        const uint32_t cp = (uint32_t)cl | ((uint32_t)ch << 16);
        const uint32_t incl = wave_incl_scan_u32(cp), excl = incl - cp;
        const uint32_t tot = (uint32_t)__builtin_amdgcn_readlane((int)incl, 63);
        offL = (int)(excl & 0xFFFFu);
        offH = (int)(excl >> 16);
        mL = (int)(tot & 0xFFFFu);
        mH = (int)(tot >> 16);
        if (lane == 0) {
            scnt[0][s] = (uint32_t)mL;
            scnt[1][s] = (uint32_t)mH;
        }
        wave_lds_sync();
    }
    __syncthreads();

    // 3. The lists in rank order: lights [0, numL), heavies from numL on, the
    //    sentinels last (AliasTableSplitGpu.cu:366-385).
    const uint32_t inclL = wave_incl_scan_u32(lane < G ? scnt[0][lane] : 0u);
    const uint32_t inclH = wave_incl_scan_u32(lane < G ? scnt[1][lane] : 0u);
    const int nLr = __builtin_amdgcn_readlane((int)inclL, 63), nHr = __builtin_amdgcn_readlane((int)inclH, 63);
    const int numL = nLr + 1, numH = nHr + 1;
    const int sl = has ? s : 0;
    const int goffL = __builtin_amdgcn_readlane((int)inclL, sl) - mL;
    const int goffH = numL + __builtin_amdgcn_readlane((int)inclH, sl) - mH;
    int first = 1;
    while (2 * first < a.chains) first *= 2;
    double tot[2] = {0.0, 0.0};
    // Compact builds: the section's list entries, the lights' chunks first.
    constexpr int GS = XU < 16 ? 3 : 4;  // chunks taken together
    constexpr int NC = COMPACT ? (XU + 1 + GS - 1) / GS * GS : 1;
    double lw[NC] = {};
    uint16_t it[NC] = {};
    const int cL = (mL + 63) >> 6, cAll = cL + ((mH + 63) >> 6);
    if constexpr (COMPACT) {
        // 3. The section's list entries into registers, then, the section
        //    weights all read, 4. their local prefixes and items into place
        //    and P(s) added.
        static_assert(!LISTS, "list weights are not kept");
        const uint32_t lo = (uint32_t)iLo | ((uint32_t)jLo << 16), off = (uint32_t)offL | ((uint32_t)offH << 16);
#pragma unroll
        for (int c0 = 0; c0 < NC; c0 += GS) {
            if (c0 < cAll) list_chunks<GS>(L, c0, cL, mL, mH, lane, a.psa_plus, lo, off, first, start, &lw[c0], &it[c0]);
        }
        __syncthreads();
        double carry = 0.0, aggL = 0.0;
#pragma unroll
        for (int c0 = 0; c0 < NC; c0 += GS) {
            if (c0 >= cAll) continue;
            double inc[GS];
#pragma unroll
            for (int u = 0; u < GS; ++u) inc[u] = wave_scan(lw[c0 + u]);
#pragma unroll
            for (int u = 0; u < GS; ++u) {
                const int c = c0 + u;
                const bool hv = c >= cL;
                const int r = ((hv ? c - cL : c) << 6) + lane, dst = hv ? goffH : goffL;
                // The lights' aggregate ends where the heavies' begins; chunks
                // past the lists add zeros.
                if (c == cL && cL < cAll) {
                    aggL = carry;
                    carry = 0.0;
                }
                const double local = carry + wave_shr1(inc[u]);
                if (r < (hv ? mH : mL)) {
                    A[dst + r] = local;
                    item[dst + r] = it[c];
                }
                carry = carry + readlane_d(inc[u], 63);
            }
        }
        if (cL >= cAll) {  // no heavies
            aggL = carry;
            carry = 0.0;
        }
        if (has && lane == 0) {
            sagg[0][s] = aggL;
            sagg[1][s] = carry;
        }
        __syncthreads();
#pragma unroll 1
        for (int hv = 0; hv < 2; ++hv) {
            const double g = lane < G ? sagg[hv][lane] : 0.0;
            const double P = fold_blocks<5>(0.0, g, s, lane), Q = fold_blocks<5>(0.0, g, G, lane);
            if (hv) tot[1] = Q;
            else tot[0] = Q;
            const int m = hv ? mH : mL, dst = hv ? goffH : goffL;
            for (int r = lane; r < m; r += 64) A[dst + r] = P + A[dst + r];
        }
        if (tid == 0) {
            item[nLr] = (uint16_t)(a.n + 1);
            item[numL + nHr] = (uint16_t)a.n;
        }
    } else {
        if (has) {
            constexpr int U = XU < 4 ? XU : 4;
    #pragma unroll 1
            for (int hv = 0; hv < 2; ++hv) {
                const int m = hv ? mH : mL, dst = hv ? goffH : goffL;
    #pragma unroll 1
                for (int g0 = 0; g0 < m; g0 += 64 * U) {
                    int pos[U];
                    if (a.psa_plus) {
                        chain_positions<U>(g0 + lane, hv ? offH : offL, hv ? jLo : iLo, pos, first);
                    } else {
    #pragma unroll
                        for (int u = 0; u < U; ++u) pos[u] = g0 + 64 * u + lane;
                    }
    #pragma unroll
                    for (int u = 0; u < U; ++u) {
                        const int r = g0 + 64 * u + lane;
                        if (r < m) {
                            B[dst + r] = hv ? L.Hw(pos[u]) : L.Lw(pos[u]);
                            item[dst + r] = (uint16_t)(start + (hv ? L.Hi(pos[u]) : L.Li(pos[u])));
                        }
                    }
                }
            }
        }
        if (tid == 0) {
            B[nLr] = 0.0;
            item[nLr] = (uint16_t)(a.n + 1);
            B[numL + nHr] = __builtin_inf();
            item[numL + nHr] = (uint16_t)a.n;
        }
        __syncthreads();

        // 4. Local prefixes into A (the section weights are all in B by now), the
        //    sections' aggregates, then P(s) + local.
        if (has) {
    #pragma unroll 1
            for (int hv = 0; hv < 2; ++hv) {
                const int m = hv ? mH : mL, dst = hv ? goffH : goffL;
                double carry = 0.0;
    #pragma unroll 1
                for (int r0 = 0; r0 < m; r0 += 64) {
                    const int r = r0 + lane;
                    const double inc = wave_scan(r < m ? B[dst + r] : 0.0);
                    const double local = carry + wave_shr1(inc);
                    if (r < m) A[dst + r] = local;
                    carry = carry + readlane_d(inc, 63);
                }
                if (lane == 0) sagg[hv][s] = carry;
            }
        }
        __syncthreads();
    #pragma unroll 1
        for (int hv = 0; hv < 2; ++hv) {
            const double v = lane < G ? sagg[hv][lane] : 0.0;
            const double P = fold_blocks<5>(0.0, v, s, lane), Q = fold_blocks<5>(0.0, v, G, lane);
            if (hv) tot[1] = Q;
            else tot[0] = Q;
            if (has) {
                const int m = hv ? mH : mL, dst = hv ? goffH : goffL;
    #pragma unroll 1
                for (int r = lane; r < m; r += 64) {
                    const double pref = P + A[dst + r];
                    A[dst + r] = pref;
                    if (LISTS) {
                        const int g = hv ? dst + r - numL : dst + r;
                        (hv ? a.Hi : a.Li)[g] = (int32_t)item[dst + r];
                        (hv ? a.Hw : a.Lw)[g] = B[dst + r];
                        (hv ? a.Hp : a.Lp)[g] = pref;
                    }
                }
            }
        }
    }
    const bool degenerate = nLr == 0 || nHr == 0;
    int64_t p = a.p_req;
    if (a.psa_plus) { p = min<int64_t>(p, (numL + numH) / 10); if (p < 2) p = 2; }
    const int64_t nToSplit = numL + numH - 2;
    const double wToSplit = tot[0] + tot[1];
    if (tid == 0) {
        A[nLr] = tot[0];
        A[numL + nHr] = tot[1];
        DevState* st = a.st;
        st->numL = numL;
        st->numH = numH;
        st->degenerate = degenerate ? 1u : 0u;
        st->p = degenerate ? 0 : p;
        st->nToSplit = nToSplit;
        st->wToSplit = wToSplit;
        if (LISTS) {
            a.Li[nLr] = (int32_t)(a.n + 1); a.Lw[nLr] = 0.0; a.Lp[nLr] = tot[0];
            a.Hi[nHr] = (int32_t)a.n; a.Hw[nHr] = __builtin_inf(); a.Hp[nHr] = tot[1];
        }
    }
    __syncthreads();

    if (degenerate) {  // the same in every thread
        // Every leftover row carries its own mass.
        if constexpr (COMPACT) {
#pragma unroll
            for (int c = 0; c < NC; ++c) {
                const int r = ((c >= cL ? c - cL : c) << 6) + lane;
                if (r < (c >= cL ? mH : mL)) store_row<AOS>(a, it[c], lw[c], (int32_t)it[c]);
            }
            return;
        }
        for (int t = tid; t < nLr + nHr; t += (int)blockDim.x) {
            const int e = t < nLr ? t : t + 1;  // past the light sentinel
            store_row<AOS>(a, item[e], B[e], (int32_t)item[e]);
        }
        return;
    }

    // 5. Splits, a thread each.
    for (int64_t k = tid; k <= p; k += blockDim.x) {
        Split r;
        if (k == 0) {
            r = Split{0, 0, 0.0};
        } else if (k == p) {
            r = Split{numL - 1, numH - 1, 0.0};
        } else if (COMPACT ? !bisect_split(k, p, nToSplit, wToSplit, A, numL, A + numL, SpillLater{}, numH, r)
                           : !bisect_split(k, p, nToSplit, wToSplit, A, numL, A + numL, B + numL, numH, r)) {
            atomicAdd(&sfall, 1u);
        }
        sp[k] = r;
        if (LISTS) a.splits[k] = r;
    }
    __syncthreads();
    if constexpr (COMPACT) {
        // The list weights over the prefixes, then the splits' spills.
#pragma unroll
        for (int c = 0; c < NC; ++c) {
            const bool hv = c >= cL;
            const int r = ((hv ? c - cL : c) << 6) + lane;
            if (r < (hv ? mH : mL)) A[(hv ? goffH : goffL) + r] = lw[c];
        }
        if (tid == 0) {
            A[nLr] = 0.0;
            A[numL + nHr] = __builtin_inf();
        }
        __syncthreads();
        for (int64_t k = tid; k < p; k += blockDim.x)
            if (k > 0) sp[k].spill = sp[k].spill + A[numL + sp[k].j] - split_target(k, p, nToSplit, wToSplit);
        __syncthreads();
    }

    // 6. Pack chains, a thread each.
    const SmallLists lists{B, item, numL};
    for (int64_t k = tid; k < p; k += blockDim.x) pack_chain<AOS>(a, lists, sp[k], sp[k + 1], W_N);
    if (tid == 0 && sfall != 0u) a.st->split_fallbacks = sfall;
}

}  // namespace atg

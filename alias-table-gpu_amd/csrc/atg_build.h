// Host-visible description of one build and the launchers of its phases.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "atg_types.h"

namespace atg {

// Pack methods (the values of atg_pack_method).
enum PackMethod : int32_t { PACK_CHUNKED = 0, PACK_BASIC = 1, PACK_NO_WEIGHTS = 2 };

// Everything a build kernel needs, passed by value (all device pointers).
struct BuildArgs {
    const void* weights;  // n weights (double or float)
    int dtype_f32;
    int64_t n;
    int64_t G;            // sections
    int64_t Ls;           // items per section
    int64_t Ls_max;       // LDS capacity of the partition kernel (items per section)
    int64_t tree_total;   // blocks of the dyadic section-prefix tree (sum over b of G >> b)
    DevState* st;
    double* section_sums;     // G
    double* tree_scratch;     // 2 * tree_scratch_half
    int64_t tree_scratch_half;
    uint64_t* slots;          // dyadic block sums (counts, light, heavy)
    double* stage_w;          // n: leftovers staged by partition pass 1 (weights)
    int32_t* stage_i;         // n: leftovers staged by partition pass 1 (items)
    uint64_t* sec_cert;       // 6 G: per-section split-certificate data (bit patterns)
    int32_t want_cert;        // compute the split certificate (learned, P-ary and grouped splits)
    int32_t* Li; double* Lw; double* Lp;  // leftover lights (capacity n + 2)
    int32_t* Hi; double* Hw; double* Hp;  // leftover heavies (capacity n + 2)
    Row* rows;                // AoS table or null
    double* tw; int32_t* ta;  // SoA table or null
    int32_t psa_plus;
    int32_t chains;
    uint32_t chain_mul;       // chain_multiplier(chains)
    int64_t p_req;            // p after the N/10 clamp (grid bound for split/pack)
    Split* splits;            // capacity p_req + 1
    int32_t pack_cap;         // list items one pack wave stages in LDS (pack_cap_items)
    // learned split index
    int32_t learned_segments;
    int32_t* knot_j;          // learned_segments + 1 exact split j at the knots
    int64_t direct_splits;    // up to this many splits launch_split_prepare finds by bisection
    int32_t pack_method;      // atg_pack_method
    // Lean light lists: the placement writes only the light prefixes; the
    // light items and weights stay in the staging, found through sec_loff
    // (G + 1 values: the lights before section s, then the light count).
    int32_t lean_lights;
    uint32_t* sec_loff;
    uint32_t* sec_ldir;       // light_dir_size(n): the section of light q << kLightDirShift
};

constexpr int kLightDirShift = 10;
inline int64_t light_dir_size(int64_t n) { return (n >> kLightDirShift) + 2; }

// The windowed pack runs every chain (of up to n / p items) at once; the staged
// one as many as fit its pool, so in rounds whose number grows with n / p, and
// the more waves there are, the more of that they hide for each other.  Builds
// with few and with many lights to a heavy, staged / windowed, us: 1e6 items
// at n / p = 33 69.6 / 67.2 and 76.4 / 72.2; 3e6 at 50 105.6 / 100.8 and 115.6
// / 111.1; 1e7 at 64 (staged by the rule) 237.8 / 244.2 and 283.2 / 258.6; 3e7
// at 100 670 / 658 and 754 / 664; 1e8 at 100 (staged) 2,080 / 2,128 and 2,261 /
// 2,120, at 150 2,041 / 2,062 and 2,542 / 2,141, at 200 2,077 / 2,055 and 2,826
// / 2,116.
// The card holds 3,072 of its waves, kWindowRound chains (12 of 13 KB of LDS a
// CU).  Up to half a round more, most of the card waits for the few left over,
// which only longer chains outweigh (Pareto and the mix of heavies, sections
// of 2048, 110,000 chains: 7e6 items 159 / 181 and 149 / 164, 1.1e7 250 / 269
// and 218 / 237, 1.4e7 316 / 317 and 270 / 280; over twelve distributions and
// shapes the windowed builds take 1.07, 1.04 and 0.97 of the staged ones, of
// 80,000 and 160,000 chains at n / p = 100 0.95 and 0.94).
constexpr int64_t kWindowRound = 3072 * 32;
// Lists that fit the staged pack's pool (1,024 items) at once or nearly are
// staged at once (whole builds, windowed by
// staged: 1,000 items at n / p = 100 1.1 to 1.8, at 200 1.1 to 1.4; 2,000 0.8 to
// 1.2 at 64, 1.1 to 1.6 at 200; 3,000 0.65 to 1.1 at 64).
constexpr int64_t kWindowMinItems = 2048;
inline bool pack_windowed_ok(int64_t n, int64_t p_req, int32_t pack_method) {
    if (pack_method != PACK_CHUNKED || p_req <= 0) return false;
    const int64_t per = n / p_req;
    if (per > 256) return true;
    const bool tail = p_req > kWindowRound && 2 * p_req < 3 * kWindowRound;
    return n > kWindowMinItems && per >= 32 && (tail ? 7 : 30) * per * per > p_req;
}
// Tables below this many items keep whole lists: finding a light in the
// staging takes the pack a few dependent reads, which the smaller writes pay
// for only where bandwidth counts (builds, us, lean against whole: 100,003
// items 51.3 and 46.0, 2^20 71.1 and 71.0, 3e6 95.2 and 95.1, 1e7 244 and 253;
// with the windowed pack 3e6 113.0 and 110.7, 5e6 158.2 and 159.0, 1e7 235.8
// and 241.4, 1e8 of R/N = 0.62 and 0.90 1,977 and 2,159, 1,990 and 2,295).
constexpr int64_t kLeanMin = (int64_t)1 << 21, kLeanMinWindowed = (int64_t)1 << 22;
inline bool lean_lights_ok(int64_t n, int64_t p_req, int32_t pack_method) {
    return pack_method == PACK_CHUNKED && p_req > 0 && n >= (pack_windowed_ok(n, p_req, pack_method) ? kLeanMinWindowed : kLeanMin);
}

// A batch packs with the staged kernel alone, whose LDS pool every chain of
// a lean list has to fit (chains hold at most n / p + 3 items, the pool at
// least min(64 (n / p + 1), 1024)).  Its tables share the card's bandwidth, so
// they are lean at any size (us, lean against whole: 2,000 tables of 20,000
// items 1,067 and 1,112, 512 of 200,000 2,404 and 2,507, 100 of 1e6 2,720 and
// 2,800).
inline bool batch_lean_ok(int64_t n, int64_t p_req) { return p_req > 0 && n / p_req <= 256; }

// x / chains = x chain_mul >> 20 for x <= 2048 and chains <= 64: with M =
// ceil(2^20 / C), x (M C - 2^20) < 2048 64 < 2^20.
inline uint32_t chain_multiplier(int32_t chains) { return ((1u << 20) + (uint32_t)chains - 1) / (uint32_t)chains; }

// Section layout of PSA+ (AliasTableSplitGpu.cu:356-357, PsaPlusNormal.cu:27-29).
inline void section_layout(int64_t n, int64_t param, int64_t* G, int64_t* Ls) {
    if (param < 1) param = 1;
    *G = n / param + 1;
    *Ls = n / *G + 1;
}

// Items of the LDS pool of one pack wave: the items of all its 64 chains
// when they fit (splits are evenly spaced in list items, n' = ceil(nToSplit
// k / p), so 64 chains hold at most 64 ceil(nToSplit / p) + 1 items, with
// nToSplit <= n + 2 and chains near 10 items when p is clamped below p_req),
// at most kPackPoolItems; a wave whose chains need more runs them in rounds.
constexpr int32_t kPackPoolItems = 1024;
inline int32_t pack_cap_items(int64_t n, int64_t p_req) {
    if (p_req < 1) p_req = 1;
    int64_t per = (n + 2 + p_req - 1) / p_req;
    if (per < 11) per = 11;
    int64_t cap = (64 * (per + 1) + 2 + 15) / 16 * 16;
    return (int32_t)(cap < kPackPoolItems ? cap : kPackPoolItems);
}
// A pack round that fits fewer chains than this into the pool, and not all of
// the wave's, hands the chains that are left to their lanes, each reading the
// lists from HBM (a wave's chains that all fit are staged: whole builds of 500
// and 1,000 items in two to five chains 45 -> 34 us).
constexpr int kPackMinStagedChains = 8;
// Weight (8 B), item (4 B) and recorded alias (4 B) per pool item, and the
// spare weight slot the light steps record into (16 B keep the alignment).
inline size_t pack_lds_bytes(int32_t cap) { return (size_t)cap * 16 + 16; }

// A split by four lanes, which look two levels of the bisection ahead: half
// the dependent reads for half as many probes again.  Pays while the reads
// wait for nothing else (whole builds, us: 100,003 items with 10,000 splits
// 54.6 -> 51.0, 3e5 items with 30,000 57.6 -> 55.3; 2^20 items with 81,920
// 70.6 -> 71.2).  The lanes keep positions in 32 bits.
constexpr int kWideLevels = 2;
inline bool split_wide_ok(int64_t n, int64_t p_req) { return p_req <= (1 << 15) && n <= ((int64_t)1 << 29); }

// Knots of the learned split index: at most `opt`, and at most one per 16
// requested splits (at least 64).  Each knot is a full bisection, so a table
// with few splits would otherwise bisect nearly every split twice; the
// splits found are the same for any knot count.
inline int32_t learned_knots(int32_t opt, int64_t p_req) {
    const int64_t k = p_req / 16 > 64 ? p_req / 16 : 64;
    return (int32_t)(k < opt ? k : opt);
}

// LDS of one partition wave: weights (8 B) and local item indices (2 B), and
// at least eight weights to read past the last.
inline size_t psa_lds_bytes(int64_t Ls_max) {
    const size_t need = (size_t)Ls_max * 10, past = ((size_t)Ls_max + 8) * 8;
    return ((need > past ? need : past) + 15) & ~(size_t)15;
}
// Sections of at most this many items run the partition kernel that holds
// half the weight registers.
constexpr int64_t kShortSectionMax = 1024;
// Rows written after the chains rather than by each of their steps: pays
// where the device is full of sections and the rows go to HBM (1e8 items at
// sections of 2048: the pass takes 0.74 against 0.82 ms; uniform weights at
// sections of 1000: 0.74 against 1.12), costs the extra pass over the section
// where each has a wave to itself from the start (101 sections: 21 against 18
// us; 1,049 sections: the same).  16-byte rows that fit the 256 MB of the
// Infinity Cache are joined there anyway, and then only short sections, four
// waves a SIMD, hide the pass (builds, later / by step, 5e6 to 1.4e7 items:
// sections of 2048, 16 chains 1.15-1.22 uniform, 1.09-1.16 exponential, 0.97-1.02
// Pareto, 0.95 heavy mix; sections of 1000 0.96-1.05, 0.93-1.01, 0.95-1.02,
// 0.95; 2e7 and more at 2048 1.03-1.09, 0.88-1.07, 0.95-1.05, 0.92).  Split rows,
// 8 and 4 bytes, come in smaller pieces and pay at any size (sections of 1000
// 0.71-0.88 uniform and exponential).
constexpr int64_t kCachedRows = (int64_t)1 << 24;
inline bool rows_later_ok(int64_t sections, int64_t resident, bool aos, int64_t n, int64_t Ls_max) {
    return sections > resident && (!aos || n > kCachedRows || Ls_max <= kShortSectionMax);
}
// A batch's kernel holds sections of any length at two waves a SIMD: it hides
// the pass nowhere, and short chains leave it nothing to gain (later / by step:
// sections of 1000 0.98-1.12 at any size; of 2048, 32 chains 0.99-1.06 up to 2e7
// items, 0.84-0.95 uniform and exponential, 1.0-1.04 Pareto from 6e7).
inline bool batch_rows_later_ok(int64_t sections, int64_t resident, int64_t items, int64_t Ls_max) {
    return sections > resident && items > kCachedRows && Ls_max > kShortSectionMax;
}
int64_t resident_blocks(const void* f, int threads, size_t lds);
// Up to this many sections the placement folds P(s) from the sections' own
// sums, without the tree's launches (builds, us, with and without the tree:
// 101 sections 46.1 and 43.1, 1,049 sections 70.4 and 66.1, 3,001 sections
// 94.2 and 97.6: a wave reads up to 24 bytes per section before its own).
constexpr int64_t kDirectPrefixMax = 2048;
int64_t block_tree_total(int64_t G);
hipError_t launch_sum(const BuildArgs& a, hipStream_t s);
hipError_t launch_partition(const BuildArgs& a, hipStream_t s);
// launch_sum and launch_partition, up to kOwnSumMax sections without the
// launch that finishes the sum: every partition wave does, while its weights
// are on their way (builds, us: 100,003 items 43.8 -> 40.6, 2^20 65.1 -> 63.0).
constexpr int64_t kOwnSumMax = 2048;
hipError_t launch_front(const BuildArgs& a, hipStream_t s);
hipError_t launch_partition_local(const BuildArgs& a, hipStream_t s);
hipError_t launch_partition_place(const BuildArgs& a, hipStream_t s);
// What the learned and P-ary splits and chunked splits start from: the
// certificate (with want_cert), the knots on request, and a degenerate table's
// rows.  launch_front leaves the certificate to it; launch_partition and
// launch_partition_place, the phases by themselves, compute it too.
hipError_t launch_split_prepare(const BuildArgs& a, bool knots, hipStream_t s);
hipError_t launch_split(const BuildArgs& a, hipStream_t s);
hipError_t launch_split_learned(const BuildArgs& a, hipStream_t s);
hipError_t launch_split_pary(const BuildArgs& a, hipStream_t s);
hipError_t launch_split_grouped(const BuildArgs& a, hipStream_t s);
hipError_t launch_pack(const BuildArgs& a, hipStream_t s);
// Lean light lists written out as lists (Li, Lw) from the staging.
hipError_t launch_lean_lights_fill(const BuildArgs& a, hipStream_t s);
// Chunked split and pack (split/pack interleave): blocks [b0, b1) of
// split_blocks (256 splits each) or pack_blocks (64 chains each).
int64_t split_blocks(const BuildArgs& a);
int64_t pack_blocks(const BuildArgs& a);
int64_t fill_blocks(int64_t n);
hipError_t launch_split_blocks(const BuildArgs& a, hipStream_t s, int64_t b0, int64_t b1);
hipError_t launch_split_learned_blocks(const BuildArgs& a, hipStream_t s, int64_t b0, int64_t b1);
hipError_t launch_split_grouped_blocks(const BuildArgs& a, hipStream_t s, int64_t b0, int64_t b1);
hipError_t launch_split_pary_blocks(const BuildArgs& a, hipStream_t s, int64_t b0, int64_t b1);
hipError_t launch_pack_blocks(const BuildArgs& a, hipStream_t s, int64_t b0, int64_t b1);
hipError_t launch_split_rows(const Row* rows, double* w, int32_t* al, int64_t n, hipStream_t s);
hipError_t launch_join_rows(const double* w, const int32_t* al, Row* rows, int64_t n, hipStream_t s);


// A whole build by one workgroup with its lists in LDS (atg_small.h): the
// state, rows, splits and (with lists) the leftover lists that the phases
// above leave, in one launch.  W_out, error_out: nullable device copies.
constexpr int kSmallMaxWaves = 16;  // waves of a workgroup, one per section: sections of up to 1024 items
constexpr int kSmallLongWaves = 4;  // longer ones
constexpr int64_t kSmallMaxItems = 8192;
constexpr size_t kSmallLdsMax = 156 * 1024;  // of 160 KB, static LDS aside
constexpr size_t kSmallLdsDefault = 63 * 1024;  // more, the static LDS aside, a kernel has to be allowed first
bool small_build_ok(int64_t n, int64_t G, int64_t Ls, int64_t p_req);
hipError_t launch_small(const BuildArgs& a, bool lists, double* W_out, uint32_t* error_out, hipStream_t s);

}  // namespace atg

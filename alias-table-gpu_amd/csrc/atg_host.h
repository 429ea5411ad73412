// Host-side helpers shared by the C ABI translation units: error reporting,
// device queries and the limits of the kernels.
#pragma once

#include <hip/hip_runtime.h>

#include <cstddef>

#include "../../include/atg.h"
#include "atg_build.h"
#include "atg_types.h"

namespace atg {

// Records a thread-local message (atg_last_error) and returns `st`.
atg_status fail(atg_status st, const char* fmt, ...);
// Compute units of the current device (256 on MI355X).
int device_cus();
// Maps DevState::error bits to a status and message.
atg_status state_status(const DevState& st);
// Sets the chain count and requested splits of a created table in place.
atg_status table_set_shape(atg_table* t, int32_t chains, int64_t num_splits);
// Whether a bisection is done wave by wave inside brackets (split_grouped),
// which needs the split certificate.  Builds, us, over the whole lists and so:
// 1e7 items, 417,000 splits 257 and 232, 156,000 257 and 256, 82,000 244 and
// 252; 3e7 items, 469,000 653 and 593; 1e8, 500,000 1,853 and 1,790, 1.6e6 2,001
// and 1,748, 4.2e6 2,098 and 1,804; where the certificate fails, 3e7 and 1.2e6
// 723 and 748, 1e8 and 2.6e6 2,209 and 2,234.  A table that turns out to have
// fewer than half of the line (many items finished by the partition) is
// bisected in the certificate's launch.
constexpr int64_t kGroupedSplits = (int64_t)1 << 18;
inline bool split_by_group(int32_t split_method, int64_t p_req) {
    return split_method == ATG_SPLIT_BISECT && p_req >= kGroupedSplits;
}
// Whether a build takes the one-launch kernel, which stands for the default
// methods: a pack or split that the caller chose runs as chosen (and reports
// its certificate and fallbacks).
inline bool one_launch_ok(const atg_build_opts& o, int64_t n, int64_t G, int64_t Ls, int64_t p_req) {
    return o.split_method == ATG_SPLIT_BISECT && o.pack_method == ATG_PACK_CHUNKED && small_build_ok(n, G, Ls, p_req);
}
// Sets the split method, knot count and split/pack interleave of a created
// table (knobs that leave the table's rows unchanged).
atg_status table_set_method(atg_table* t, int32_t split_method, int32_t learned_segments, int32_t interleave);

constexpr int64_t kMaxSectionLen = 2048;
constexpr int kInterleaveChunks = 8;  // split/pack interleave chunks
constexpr int64_t kMaxN = 0x7FFFFFF0LL;

template <typename T>
hipError_t dalloc(T** p, size_t count) {
    *p = nullptr;
    if (count == 0) count = 1;
    return hipMalloc((void**)p, count * sizeof(T));
}

}  // namespace atg

#define HIPCHK(call)                                                                         \
    do {                                                                                     \
        hipError_t e_ = (call);                                                              \
        if (e_ != hipSuccess)                                                                \
            return ::atg::fail(e_ == hipErrorOutOfMemory ? ATG_ENOMEM : ATG_EDEVICE, "%s: %s (%s:%d)", \
                               #call, hipGetErrorString(e_), __FILE__, __LINE__);            \
    } while (0)

// One-launch builds of small single tables (atg_small.h).
#include <algorithm>

#include "atg_small.h"

namespace atg {

// THREADS bounds the workgroup: 16 waves for sections of up to 1024 items, 4
// for longer ones, whose weights take more registers.
template <typename T, bool AOS, int XU, int THREADS, bool LISTS>
__global__ __launch_bounds__(THREADS) void build_small(BuildArgs a, double* W_out, uint32_t* error_out) {
    extern __shared__ double small_lds[];
    small_build<T, AOS, XU, LISTS, false>(a, W_out, error_out, small_lds);
}

template <typename T, bool AOS, bool LISTS>
static hipError_t launch_small_t(const BuildArgs& a, double* W_out, uint32_t* error_out, hipStream_t s) {
    const bool shorts = a.Ls <= kShortSectionMax;
    void (*k)(BuildArgs, double*, uint32_t*) =
        a.Ls <= 128 ? build_small<T, AOS, 2, 64 * kSmallMaxWaves, LISTS>
        : shorts    ? build_small<T, AOS, kShortSectionMax / 64, 64 * kSmallMaxWaves, LISTS>
                    : build_small<T, AOS, PSA_MAX_LEN / 64, 64 * kSmallLongWaves, LISTS>;
    const size_t lds = SmallLds(a.n, a.p_req).bytes();
    // The limit is state of the process: always the most that any table needs,
    // so that no call lowers it under another thread's launch or a captured one.
    if (lds > kSmallLdsDefault) {
        const hipError_t e = hipFuncSetAttribute((const void*)k, hipFuncAttributeMaxDynamicSharedMemorySize, (int)kSmallLdsMax);
        if (e != hipSuccess) return e;
    }
    // A wave per section and a thread per pack chain.
    const int64_t most = shorts ? kSmallMaxWaves : kSmallLongWaves;
    const int64_t waves = std::min(most, std::max(a.G, (a.p_req + 63) / 64));
    hipLaunchKernelGGL(k, dim3(1), dim3((unsigned)(64 * waves)), lds, s, a, W_out, error_out);
    return hipGetLastError();
}

template <typename T, bool AOS>
static hipError_t launch_small_l(const BuildArgs& a, bool lists, double* W_out, uint32_t* error_out, hipStream_t s) {
    return lists ? launch_small_t<T, AOS, true>(a, W_out, error_out, s) : launch_small_t<T, AOS, false>(a, W_out, error_out, s);
}

hipError_t launch_small(const BuildArgs& a, bool lists, double* W_out, uint32_t* error_out, hipStream_t s) {
    if (a.dtype_f32)
        return a.rows ? launch_small_l<float, true>(a, lists, W_out, error_out, s)
                      : launch_small_l<float, false>(a, lists, W_out, error_out, s);
    return a.rows ? launch_small_l<double, true>(a, lists, W_out, error_out, s)
                  : launch_small_l<double, false>(a, lists, W_out, error_out, s);
}

bool small_build_ok(int64_t n, int64_t G, int64_t Ls, int64_t p_req) {
    const int64_t waves = Ls <= kShortSectionMax ? kSmallMaxWaves : kSmallLongWaves;
    return G <= waves && n <= kSmallMaxItems && SmallLds(n, p_req).bytes() <= kSmallLdsMax;
}

}  // namespace atg

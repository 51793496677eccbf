// One format's instances of the direct kernel (each in a source file of its own: they compile in
// parallel) and the choice between them.
#pragma once
#include "direct_body.h"

namespace w4a16 {

template <int FMT, typename E, int R, int NWN, int KW, bool MOE>
static hipError_t launch_direct_t(const PrefillParams& p, hipStream_t st) {
    auto* k = &direct_kernel<FMT, E, R, NWN, KW, MOE>;
    constexpr size_t lds = direct_lds(R, NWN, KW);
    static_assert(lds <= 160 * 1024 - 64, "LDS");
    // set on every launch: once per process would miss other devices and race between threads
    (void)hipFuncSetAttribute(reinterpret_cast<const void*>(k), hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    (void)hipGetLastError();
    const int64_t blocks = (int64_t)8 * ((p.col_tiles + 7) / 8) * p.ksplit * p.row_tiles;
    if (blocks < 1 || blocks > INT32_MAX) return hipErrorInvalidValue;
    hipLaunchKernelGGL(k, dim3((unsigned)blocks), dim3(64 * NWN * KW), lds, st, p);
    return hipGetLastError();
}

template <int FMT, typename E>
static hipError_t launch_direct_dense(const PrefillParams& p, const DirectShape& s, hipStream_t st) {
    switch (100 * s.r + 10 * s.nwn + s.kw) {
        case 122: return launch_direct_t<FMT, E, 1, 2, 2, false>(p, st);
        case 222: return launch_direct_t<FMT, E, 2, 2, 2, false>(p, st);
        case 322: return launch_direct_t<FMT, E, 3, 2, 2, false>(p, st);
        case 422: return launch_direct_t<FMT, E, 4, 2, 2, false>(p, st);
        case 424: return launch_direct_t<FMT, E, 4, 2, 4, false>(p, st);
        case 722: return launch_direct_t<FMT, E, 7, 2, 2, false>(p, st);
        case 741: return launch_direct_t<FMT, E, 7, 4, 1, false>(p, st);
        default: return hipErrorInvalidValue;
    }
}

}  // namespace w4a16

// One format's instances of the direct kernel (each in a source file of its own: they compile in
// parallel) and the choice between them.
#pragma once
#include "direct_body.h"

namespace w4a16 {

static hipError_t launch_direct_any(void (*k)(PrefillParams), int threads, size_t lds, const PrefillParams& p, hipStream_t st) {
    // set on every launch: once per process would miss other devices and race between threads
    (void)hipFuncSetAttribute(reinterpret_cast<const void*>(k), hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    (void)hipGetLastError();
    const int64_t tiles = (int64_t)p.col_tiles * p.ksplit * p.row_tiles;
    if (tiles < 1 || tiles > INT32_MAX - 8) return hipErrorInvalidValue;
    hipLaunchKernelGGL(k, dim3((unsigned)((tiles + 7) / 8 * 8)), dim3(threads), lds, st, p);
    return hipGetLastError();
}

template <int FMT, typename E, int R, int NWN, int KW>
static hipError_t launch_direct_t(const PrefillParams& p, hipStream_t st) {
    constexpr size_t lds = direct_lds(R, NWN, KW);
    static_assert(lds <= 160 * 1024 - 64, "LDS");   // a flag stands beside it
    return launch_direct_any(&direct_kernel<FMT, E, R, NWN, KW>, 64 * NWN * KW, lds, p, st);
}

template <int FMT, typename E>
static hipError_t launch_direct_dense(const PrefillParams& p, const DirectShape& s, hipStream_t st) {
    switch (100 * s.r + 10 * s.nwn + s.kw) {
        case 122: return launch_direct_t<FMT, E, 1, 2, 2>(p, st);
        case 222: return launch_direct_t<FMT, E, 2, 2, 2>(p, st);
        case 322: return launch_direct_t<FMT, E, 3, 2, 2>(p, st);
        case 422: return launch_direct_t<FMT, E, 4, 2, 2>(p, st);
        case 424: return launch_direct_t<FMT, E, 4, 2, 4>(p, st);
        case 722: return launch_direct_t<FMT, E, 7, 2, 2>(p, st);
        case 741: return launch_direct_t<FMT, E, 7, 4, 1>(p, st);
        default: return hipErrorInvalidValue;
    }
}

// LDS of an expert-tile instance: its largest over the tile heights
template <int RMAX, int NWN, int KW>
constexpr size_t direct_moe_lds() {
    size_t m = 0;
    for (int r = 1; r <= RMAX; ++r)
        if (direct_lds(r, NWN, KW) > m) m = direct_lds(r, NWN, KW);
    return m;
}

template <int FMT, int RMAX, int NWN, int KW>
static hipError_t launch_direct_moe_t(const PrefillParams& p, hipStream_t st) {
    constexpr size_t lds = direct_moe_lds<RMAX, NWN, KW>();
    static_assert(lds <= 160 * 1024, "LDS");
    return launch_direct_any(&direct_moe_kernel<FMT, RMAX, NWN, KW>, 64 * NWN * KW, lds, p, st);
}

template <int FMT>
static hipError_t launch_direct_moe_f(const PrefillParams& p, const DirectShape& s, hipStream_t st) {
    switch (100 * s.r + 10 * s.nwn + s.kw) {
        case 424: return launch_direct_moe_t<FMT, 4, 2, 4>(p, st);
        case 741: return launch_direct_moe_t<FMT, 7, 4, 1>(p, st);
        case 742: return launch_direct_moe_t<FMT, 7, 4, 2>(p, st);
        default: return hipErrorInvalidValue;
    }
}

}  // namespace w4a16

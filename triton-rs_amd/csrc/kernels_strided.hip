// Launchers for the generic strided GEMM (strided_body.h) and the standalone dequant kernels.
#include <type_traits>

#include "strided_body.h"

namespace w4a16 {

template <int FMT, typename E>
__global__ void __launch_bounds__(256) strided_gemm_kernel(StridedParams p) {
    strided_gemm_body<FMT, E>(p);
}

// A gated launch is a fallback that usually exits at once (the act-order route runs it
// behind the tiled prefill, for a g_idx that route cannot take): launching one workgroup per
// tile would cost about 4 us of empty workgroups at M = 2048, N = 6144, so it gets at most
// STR_GATED_GRID workgroups that walk the tiles.
constexpr int STR_GATED_GRID = 512;

template <typename E>
static void launch_strided_e(int fmt, const StridedParams& p, hipStream_t st) {
    const int tm = (p.m + STR_BM - 1) / STR_BM, tn = (p.n + STR_BN - 1) / STR_BN;
    const dim3 grid = p.gate && (int64_t)tm * tn > STR_GATED_GRID ? dim3(STR_GATED_GRID) : dim3(tm, tn);
    const dim3 block(256);
    if (fmt == FMT_AWQ) hipLaunchKernelGGL((strided_gemm_kernel<FMT_AWQ, E>), grid, block, 0, st, p);
    else if (fmt == FMT_GPTQ) hipLaunchKernelGGL((strided_gemm_kernel<FMT_GPTQ, E>), grid, block, 0, st, p);
    else if (fmt == FMT_GPTQ_SYM) hipLaunchKernelGGL((strided_gemm_kernel<FMT_GPTQ_SYM, E>), grid, block, 0, st, p);
    else if constexpr (std::is_same<E, half_t>::value)   // prepared layout: fp16 only
        hipLaunchKernelGGL((strided_gemm_kernel<FMT_PREP, E>), grid, block, 0, st, p);
}

hipError_t launch_strided_gemm(int fmt, const StridedParams& p, hipStream_t st, bool bf16) {
    (void)hipGetLastError();  // launch errors below are ours, not an earlier call's
    if (bf16) launch_strided_e<bf16_t>(fmt, p, st);
    else launch_strided_e<half_t>(fmt, p, st);
    return hipGetLastError();
}

// ------------------------------------------------------------------ dequant

// What dequant_block_kernel does not take: group indexes, tensors off 16 bytes, groups that are no
// multiple of 8 rows. One thread per packed word. GPTQ word (kp, n) -> 8 consecutive k of column n;
// AWQ word (k, wn) -> 8 consecutive columns of row k. E: fp16 or bfloat16 scales and output.
template <int FMT, typename E>
__global__ void __launch_bounds__(256) dequant_kernel(DequantParams p) {
    typedef typename vec8<E>::type e8_t;
    const E* scales = reinterpret_cast<const E*>(p.scales);
    E* out = reinterpret_cast<E*>(p.out);
    const int64_t NW = (FMT == FMT_AWQ) ? (p.N >> 3) : p.N;
    const int64_t rows = (FMT == FMT_AWQ) ? p.K : (p.K >> 3);
    const int64_t idx = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (idx >= rows * NW) return;
    const int64_t r = idx / NW, c = idx - r * NW;
    const uint32_t word = p.qweight[idx];
    E v[8];
    if constexpr (FMT == FMT_AWQ) {
        const int k = (int)r;
        const int g = p.g_idx ? min(max(p.g_idx[k], 0), p.K / p.G - 1) : k / p.G;
        const uint32_t qz = p.qzeros[(int64_t)g * NW + c];
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            const int n = (int)(8 * c + j);
            v[j] = dequant1(nib(word, awq_slot(n)), zero_of<FMT>(qz, n, 0),
                            scales[(int64_t)g * p.N + n]);
        }
        if (!p.transposed) {
            *reinterpret_cast<e8_t*>(out + (int64_t)k * p.N + 8 * c) =
                e8_t{v[0], v[1], v[2], v[3], v[4], v[5], v[6], v[7]};
        } else {
#pragma unroll
            for (int j = 0; j < 8; ++j) out[(8 * c + j) * p.K + k] = v[j];
        }
    } else {
        const int n = (int)c;
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            const int k = (int)(8 * r + j);
            const int g = p.g_idx ? min(max(p.g_idx[k], 0), p.K / p.G - 1) : k / p.G;
            uint32_t qz = 0;
            if constexpr (FMT == FMT_GPTQ) qz = p.qzeros[(int64_t)g * (p.N >> 3) + (n >> 3)];
            v[j] = dequant1(nib(word, j), zero_of<FMT>(qz, n, p.zero_offset),
                            scales[(int64_t)g * p.N + n]);
        }
        if (p.transposed) {
            *reinterpret_cast<e8_t*>(out + (int64_t)n * p.K + 8 * r) =
                e8_t{v[0], v[1], v[2], v[3], v[4], v[5], v[6], v[7]};
        } else {
#pragma unroll
            for (int j = 0; j < 8; ++j) out[(8 * r + j) * p.N + n] = v[j];
        }
    }
}

// Plain group order, groups of a multiple of 8 rows and 16-byte aligned tensors: one thread per
// 8 x 8 block of weights, which has one group, so that scales and zeros are loaded once, and whose
// lines are 16-byte stores whichever way the words run. Bound by HBM. The lanes of a wave are
// NL x KL blocks along N and K: 8 x 8 for [N, K] (a store instruction writes 8 lines of 128 bytes;
// one thread per word wrote 16 bytes of 64 lines), 64 x 1 for [K, N]. The four waves lie along K for
// GPTQ and [N, K] (512 bytes of a line), else along N (for AWQ 128 bytes of a row of words).
// 4096 x 14336, one thread per word, now: GPTQ [N, K] 83.0, 35.0 us (4.2 TB/s), [K, N] 67.8, 30.5 us;
// AWQ [N, K] 747, 37.3 us, [K, N] 39.8, 30.3 us (4.9 TB/s).
template <int FMT, typename E, bool T>
__global__ void __launch_bounds__(256) dequant_block_kernel(DequantParams p) {
    typedef typename vec8<E>::type e8_t;
    constexpr bool AWQ = FMT == FMT_AWQ;
    constexpr int NL = T ? 8 : 64, KL = 64 / NL;
    constexpr int WK = T && !AWQ ? 4 : 1, WN = 4 / WK;
    const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
    const int NB = p.N >> 3, KB = p.K >> 3;
    const int tk = (KB + KL * WK - 1) / (KL * WK), tn = (NB + NL * WN - 1) / (NL * WN);
    // blocks of the output's contiguous direction in turn
    const int b = blockIdx.x, bk = T ? b % tk : b / tn, bn = T ? b / tk : b % tn;
    const int kb = (bk * WK + (WK > 1 ? wave : 0)) * KL + (T ? lane & 7 : 0);
    const int nb = (bn * WN + (WN > 1 ? wave : 0)) * NL + (T ? lane >> 3 : lane);
    if (kb >= KB || nb >= NB) return;
    uint32_t w[8];
    if constexpr (AWQ) {
#pragma unroll
        for (int i = 0; i < 8; ++i) w[i] = p.qweight[(size_t)(8 * kb + i) * NB + nb];
    } else {
        const u32x4* q = reinterpret_cast<const u32x4*>(p.qweight + (size_t)kb * p.N + 8 * nb);
        const u32x4 a = q[0], c = q[1];
        w[0] = a.x; w[1] = a.y; w[2] = a.z; w[3] = a.w;
        w[4] = c.x; w[5] = c.y; w[6] = c.z; w[7] = c.w;
    }
    const int g = 8 * kb / p.G;
    const e8_t sc = *reinterpret_cast<const e8_t*>(reinterpret_cast<const E*>(p.scales) + (size_t)g * p.N + 8 * nb);
    uint32_t qz = 0;
    if constexpr (FMT != FMT_GPTQ_SYM) qz = p.qzeros[(size_t)g * NB + nb];
    int z[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) z[i] = zero_of<FMT>(qz, i, p.zero_offset);
    E* out = reinterpret_cast<E*>(p.out);
    if constexpr (T) {
#pragma unroll
        for (int n = 0; n < 8; ++n) {
            e8_t v;
#pragma unroll
            for (int k = 0; k < 8; ++k)
                v[k] = dequant1(AWQ ? nib(w[k], awq_slot(n)) : nib(w[n], k), z[n], (E)sc[n]);
            *reinterpret_cast<e8_t*>(out + (size_t)(8 * nb + n) * p.K + 8 * kb) = v;
        }
    } else {
#pragma unroll
        for (int k = 0; k < 8; ++k) {
            e8_t v;
#pragma unroll
            for (int n = 0; n < 8; ++n)
                v[n] = dequant1(AWQ ? nib(w[k], awq_slot(n)) : nib(w[n], k), z[n], (E)sc[n]);
            *reinterpret_cast<e8_t*>(out + (size_t)(8 * kb + k) * p.N + 8 * nb) = v;
        }
    }
}

template <int FMT, typename E>
static void launch_dequant_block(const DequantParams& p, hipStream_t st) {
    const int NB = p.N >> 3, KB = p.K >> 3;
    // blocks per workgroup along K and N, as in the kernel
    const int ck = !p.transposed ? 1 : FMT == FMT_AWQ ? 8 : 32, cn = !p.transposed ? 256 : FMT == FMT_AWQ ? 32 : 8;
    const dim3 grid((unsigned)((KB + ck - 1) / ck) * (unsigned)((NB + cn - 1) / cn)), block(256);
    if (p.transposed) hipLaunchKernelGGL((dequant_block_kernel<FMT, E, true>), grid, block, 0, st, p);
    else hipLaunchKernelGGL((dequant_block_kernel<FMT, E, false>), grid, block, 0, st, p);
}

template <typename E>
static void launch_dequant_e(int fmt, const DequantParams& p, hipStream_t st) {
    const uintptr_t bits = reinterpret_cast<uintptr_t>(p.qweight) | reinterpret_cast<uintptr_t>(p.scales) |
                           reinterpret_cast<uintptr_t>(p.out);
    if (!p.g_idx && p.K % 8 == 0 && p.N % 8 == 0 && p.G % 8 == 0 && bits % 16 == 0) {
        if (fmt == FMT_AWQ) launch_dequant_block<FMT_AWQ, E>(p, st);
        else if (fmt == FMT_GPTQ) launch_dequant_block<FMT_GPTQ, E>(p, st);
        else launch_dequant_block<FMT_GPTQ_SYM, E>(p, st);
        return;
    }
    const int64_t words = (int64_t)p.K * p.N / 8;
    const dim3 grid((unsigned)((words + 255) / 256)), block(256);
    if (fmt == FMT_AWQ) hipLaunchKernelGGL((dequant_kernel<FMT_AWQ, E>), grid, block, 0, st, p);
    else if (fmt == FMT_GPTQ) hipLaunchKernelGGL((dequant_kernel<FMT_GPTQ, E>), grid, block, 0, st, p);
    else hipLaunchKernelGGL((dequant_kernel<FMT_GPTQ_SYM, E>), grid, block, 0, st, p);
}

hipError_t launch_dequant(int fmt, const DequantParams& p, hipStream_t st, bool bf16) {
    (void)hipGetLastError();  // launch errors below are ours, not an earlier call's
    if (bf16) launch_dequant_e<bf16_t>(fmt, p, st);
    else launch_dequant_e<half_t>(fmt, p, st);
    return hipGetLastError();
}

}  // namespace w4a16

// Direct kernel (direct_body.h), host side: which of its instances a shape takes, and whether it
// takes the place of the other kernels.
#include "device_common.h"
#include "launch.h"

#include <cmath>

namespace w4a16 {

hipError_t launch_direct_gptq(const PrefillParams& p, const DirectShape& s, hipStream_t st);
hipError_t launch_direct_gptq_bf16(const PrefillParams& p, const DirectShape& s, hipStream_t st);
hipError_t launch_direct_awq(const PrefillParams& p, const DirectShape& s, hipStream_t st);
hipError_t launch_direct_awq_bf16(const PrefillParams& p, const DirectShape& s, hipStream_t st);
hipError_t launch_direct_prep(const PrefillParams& p, const DirectShape& s, hipStream_t st);
hipError_t launch_direct_moe_gptq(const PrefillParams& p, const DirectShape& s, hipStream_t st);
hipError_t launch_direct_moe_awq(const PrefillParams& p, const DirectShape& s, hipStream_t st);
hipError_t launch_direct_moe_prep(const PrefillParams& p, const DirectShape& s, hipStream_t st);

// Formats, groups and sizes the kernel reads: 32-bit byte offsets below 2^31 (offsets from 2^31 up
// mark what reads as zero), a stage of 64 rows in whole groups or in two groups of 32
static bool direct_ok(int fmt, int N, int K, int G, long long a_rows) {
    const long long lim = 1ll << 31;
    if (N < 8 || K < 64 || G < 1 || K % G || K % 64 || !(G == 32 || G % 64 == 0)) return false;
    if (fmt == FMT_PREP ? (N % 16 || K % 128 || !prep_group_ok(G) || (long long)prep_total_bytes(K, N, G) >= lim)
                        : N % (fmt == FMT_AWQ ? 32 : 8) != 0)
        return false;
    return (long long)K * N / 2 < lim && a_rows * K * 2 < lim && (long long)(K / G) * N * 2 < lim;
}

// Time model, fitted to graph-replay times over M = 16 .. 1024 (GPTQ, K, N = 1792 .. 28672; within
// 10 % of nearly all of 200 measured points): a stage of a wave takes us[R] with one wave per SIMD;
// an eight-wave workgroup 1.75 of a four-wave one, and a second one on the same CU 0.65 more (two
// fit with up to 80 KiB of LDS); 5 us of launch, first loads and store, 1 us for the sum over the
// K groups; split K: the partials written and read at 4.4 TB/s and 2 us for the hand-over.
struct DirectCfg { int r, nwn, kw, lds_kb; double us; };
static const DirectCfg CFGS[] = {
    {1, 2, 2, 56, 0.42}, {2, 2, 2, 72, 0.51}, {3, 2, 2, 88, 0.59}, {4, 2, 2, 104, 0.63},
    {4, 2, 4, 156, 0.63}, {7, 2, 2, 114, 0.89}, {7, 4, 1, 72, 0.87},
};

DirectShape direct_shape(int fmt, int M, int N, int K, int G, int num_cus, bool bf16,
                         size_t max_partial_bytes, size_t max_tiles) {
    DirectShape best{};
    if (M < 1 || !direct_ok(fmt, N, K, G, M) || (bf16 && fmt == FMT_PREP)) return best;
    for (const DirectCfg& c : CFGS) {
        // up to 48 rows the tile that holds them; beyond, tiles of 64 or 112 rows
        if (M <= 48 ? c.r != (M + 15) / 16 : c.r < 4) continue;
        const int bn = 64 * c.nwn, ct = (N + bn - 1) / bn, rt = (M + 16 * c.r - 1) / (16 * c.r);
        const double us = c.us * (bf16 ? 1.1 : 1.0) + (fmt == FMT_AWQ ? 0.06 : 0.0);
        for (int ks = 1; ks <= 8; ks *= 2) {
            // at most 8 ways, and at least four stages per wave and split
            const int ns = (K / 64 + ks * c.kw - 1) / (ks * c.kw);
            if (ks > 1 && ns < 4) break;
            const size_t tile = (size_t)bn * 16 * c.r * 4;
            const size_t part = ks > 1 ? (size_t)ks * ct * rt * tile : 0;
            if (ks > 1 && (part > max_partial_bytes || part > ((size_t)128 << 20) || (size_t)ct * rt > max_tiles)) break;
            const long long wgs = (long long)ct * rt * ks, n = (wgs + num_cus - 1) / num_cus;
            const double load = c.lds_kb > 80 ? (double)n : n % 2 ? 0.825 * (double)(n - 1) + 1.0 : 0.825 * (double)n;
            const double run = load * ns * us * (c.nwn * c.kw > 4 ? 1.75 : 1.0);
            const double hbm = ((double)K * N / 2 + (double)M * (K + N) * 2) / 4.5e6;
            const double t = 5.0 + (run > hbm ? run : hbm) + (c.kw > 1 ? 1.0 : 0.0) +
                             (ks > 1 ? 2.0 + 2.0 * (double)part / 4.4e6 : 0.0);
            if (!best.ok || t < best.us) {
                best.ok = true;
                best.r = c.r; best.nwn = c.nwn; best.kw = c.kw; best.ksplit = ks;
                best.col_tiles = ct; best.row_tiles = rt;
                best.partial_bytes = part;
                best.us = t;
            }
        }
    }
    return best;
}

hipError_t launch_direct(int fmt, PrefillParams p, const DirectShape& s, hipStream_t st, bool bf16) {
    if (!s.ok || (s.ksplit > 1 && (!p.ws || !p.counters))) return hipErrorInvalidValue;
    p.col_tiles = s.col_tiles;
    p.row_tiles = s.row_tiles;
    p.ksplit = s.ksplit;
    if (fmt == FMT_GPTQ_SYM) {   // no zeros: an empty buffer reads zero, the offset is the zero point
        p.qzeros = nullptr;
        p.zero_offset = 8;
        fmt = FMT_GPTQ;
    }
    if (fmt == FMT_GPTQ) return bf16 ? launch_direct_gptq_bf16(p, s, st) : launch_direct_gptq(p, s, st);
    if (fmt == FMT_AWQ) return bf16 ? launch_direct_awq_bf16(p, s, st) : launch_direct_awq(p, s, st);
    if (fmt == FMT_PREP && !bf16) return launch_direct_prep(p, s, st);
    return hipErrorInvalidValue;
}

// By expert: 256 columns per workgroup; where K may be summed in parts and the tiles would not give
// every CU two workgroups, K over two groups of waves, for tiles of up to 64 rows over four, 128
// columns wide (16 tokens, 8 experts, K = 14336 -> N = 4096: 61 us, half of it HBM's; 512 tokens:
// 197 us against 226 us in one group)
DirectShape direct_moe_shape(int fmt, int N, int K, int G, long long a_rows, int tile_bm, int est_tiles,
                             int est_rows, int num_cus, bool split) {
    DirectShape s{};
    if (!direct_ok(fmt, N, K, G, a_rows) || (fmt != FMT_PREP && G % 64)) return s;
    s.ok = true;
    s.ksplit = 1;
    const int ct = (N + 255) / 256;
    const bool few = split && (long long)est_tiles * ct < 2 * num_cus;
    s.r = few && tile_bm <= 64 ? 4 : 7;
    s.nwn = few && tile_bm <= 64 ? 2 : 4;
    s.kw = !few ? 1 : tile_bm <= 64 ? 4 : 2;
    s.col_tiles = (N + 64 * s.nwn - 1) / (64 * s.nwn);
    // the dense time model's stage times (R = 5, 6 in between) for tiles of est_rows rows
    static const double US[] = {0.42, 0.51, 0.59, 0.63, 0.72, 0.80, 0.88};
    const double wgs = (double)est_tiles * s.col_tiles / num_cus;
    const double load = s.kw > 1 ? std::ceil(wgs) : wgs <= 1 ? 1.0 : 0.825 * std::ceil(wgs);
    s.us = load * ((K / 64 + s.kw - 1) / s.kw) * US[(est_rows + 15) / 16 - 1] * (s.kw > 1 ? 1.75 : 1.0);
    return s;
}

hipError_t launch_direct_moe(int fmt, PrefillParams p, const DirectShape& s, int tile_bm, int max_tiles, hipStream_t st) {
    if (!s.ok || !p.tiles || !p.num_tiles || tile_bm > 16 * s.r || max_tiles < 1 || p.gate) return hipErrorInvalidValue;
    p.col_tiles = s.col_tiles;
    p.row_tiles = max_tiles;
    p.ksplit = 1;
    if (fmt == FMT_GPTQ_SYM) {   // as launch_direct
        p.qzeros = nullptr;
        p.zero_offset = 8;
        fmt = FMT_GPTQ;
    }
    return fmt == FMT_GPTQ ? launch_direct_moe_gptq(p, s, st)
           : fmt == FMT_AWQ ? launch_direct_moe_awq(p, s, st)
           : fmt == FMT_PREP ? launch_direct_moe_prep(p, s, st) : hipErrorInvalidValue;
}

}  // namespace w4a16

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

// Time model. A workgroup runs ns stages of us each after 5 to 6 us of launch, first loads, store and
// the sum over the K groups; every further round of workgroups pays about that again. Instances of
// more than 80 KiB of LDS run one workgroup on a CU, the others two, which together take 1.65 to 1.82
// of one's time. Beside it the tiles' operands come through the L2s (a tile's x and words at 10.7 TB/s in all;
// the two add as their fourth powers). No call is faster than its operands from HBM. A split of K:
// hand-over, the partials written and read, and the last workgroup's sum.
// Fitted to graph-replay times of all 64- and 112-row instances (K, N = 1024 .. 28672, 30 shapes, M =
// 65 .. 8192, every format, fp16 and bf16; 15000 points): nine of ten within 7 %, and the instance it
// puts lowest within 3 % of the best in 98 of 100 calls; up to 48 rows, where it only chooses the split
// of K, in 93 of 100. Without the fixed cost of further rounds 1792 -> 4096 at 2048 rows took four
// rounds of 64-row tiles (60.7 us), modelled at 37.
struct DirectCfg {
    int r, nwn, kw;
    double pair;    // two workgroups per CU: their stage against one's (0: one per CU)
    double us;      // a stage, GPTQ in fp16 (a workgroup's eight waves together)
    double first, more;   // fixed cost of a call, of a further round
    double split, sum;    // split K: hand-over, and the last sum per MB of a tile's partials
};
static const DirectCfg CFGS[] = {
    {1, 2, 2, 1.65, 0.42, 5.0, 0.0, 2.0, 0.0}, {2, 2, 2, 1.65, 0.51, 5.0, 0.0, 2.0, 0.0},
    {3, 2, 2, 0, 0.59, 5.0, 0.0, 2.0, 0.0},    {4, 2, 2, 0, 0.605, 5.2, 4.1, 0.8, 8.3},
    {4, 2, 4, 0, 0.985, 6.2, 6.0, 0.8, 10.4},  {7, 2, 2, 0, 0.803, 6.0, 6.7, 0.7, 8.5},
    {7, 4, 1, 1.82, 0.708, 5.2, 5.3, 1.9, 7.6},
};

// What the other formats and bf16 add to a stage of a wave
static double stage_extra(int fmt, bool bf16, bool low) {
    if (bf16) return fmt == FMT_AWQ ? (low ? 0.12 : 0.16) : low ? 0.1 : 0.12;
    return fmt == FMT_AWQ && low ? 0.05 : fmt == FMT_AWQ || fmt == FMT_PREP ? 0.03 : 0.0;
}

DirectShape direct_shape(int fmt, int M, int N, int K, int G, int num_cus, bool bf16,
                         size_t max_partial_bytes, size_t max_tiles) {
    DirectShape best{};
    if (M < 1 || !direct_ok(fmt, N, K, G, M) || (bf16 && fmt == FMT_PREP)) return best;
    for (const DirectCfg& c : CFGS) {
        // up to 48 rows the tile that holds them; beyond, tiles of 64 or 112 rows
        if (M <= 48 ? c.r != (M + 15) / 16 : c.r < 4) continue;
        const int bn = 64 * c.nwn, ct = (N + bn - 1) / bn, rt = (M + 16 * c.r - 1) / (16 * c.r);
        double us = c.us + stage_extra(fmt, bf16, c.r < 4) * (c.nwn * c.kw > 4 ? 2.2 : 1.0);
        // AWQ rows come in 64-byte pieces here, from HBM for the first row tiles; the three ring slots
        // of this instance do not cover it (4096 -> 14336, 128 rows 30.7 us, GPTQ 26.3)
        if (fmt == FMT_AWQ && c.kw == 4 && rt <= 2) us += 0.3;
        for (int ks = 1; ks <= 8; ks *= 2) {
            // at most 8 ways, and at least four stages per wave and split
            const int ns = (K / 64 + ks * c.kw - 1) / (ks * c.kw);
            if (ks > 1 && ns < 4) break;
            const size_t tile = (size_t)bn * 16 * c.r * 4;
            const size_t part = ks > 1 ? (size_t)ks * ct * rt * tile : 0;
            if (ks > 1 && (part > max_partial_bytes || part > ((size_t)128 << 20) || (size_t)ct * rt > max_tiles)) break;
            const long long wgs = (long long)ct * rt * ks, n = (wgs + num_cus - 1) / num_cus;
            const long long rounds = c.pair > 0 ? (n + 1) / 2 : n;
            const double load = c.pair > 0 ? c.pair * (double)(n / 2) + (double)(n % 2) : (double)n;
            const double run = load * ns * us + c.more * (double)(rounds - 1);
            const double hbm = ((double)K * N / 2 + (double)M * (K + N) * 2) / 4.5e6;
            const double l2 = ((double)ct * M * K * 2 + (double)rt * K * N / 2) / 10.7e6;
            const double both = std::sqrt(std::sqrt(run * run * run * run + l2 * l2 * l2 * l2));
            const double t = c.first + (both > hbm ? both : hbm) +
                             (ks > 1 ? c.split + 2.0 * (double)part / 4.4e6 + c.sum * 1e-6 * (double)(ks * tile) : 0.0);
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
    // a stage of a tile of est_rows rows (1 to 7 blocks of 16), one wave per SIMD: the expert kernel's own
    // times, compared here only between its instances (the dense instances' are fitted apart above)
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

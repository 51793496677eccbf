// W4A16 GEMM with the weights dequantised in registers ("direct"): from a few rows to some thousands
// (beyond 64 where a time model puts it ahead of the prefill kernel), dense or grouped by expert. Any checkpoint format, fp16 or bf16, and the prepared
// layout (fp16); any N that is a multiple of 8 (AWQ 32, prepared 16), K of 64 (prepared 128),
// groups of 32 rows or a multiple of 64.
//
// What it is for. The prefill kernel dequantises into LDS and shares that B tile between its
// waves, which pays where 256-row tiles fill the chip. Where they do not, mostly below a thousand rows, it
// splits K over workgroups, and the fp32 partials (written and read back at about 4.4 TB/s) and
// the last workgroup's sum cost more than the product. Here every wave owns 64 columns and makes
// its own B operands (v_mfma_f32_16x16x32, 8 rows of one column per lane) from packed words, so
// nothing but x and the packed words passes through LDS, a tile can be 16 to 112 rows high, and
// K is split over the waves of a workgroup first (their sums meet in LDS), over workgroups last.
//
// A workgroup: NWN waves along N (64 columns each) x KW groups along K, a tile of 16 R rows. One
// stage is 64 k. x and the words, scales and zeros of a stage come by LDS-DMA into a ring of D
// slots per K group; at the top of a stage the next one has landed, so that a step's operands are
// read from LDS, and its words dequantised, during the step before it.
//
// What bounds it: instruction issue. A stage of a wave is about 151 VALU (16 per packed word: two
// v_perm and two shifts put a byte into both halves of a register, v_and_or makes (1024 + q,
// 1024 + 16 q'), v_pk_fma gives (q - z, q' - z) exactly, v_pk_mul rounds (q - z) s once), 8 R
// MFMAs and 50 others; measured 0.42 to 0.88 us (R = 1 to 7) against 0.33 to 0.62 us of issue.
// Counters (K = 4096, N = 28672, one wave per SIMD): of a wave's time 59 % issuing and 20 % waiting
// for its turn at 48 rows of AWQ, 64 and 18 % at 200 of GPTQ, 73 and 15 % in bf16 (254 VALU a stage).
// Measured (K = 4096, GPTQ, weight sets in turn; before: the prefill kernel, from 48 rows down the
// small-batch kernels): N = 6144: M = 128 / 200 / 512 / 1024 / 2048 30.8 / 37.0 / 47.7 / 72.5 / 107.3 ->
// 19.0 / 22.3 / 34.4 / 58.1 / 101.4 us; N = 28672: M = 16 / 48 / 200 24.6 / 46.7 / 69.4 -> 18.6 / 24.8 /
// 55.9 us; AWQ M = 48: N = 4096 / 6144 / 28672 25.0 / 25.5 / 42.4 -> 12.5 / 14.0 / 27.8 us.
#pragma once
#include <type_traits>

#include "device_common.h"
#include "launch.h"
#include "lds_dma.h"
#include "splitk.h"

namespace w4a16 {

constexpr int DIR_K = 64;                     // k rows per stage
constexpr int DIR_CPL = 4;                    // columns per lane
constexpr int direct_bn(int nwn) { return 16 * DIR_CPL * nwn; }
// Ring in LDS, per K group: D slots (stages), each x (16 R rows x 128 bytes) and, per wave, the
// packed words (2 KiB) and the scales and zeros of their columns (512 bytes)
constexpr int DIR_WST = 2048 + 512;
// (four where two workgroups, or two K groups, then still fit: five row blocks and three slots left
// an expert's K = 14336 -> N = 4096 at 205 us for 512 tokens, four slots 197)
constexpr int direct_depth(int r, int kw) { return r <= 2 || (r <= 5 && kw <= 2) ? 4 : 3; }
constexpr size_t direct_ring(int r, int nwn, int kw) {
    return (size_t)direct_depth(r, kw) * ((size_t)r * 16 * DIR_K * 2 + (size_t)nwn * DIR_WST);
}
// LDS: the K groups' rings, later half of their sums
constexpr size_t direct_lds(int r, int nwn, int kw) {
    const size_t x = kw * direct_ring(r, nwn, kw);
    const size_t s = kw > 1 ? (size_t)(kw / 2) * nwn * r * DIR_CPL * 1024 : 0;
    return x > s ? x : s;
}

// B bytes per lane from rsrc + voff + soff into LDS at dst + B * lane (dst, soff uniform)
template <int B>
__device__ __forceinline__ void dma_lds(bufrsrc_t r, unsigned char* dst, uint32_t voff, uint32_t soff) {
    if constexpr (B == 16) __builtin_amdgcn_raw_ptr_buffer_load_lds(r, (__attribute__((address_space(3))) void*)dst, 16, (int)voff, (int)soff, 0, 0);
    else __builtin_amdgcn_raw_ptr_buffer_load_lds(r, (__attribute__((address_space(3))) void*)dst, 4, (int)voff, (int)soff, 0, 0);
}

// Workgroup b's column tile, row tile and K split. Workgroups go to the XCDs in turn (b mod 8); each
// XCD takes an eighth of all (column tile, K split, row tile) in that order, row tiles fastest, so
// that a column tile's weights are fetched into one L2 once, and the XCDs get equal shares whatever
// the number of column tiles
__device__ __forceinline__ bool direct_place(const PrefillParams& p, int rts, int& ct, int& rt, int& bz) {
    const int total = rts * p.ksplit * p.col_tiles, share = (total + 7) >> 3;
    const int i = blockIdx.x >> 3, idx = (blockIdx.x & 7) * share + i;
    if (i >= share || idx >= total) return false;
    const int u = idx / rts;
    rt = idx - u * rts;
    ct = u / p.ksplit;
    bz = u - ct * p.ksplit;
    return true;
}

// One tile: rows [m0, m0 + rows) (MOE: of the sorted pairs), 16 R at most
template <int FMT, typename E, int R, int NWN, int KW, bool MOE>
__device__ __forceinline__ void direct_tile(const PrefillParams& p, unsigned char* lds, int ct, int rt, int bz,
                                            int m0, int rows) {
    constexpr bool BF = std::is_same<E, bf16_t>::value;
    typedef typename vec8<E>::type v8_t;
    constexpr bool PREP = FMT == FMT_PREP, AWQ = FMT == FMT_AWQ;
    static_assert(!AWQ || NWN == 4 || NWN == 2, "AWQ: the waves load their rows together");
    constexpr int CPL = DIR_CPL, WC = 16 * CPL, BN = NWN * WC, BM = 16 * R;
    constexpr int W = NWN * KW, D = direct_depth(R, KW);
    constexpr int A_ST = BM * DIR_K * 2;            // bytes of x per stage
    constexpr int DL = (2 * R + NWN - 1) / NWN;     // x loads per wave and stage (8 rows each)
    constexpr int RL = 4;                           // word loads (2), scales, zeros

    const int t = threadIdx.x, lane = t & 63;
    const int wave = __builtin_amdgcn_readfirstlane(t >> 6);
    const int wn = wave % NWN, kw = wave / NWN;
    const int j = lane & 15, h = lane >> 4;
    const int ksp = MOE ? 1 : p.ksplit;

    const int n0 = ct * BN, nw0 = n0 + wn * WC;    // first column of the workgroup, the wave
    const int NW = p.N >> 3, KB = p.K / DIR_K;
    // K stages of this wave's share: [s0, s0 + ns); a stage from kend on reads zeros: its loads go
    // through descriptors of no bytes (bytes(kb, n): n, or 0 past kend)
    const int ns = (KB + ksp * KW - 1) / (ksp * KW);
    const int s0 = (bz * KW + kw) * ns, kend = min(s0 + ns, KB);
    auto bytes = [&](int kb, uint32_t n) __attribute__((always_inline)) { return kb < kend ? n : 0u; };
    unsigned char* Ab = lds + (size_t)kw * direct_ring(R, NWN, KW);
    unsigned char* Wb = Ab + D * A_ST;
    // ---- x: row r of the tile, 8 chunks of 8 k per stage; chunk c at position c ^ (r & 7). A
    // load covers 8 rows of 128 bytes. Dense: rows past M lie past the buffer's end and read
    // zero. Experts: rows through sorted_ids, one offset per load
    // Offsets per lane are fixed; the stage's k offset is the loads' scalar offset (which the
    // range check leaves out: lanes out of range are so by their own offset)
    const int a_rows = MOE ? (p.num_pairs + p.a_div - 1) / p.a_div : p.M;
    const uint32_t xbytes = (uint32_t)a_rows * (uint32_t)p.K * 2u;
    const uint32_t achunk = 8u * (uint32_t)((lane & 7) ^ (lane >> 3));
    uint32_t aoff[DL];
#pragma unroll
    for (int q = 0; q < DL; ++q) {
        const int row = (wn * DL + q) % (2 * R) * 8 + (lane >> 3);
        int m = -1;
        if (row < rows) {
            m = m0 + row;
            if constexpr (MOE) {
                const int pair = p.sorted_ids[m];
                m = (unsigned)pair < (unsigned)p.num_pairs ? pair / p.a_div : -1;
            }
        }
        aoff[q] = m >= 0 ? ((uint32_t)m * (uint32_t)p.K + achunk) * 2u : DMA_OOB;
    }
    auto load_a = [&](int s, const int slot) __attribute__((always_inline)) {
        const int kb = s0 + s;
        const bufrsrc_t xr = make_rsrc(p.x, bytes(kb, xbytes));
#pragma unroll
        for (int q = 0; q < DL; ++q)
            dma_lds<16>(xr, Ab + slot * A_ST + (wn * DL + q) % (2 * R) * 1024, aoff[q], (uint32_t)kb * (DIR_K * 2u));
    };

    // ---- words, scales and zeros of a stage into the wave's 2.5 KiB of a ring slot
    //  GPTQ: 8 packed rows of the wave's 64 columns, 256 bytes each
    //  AWQ: the workgroup's 64 rows, loaded by its waves together. 128 bytes each (4 waves):
    //  16-byte chunk c of a row at position c ^ 2 key, key the lane group that reads the row; 64
    //  bytes each (2 waves): the rows that the four lane groups read together one after another
    //  (either way the four lane groups of a read fall in different banks)
    //  prepared: half a block (512 bytes) of each of the wave's 4 strips
    const uint32_t sb = PREP ? (uint32_t)prep_strip_bytes(p.K, p.G) : 0u;
    const uint32_t tb = PREP ? prep_table_words(p.K, p.G) * 4u : 0u;
    const uint32_t wbytes = PREP ? (uint32_t)(p.N / 16) * sb : (uint32_t)((size_t)p.K * p.N / 2);
    const uint32_t sbytes = PREP ? wbytes : (uint32_t)((size_t)(p.K / p.G) * p.N * 2);
    const uint32_t zbytes = PREP ? wbytes : p.qzeros ? (uint32_t)((size_t)(p.K / p.G) * NW * 4) : 0u;
    const void* sp = PREP ? (const void*)p.qweight : (const void*)p.scales;
    const void* zp = PREP ? (const void*)p.qweight : (const void*)p.qzeros;
    // order of a stage's k over (step st, lane group h): 32 st + 8 h for groups of whole stages;
    // 16 h + 8 st for groups of 32 rows (a lane's rows then lie in one group) and prepared words
    const bool nat = !PREP && p.G % DIR_K == 0;
    uint32_t wbase[2], sbase, zbase;
    if constexpr (PREP) {
#pragma unroll
        for (int q = 0; q < 2; ++q) {
            const int strip = nw0 / 16 + 2 * q + (lane >> 5);
            wbase[q] = 16 * strip < p.N ? (uint32_t)strip * sb + tb + (uint32_t)(lane & 31) * 16u : DMA_OOB;
        }
        const int strip = nw0 / 16 + (lane >> 4);
        sbase = zbase = 16 * strip < p.N ? (uint32_t)strip * sb + (uint32_t)(lane & 15) * 4u : DMA_OOB;
    } else {
#pragma unroll
        for (int q = 0; q < 2; ++q) {
            if constexpr (AWQ) {   // N % 32 == 0: a 16-byte chunk lies inside its row
                int row, c;
                if constexpr (NWN == 4) {
                    row = (2 * wn + q) * 8 + (lane >> 3);
                    const int key = (nat ? row >> 3 : row >> 4) & 3;
                    c = (n0 >> 3) + 4 * ((lane & 7) ^ (2 * key));
                } else {
                    const int rho = (2 * wn + q) * 16 + (lane >> 2), st = rho >> 5, r = (rho & 31) >> 2, hh = rho & 3;
                    row = nat ? 32 * st + 8 * hh + r : 16 * hh + 8 * st + r;
                    c = (n0 >> 3) + 4 * (lane & 3);
                }
                wbase[q] = c < NW ? ((uint32_t)row * (uint32_t)NW + (uint32_t)c) * 4u : DMA_OOB;
            } else {
                const int n = nw0 + 4 * (lane & 15);
                wbase[q] = n < p.N ? ((uint32_t)(4 * q + (lane >> 4)) * (uint32_t)p.N + (uint32_t)n) * 4u : DMA_OOB;
            }
        }
        // groups of 32 rows: the stage's second group in lanes 32..63
        const uint32_t g2 = p.G < DIR_K ? (uint32_t)lane >> 5 : 0u;
        const int n = nw0 + 2 * (lane & 31), z = (nw0 >> 3) + (lane & 31);
        sbase = n < p.N ? (g2 * (uint32_t)p.N + (uint32_t)n) * 2u : DMA_OOB;
        zbase = z < NW && (lane & 31) < 8 ? (g2 * (uint32_t)NW + (uint32_t)z) * 4u : DMA_OOB;
    }
    // the group of the next stage whose scales are loaded (stages come in order)
    const int gd = p.G < DIR_K ? 1 : p.G / DIR_K;              // stages per group
    const uint32_t gm = p.G < DIR_K ? DIR_K / p.G : 1;         // groups per stage
    uint32_t gi = (uint32_t)(s0 / gd) * gm;
    int gc = s0 % gd;
    auto load_w = [&](int s, const int slot) __attribute__((always_inline)) {
        const int kb = s0 + s;
        unsigned char* dst = Wb + slot * (NWN * DIR_WST) + wn * 2048;
        unsigned char* meta = Wb + slot * (NWN * DIR_WST) + NWN * 2048 + wn * 512;
        const bufrsrc_t wr = make_rsrc(p.qweight, bytes(kb, wbytes));
        const bufrsrc_t sr = make_rsrc(sp, bytes(kb, sbytes)), zr = make_rsrc(zp, bytes(kb, zbytes));
        uint32_t so, ss, sz;
        if constexpr (PREP) {
            so = (uint32_t)(kb >> 1) * 1024u + (uint32_t)(kb & 1) * 512u;
            // table rows of the stage's two 32-row halves (the same for groups of 64 rows or more)
            ss = (p.G >= 128 ? (uint32_t)kb >> 1 : gi) * 64u;
            sz = ss + (gm - 1) * 64u;
        } else {
            so = AWQ ? (uint32_t)kb * (uint32_t)(DIR_K * NW) * 4u : (uint32_t)kb * (uint32_t)(8 * p.N) * 4u;
            ss = gi * (uint32_t)p.N * 2u;
            sz = gi * (uint32_t)NW * 4u;
        }
        dma_lds<16>(wr, dst, wbase[0], so);
        dma_lds<16>(wr, dst + 1024, wbase[1], so);
        dma_lds<4>(sr, meta, sbase, ss);
        dma_lds<4>(zr, meta + 256, zbase, sz);
        const bool next = ++gc == gd;
        gi += next ? gm : 0u;
        gc = next ? 0 : gc;
    };

    // ---- Per column, for the fp16 pairs v of the exponent trick (1024 + q, or 1024 + 16 q where
    // the nibble stays at bits 4..7): q - z = v - (1024 + z), or fma(v, 1/16, -(64 + z)), both
    // exact; then one rounded product with the scale. bf16: the scale and -z s in fp32.
    constexpr uint32_t H16 = 0x2C00u;                 // fp16 1/16
    const half2_t sixteenth = as_h2(H16 | (H16 << 16)), one16 = as_h2(0x3C00u | (H16 << 16));
    (void)sixteenth; (void)one16;
    half2_t he[CPL], ho[PREP ? CPL : 1], hs[CPL];
    float fs[CPL], fnz[CPL];
    (void)he; (void)ho; (void)hs; (void)fs; (void)fnz;
    const int mhalf = PREP ? (h >> 1) * 256 : p.G < DIR_K ? (h >> 1) * 128 : 0;
    const uint32_t zo = AWQ ? 0u : (uint32_t)p.zero_offset;
    uint32_t e[CPL], zw = 0;   // raw scales (or table entries) and zero word of the next stage
    auto read_meta = [&](const int slot) __attribute__((always_inline)) {
        const unsigned char* meta = Wb + slot * (NWN * DIR_WST) + NWN * 2048 + wn * 512 + mhalf;
        if constexpr (PREP) {
#pragma unroll
            for (int c = 0; c < CPL; ++c) e[c] = *reinterpret_cast<const uint32_t*>(meta + 64 * c + 4 * j);
        } else {
            const u32x2 v = *reinterpret_cast<const u32x2*>(meta + 8 * j);
            e[0] = v.x; e[1] = v.y;
            zw = *reinterpret_cast<const uint32_t*>(meta + 256 + 4 * (j >> 1));
        }
    };
    auto set_meta = [&]() __attribute__((always_inline)) {
        const uint32_t zs = zw >> (AWQ ? 8 * (j & 1) : 16 * (j & 1));
#pragma unroll
        for (int c = 0; c < CPL; ++c) {
            // -(1024 + z): 0xE400 + z; -(64 + z): 0xD400 + 16 z (z <= 31)
            if constexpr (PREP) {
                const uint32_t z = e[c] >> 16;
                he[c] = as_h2(z * 0x10001u + 0xE400E400u);
                ho[c] = as_h2(z * 0x100010u + 0xD400D400u);
                hs[c] = as_h2(perm(e[c], e[c], 0x01000100u));
            } else {
                const uint32_t z = (zs >> (AWQ ? 4 * (c >> 1) + 16 * (c & 1) : 4 * c)) & 0xFu;
                const uint32_t s2 = e[c >> 1];
                if constexpr (BF) {
                    fs[c] = c & 1 ? __uint_as_float(s2 & 0xFFFF0000u) : __uint_as_float(s2 << 16);
                    fnz[c] = -(float)(z + zo) * fs[c];
                } else {
                    if constexpr (AWQ) he[c] = as_h2(c < 2 ? z * 0x10001u + 0xE400E400u : z * 0x100010u + 0xD400D400u);
                    else he[c] = as_h2(z * 0x100001u + (0xD400E400u + zo * 0x100001u));
                    hs[c] = as_h2(perm(s2, s2, c & 1 ? 0x03020302u : 0x01000100u));
                }
            }
        }
    };
    // The words of step st of the stage in ring slot sl: for GPTQ and the prepared layout one per
    // column, for AWQ the lane's half of 8 rows' words
    constexpr int NWD = AWQ ? 8 : CPL;
    auto read_w = [&](const int sl, const int st, uint32_t (&w)[NWD]) __attribute__((always_inline)) {
        const unsigned char* slot = Wb + sl * (NWN * DIR_WST);
        if constexpr (AWQ) {
            const int row = nat ? 32 * st + 8 * h : 16 * h + 8 * st;
            const uint32_t* wp = reinterpret_cast<const uint32_t*>(
                NWN == 4 ? slot + row * 128 + (((2 * wn + (j >> 3)) ^ (2 * h)) << 4) + ((j >> 1) & 3) * 4
                         : slot + (32 * st + h) * 64 + (2 * wn + (j >> 3)) * 16 + ((j >> 1) & 3) * 4);
#pragma unroll
            for (int r = 0; r < 8; ++r) w[r] = wp[(NWN == 4 ? 32 : 64) * r];
        } else if constexpr (PREP) {
            // rows 16 h + 8 st .. of strip c: word 2 (h & 1) + st of lane chunk (h / 2, j)
#pragma unroll
            for (int c = 0; c < CPL; ++c)
                w[c] = *reinterpret_cast<const uint32_t*>(slot + wn * 2048 + c * 512 + ((h >> 1) * 16 + j) * 16 + (h & 1) * 8 + st * 4);
        } else {
            const u32x4 v = *reinterpret_cast<const u32x4*>(slot + wn * 2048 + (nat ? 4 * st + h : 2 * h + st) * 256 + j * 16);
            w[0] = v.x; w[1] = v.y; w[2] = v.z; w[3] = v.w;
        }
    };
    // the B operands from a step's words: column c of the lane, 8 rows in natural order
    auto dequant = [&](const uint32_t (&w)[NWD], v8_t (&bf)[CPL]) __attribute__((always_inline)) {
        if constexpr (AWQ) {
            uint32_t pr[CPL][4];
            const uint32_t sel = j & 1 ? 0x07050301u : 0x06040200u;   // bytes of the lane's columns
#pragma unroll
            for (int rp = 0; rp < 4; ++rp) {
                // bytes (row a: columns 0 | 2, 1 | 3; row b: the same)
                const uint32_t P = perm(w[2 * rp + 1], w[2 * rp], sel);
                if constexpr (BF) {
                    const uint32_t e = P & 0x0F0F0F0Fu, o = (P >> 4) & 0x0F0F0F0Fu;
#pragma unroll
                    for (int c = 0; c < CPL; ++c) {
                        const uint32_t v = c < 2 ? e : o;
                        const float a = (float)((v >> (8 * (c & 1))) & 0xFFu), b = (float)((v >> (8 * (c & 1) + 16)) & 0xFFu);
                        pr[c][rp] = pack2(bf16_t{}, __builtin_fmaf(a, fs[c], fnz[c]), __builtin_fmaf(b, fs[c], fnz[c]));
                    }
                } else {
                    const uint32_t Q = P >> 8;
                    pr[0][rp] = as_u32((nib_pair(P) + he[0]) * hs[0]);
                    pr[1][rp] = as_u32((nib_pair(Q) + he[1]) * hs[1]);
                    pr[2][rp] = as_u32(__builtin_elementwise_fma(nib_pair16(P), sixteenth, he[2]) * hs[2]);
                    pr[3][rp] = as_u32(__builtin_elementwise_fma(nib_pair16(Q), sixteenth, he[3]) * hs[3]);
                }
            }
#pragma unroll
            for (int c = 0; c < CPL; ++c) bf[c] = __builtin_bit_cast(v8_t, u32x4{pr[c][0], pr[c][1], pr[c][2], pr[c][3]});
        } else {
#pragma unroll
            for (int c = 0; c < CPL; ++c) {
                const uint32_t v = w[c];
                uint32_t q[4];
                if constexpr (PREP) {
                    const uint32_t u = v >> 8;
                    q[0] = as_u32((nib_pair(v) + he[c]) * hs[c]);
                    q[1] = as_u32(__builtin_elementwise_fma(nib_pair16(v), sixteenth, ho[c]) * hs[c]);
                    q[2] = as_u32((nib_pair(u) + he[c]) * hs[c]);
                    q[3] = as_u32(__builtin_elementwise_fma(nib_pair16(u), sixteenth, ho[c]) * hs[c]);
                } else if constexpr (BF) {
                    const uint32_t e = v & 0x0F0F0F0Fu, o = (v >> 4) & 0x0F0F0F0Fu;
#pragma unroll
                    for (int i = 0; i < 4; ++i)
                        q[i] = pack2(bf16_t{}, __builtin_fmaf((float)((e >> (8 * i)) & 0xFFu), fs[c], fnz[c]),
                                     __builtin_fmaf((float)((o >> (8 * i)) & 0xFFu), fs[c], fnz[c]));
                } else {
                    // byte i (rows 2 i, 2 i + 1) in both halves: (1024 + q_2i, 1024 + 16 q_2i+1)
                    const uint32_t lo = perm(v, v, 0x01000100u), hi = perm(v, v, 0x03020302u);
                    const uint32_t src[4] = {lo, lo >> 8, hi, hi >> 8};
#pragma unroll
                    for (int i = 0; i < 4; ++i) {
                        const half2_t n = as_h2(and_or(src[i], vconst(0x00F0000Fu), vconst(MAGIC2)));
                        q[i] = as_u32(__builtin_elementwise_fma(n, one16, he[c]) * hs[c]);
                    }
                }
                bf[c] = __builtin_bit_cast(v8_t, u32x4{q[0], q[1], q[2], q[3]});
            }
        }
    };

    float4_t acc[R][CPL];
#pragma unroll
    for (int r = 0; r < R; ++r)
#pragma unroll
        for (int c = 0; c < CPL; ++c) acc[r][c] = float4_t{0.f, 0.f, 0.f, 0.f};
    // A operand of step st: chunk (natural 4 st + h, else 2 h + st) of row j of a block
    uint32_t apos[2];
#pragma unroll
    for (int st = 0; st < 2; ++st)
        apos[st] = (uint32_t)(j * 128 + (((nat ? 4 * st + h : 2 * h + st) ^ (j & 7)) << 4));

    auto load = [&](int s, const int slot) __attribute__((always_inline)) {
        asm volatile("" ::: "memory");
        load_a(s, slot);
        load_w(s, slot);
        asm volatile("" ::: "memory");
    };
    // At the top of stage s: stage s + 1 is in LDS once only the loads of the stages after it are
    // in flight (D - 3 stages); after the barrier everybody's are, and every wave is past its
    // reads of stage s - 1's slot
    auto ready = [&]() __attribute__((always_inline)) {
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        wait_vmcnt<(D - 3) * (DL + RL)>();
        if constexpr (NWN > 1) __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
    };
    // Software pipeline over the steps: while a step's MFMAs run, the next step's x operands and
    // the words of the step after it are read from LDS, and the next step's B operands are made
    v8_t af[2][R], bf[2][CPL];
    uint32_t w[2][NWD];
    auto read_a = [&](const int slot, const int st) __attribute__((always_inline)) {
        const unsigned char* A = Ab + slot * A_ST;
#pragma unroll
        for (int r = 0; r < R; ++r) af[st][r] = *reinterpret_cast<const v8_t*>(A + r * 2048 + apos[st]);
    };
    auto mul = [&](const int st) __attribute__((always_inline)) {
#pragma unroll
        for (int r = 0; r < R; ++r)
#pragma unroll
            for (int c = 0; c < CPL; ++c) acc[r][c] = mfma16x16x32(af[st][r], bf[st][c], acc[r][c]);
    };
    // A step's reads and arithmetic stay inside it. Long steps are spread by hand, one MFMA to an LDS
    // read and a share of the step's about 80 VALU instructions: the compiler's own order ends in runs
    // of 60 VALU and 25 MFMAs, which one or two waves per SIMD do not overlap (K = 4096, GPTQ: bf16,
    // 200 rows N = 6144 / 28672 32.8 / 72.4 -> 29.6 / 61.6 us; fp16, N = 28672 112 / 220 rows 57.4 /
    // 60.3 -> 54.6 / 58.8 us). fp16 below five row blocks: no gain (333 rows, N = 6144 45.0, 45.7 us).
    // bf16 with one row block has too few MFMAs to spread over: left to the compiler (AWQ, 9 rows,
    // 1792 -> 4096 / 4096 -> 6144 / 14336 -> 4096 10.0 / 15.9 / 20.4 -> 8.5 / 12.8 / 17.1 us)
    auto order = [&]() __attribute__((always_inline)) {
        if constexpr ((BF && R >= 2) || R >= 5) {
            constexpr int M = CPL * R, V = (80 + M - 1) / M;
#pragma unroll
            for (int i = 0; i < M; ++i) {
                __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
                if (i < R + 6) __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
                __builtin_amdgcn_sched_group_barrier(0x002, V, 0);
            }
        }
        __builtin_amdgcn_sched_barrier(0);
    };
    auto stage = [&](int s, const int u) __attribute__((always_inline)) {
        const int nx = (u + 1) % D;
        if (s) ready();
        load(s + D - 1, (u + D - 1) % D);
        read_a(u, 1);
        read_w(nx, 0, w[0]);
        read_meta(nx);
        dequant(w[1], bf[1]);
        mul(0);
        order();
        read_a(nx, 0);
        set_meta();
        dequant(w[0], bf[0]);
        read_w(nx, 1, w[1]);
        mul(1);
        order();
    };
#pragma unroll
    for (int s = 0; s < D - 1; ++s) load(s, s);
    ready();
    read_meta(0);
    read_w(0, 0, w[0]);
    read_w(0, 1, w[1]);
    read_a(0, 0);
    set_meta();
    dequant(w[0], bf[0]);
    for (int s = 0; s < ns; s += D) {
#pragma unroll
        for (int u = 0; u < D; ++u) {
            if (u && s + u >= ns) break;
            stage(s + u, u);
        }
    }
    wait_vmcnt<0>();   // no LDS write may be in flight when the LDS is used again or given back

    // ---- the K groups' sums, halves added pairwise through LDS
    if constexpr (KW > 1) {
        float4_t* red = reinterpret_cast<float4_t*>(lds);
#pragma unroll
        for (int half = KW / 2; half >= 1; half /= 2) {
            __syncthreads();
            if (kw >= half && kw < 2 * half) {
#pragma unroll
                for (int r = 0; r < R; ++r)
#pragma unroll
                    for (int c = 0; c < CPL; ++c)
                        red[((((kw - half) * NWN + wn) * R + r) * CPL + c) * 64 + lane] = acc[r][c];
            }
            __syncthreads();
            if (kw < half) {
#pragma unroll
                for (int r = 0; r < R; ++r)
#pragma unroll
                    for (int c = 0; c < CPL; ++c)
                        acc[r][c] += red[(((kw * NWN + wn) * R + r) * CPL + c) * 64 + lane];
            }
        }
    }

    // rows 16 r + 4 h + i of the lane's columns (col0: its first)
    auto store_rows = [&](int r, int col0, const float4_t (&v)[CPL]) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int row = 16 * r + 4 * h + i;
            if (row >= rows) continue;
            int m = m0 + row;
            if constexpr (MOE) {
                m = p.sorted_ids[m0 + row];
                if ((unsigned)m >= (unsigned)p.num_pairs) continue;
            }
            E* o = reinterpret_cast<E*>(p.out) + (size_t)m * p.N + col0;
            if constexpr (PREP) {
#pragma unroll
                for (int c = 0; c < CPL; ++c)
                    if (col0 + 16 * c < p.N) o[16 * c] = (E)v[c][i];
            } else {
                if (col0 >= p.N) continue;
                *reinterpret_cast<u32x2*>(o) = u32x2{pack2(E{}, v[0][i], v[1][i]), pack2(E{}, v[2][i], v[3][i])};
            }
        }
    };
    const int lcol = PREP ? j : CPL * j;
    if constexpr (!MOE) if (ksp > 1) {   // not by expert: no room for the flag beside 160 KiB of rings
        // partials in operand order, then the last split of the tile to arrive adds all of
        // them in split order
        __shared__ int last_flag;
        constexpr int TILE = NWN * R * CPL * 256;
        const int tile = ct * p.row_tiles + rt;
        float* base = p.ws + (size_t)tile * ksp * TILE;
        // Stored as 64-bit words: a 16-byte buffer store with a scalar offset lost its first dword
        // here when the next instruction overwrote that register (the compiler puts no wait state
        // between the two, and lanes 12..15 of each 16 stored the new value)
        if (kw == 0) {
#pragma unroll
            for (int r = 0; r < R; ++r)
#pragma unroll
                for (int c = 0; c < CPL; ++c)
                    st_partial4<SCOPE_DEVICE>(base + (size_t)bz * TILE + (((wn * R + r) * CPL + c) * 64 + lane) * 4, acc[r][c]);
        }
        if (!splitk_arrive(splitk_counter(p.counters, tile), ksp, &last_flag)) return;
        // the waves share the NWN R row blocks of 64 columns, NG at a time, with the 16-byte loads
        // (sc1: coherent between the XCDs) of a few splits in flight together
        constexpr int NG = 2, AUX_SC1 = 16;
        const bufrsrc_t pr = make_rsrc(base, (uint32_t)ksp * (TILE * 4u));
        for (int q0 = wave * NG; q0 < NWN * R; q0 += W * NG) {
            float4_t v[NG][CPL];
#pragma unroll
            for (int g = 0; g < NG; ++g)
#pragma unroll
                for (int c = 0; c < CPL; ++c) v[g][c] = float4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll 4
            for (int sp = 0; sp < ksp; ++sp)
#pragma unroll
                for (int g = 0; g < NG; ++g)
#pragma unroll
                    for (int c = 0; c < CPL; ++c)
                        v[g][c] += __builtin_bit_cast(float4_t, __builtin_amdgcn_raw_buffer_load_b128(
                            pr, (uint32_t)((((q0 + g) * CPL + c) * 64 + lane) * 16), (uint32_t)sp * (TILE * 4u), AUX_SC1));
#pragma unroll
            for (int g = 0; g < NG; ++g) {
                const int q = q0 + g, gw = q / R;
                if (q < NWN * R) store_rows(q - gw * R, n0 + gw * WC + lcol, v[g]);
            }
        }
        return;
    }
    if (kw == 0) {
#pragma unroll
        for (int r = 0; r < R; ++r) store_rows(r, nw0 + lcol, acc[r]);
    }
}

template <int FMT, typename E, int R, int NWN, int KW>
__global__ void __launch_bounds__(64 * NWN * KW, 2) direct_kernel(PrefillParams p) {
    extern __shared__ __attribute__((aligned(16))) unsigned char lds[];
    if (p.gate && *p.gate != p.gate_want) return;   // uniform: the whole grid returns
    int ct, rt, bz;
    if (!direct_place(p, p.row_tiles, ct, rt, bz)) return;
    direct_tile<FMT, E, R, NWN, KW, false>(p, lds, ct, rt, bz, rt * 16 * R, min(16 * R, p.M - rt * 16 * R));
}

// 8 experts of 4096 -> 28672 and 14336 -> 4096, top 2: 16 tokens 228 + 182 -> 124 + 63 us (traced;
// the weights alone take 92 + 46 at the rate of a large copy), 512 tokens 422 + 203 -> 318 + 176 us.
// Grouped by expert: row tile rt is entry rt of the tile list ({first sorted row, rows, expert, 0});
// the tile's rows, known on the device only, pick the code for their number of 16-row blocks, so
// that a tile costs what its rows need. The K groups' LDS must hold 16 RMAX rows.
template <int FMT, int RMAX, int NWN, int KW>
__global__ void __launch_bounds__(64 * NWN * KW, 2) direct_moe_kernel(PrefillParams p) {
    extern __shared__ __attribute__((aligned(16))) unsigned char lds[];
    const int rts = min(*p.num_tiles, p.row_tiles);
    int ct, rt, bz;
    if (rts <= 0 || !direct_place(p, rts, ct, rt, bz)) return;
    const int32_t* td = p.tiles + 4 * rt;
    const int m0 = td[0], rows = td[1], e = td[2];
    p.qweight += (size_t)e * p.qweight_stride;
    if (FMT != FMT_PREP) {
        p.scales += (size_t)e * p.scales_stride;
        if (p.qzeros) p.qzeros += (size_t)e * p.qzeros_stride;
    }
    auto run = [&](auto r) __attribute__((always_inline)) {
        direct_tile<FMT, half_t, decltype(r)::value, NWN, KW, true>(p, lds, ct, rt, bz, m0, rows);
    };
    if (rows <= 16) run(std::integral_constant<int, 1>{});
    else if (rows <= 32) run(std::integral_constant<int, 2>{});
    else if (rows <= 48) run(std::integral_constant<int, 3>{});
    else if (rows <= 64) run(std::integral_constant<int, 4>{});
    else if constexpr (RMAX > 4) {
        if (rows <= 80) run(std::integral_constant<int, 5>{});
        else if (rows <= 96) run(std::integral_constant<int, 6>{});
        else run(std::integral_constant<int, 7>{});
    }
}

}  // namespace w4a16

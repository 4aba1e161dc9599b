// k_qgemm_tile.hip -- quantized GEMM Y[M][N] = X[M][K] . W[N][K]^T on the bf16 matrix cores for prompts
// that make enough tiles (qgemm_tiled; IWeightTensor.MatMul over many rows; NeuralNet.cs:145-298,
// MatMulF32Q8.cs:23-80) and rows of whole 256-element super-blocks.
//
// Exactness is that of k_qgemm.hip: integer weight codes in bf16, activations as three bf16
// parts whose sum is the fp32 value, fp32 accumulation, block scales applied to the fp32 result
// of each 32-element sub-block.  The code offset and the min term of a sub-block multiply the sum
// of its activations.  Whoever writes the parts writes that sum too (xp_sums, three bf16 parts),
// and a super-block's terms sum_j b_j sx_j (b = -(sc * offset + m), three bf16 parts built in
// registers) are one small product over its 8 (Q6_K: 16) sums: the six leading part products,
// exact to 2^-24 of each term, 3 (6) matrix instructions per tile and super-block in place of one
// fused multiply-add per output and sub-block.
//
// What bounds it: the matrix cores issue three products (hi, mid, lo) per useful one, so the
// ceiling is a third of the bf16 rate; next come the CU's data paths.  A wave that loads its own
// activation parts moves 6 bytes per token and k through the CU's 64 B/clk vector-memory path
// for 32-64 rows of work, which limits the K-split kernel (k_qgemm.hip: up to 16 tokens, and
// prompts of few tiles) to 15-27 % matrix-core use.  Hence:
//   * a wave computes 64 rows x 32 TT tokens (v_mfma_f32_32x32x16_bf16: a lane owns one weight
//     row per tile, so block scales are decoded by 2 lanes instead of 4);
//   * WR waves of a workgroup take different rows and share one copy of the parts in LDS, which
//     cuts the part traffic per product by WR; each wave's weights are its own;
//   * WK > 1: groups of WR waves take different K ranges (matrices of few rows, where rows and
//     tokens alone do not fill the chip); their tiles are added through LDS in a fixed order;
//   * parts and weights go straight into LDS (global_load_lds_dwordx4) two steps or more ahead of
//     use, so no registers hold loads in flight and two workgroups fit a CU.
//
// Operand layout: A = activation parts (32 tokens x 16 k), B = weight codes (16 k x 32 rows).
// Lane l supplies token / row l % 32 and 8 of the 16 k-values: group g = 2 mf + l / 32 of the
// sub-block's four 8-element groups for product mf = 0, 1, so product mf covers 16-element half
// mf of the sub-block (the halves that carry their own scale in Q6_K).  D lane l holds tokens
// 8 (i / 4) + 4 (l / 32) + i % 4 of weight row l % 32 in register i.
#include <algorithm>
#include <type_traits>

#include "smx_qgemm.h"

#ifndef SMX_TILE_FMT
#error "compile with -DSMX_TILE_FMT=<Fmt>"
#endif

namespace smx {

namespace {

template <int N> using ic = std::integral_constant<int, N>;

typedef float f32x16 __attribute__((ext_vector_type(16)));

__device__ __forceinline__ f32x16 mfma32(uint4 a, uint4 b, f32x16 c)
{
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(as_bf16x8(a), as_bf16x8(b), c, 0, 0, 0);
}

// 16 bytes (4 bytes) per active lane from base + off (base wave-uniform) into LDS at l + 16 (4) * lane
__device__ __forceinline__ void lds_dma16s(const uint8_t *base, uint32_t off, const void *l)
{
    const uint32_t la = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) const void *)l;
    asm volatile("s_nop 0\n\tglobal_load_lds_dwordx4 %0, %1" ::"v"(off), "s"(base), "{m0}"(la) : "memory");
}
__device__ __forceinline__ void lds_dma4s(const uint8_t *base, uint32_t off, const void *l)
{
    const uint32_t la = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) const void *)l;
    asm volatile("s_nop 0\n\tglobal_load_lds_dword %0, %1" ::"v"(off), "s"(base), "{m0}"(la) : "memory");
}

__device__ __forceinline__ uint32_t or_and(uint32_t e, uint32_t m, uint32_t o)
{
    return __builtin_amdgcn_bitop3_b32(e, m, o, 0xEA);   // (e & m) | o
}

// 4-bit codes: 16 + q = bf16 0x4180 | q << 3.  Codes sit high in the mantissa, so that the implicit
// leading one, and with it the offset that the activation sums remove, is as small as the code
// width allows: 16 + q (4 bits), 32 + q (5 bits), 64 + q (6 bits).
__device__ __forceinline__ uint4 codes4(uint32_t v)
{
    return make_uint4(or_and(v << 3, 0x00780078u, 0x41804180u), or_and(v >> 1, 0x00780078u, 0x41804180u),
                      or_and(v >> 5, 0x00780078u, 0x41804180u), or_and(v >> 9, 0x00780078u, 0x41804180u));
}

// int8 codes, signed and exact in bf16: no offset
__device__ __forceinline__ uint4 codes8(uint32_t a, uint32_t b)
{
    auto f = [](uint32_t v, int k) { return (float)(int8_t)(v >> (8 * k)); };
    return make_uint4(pack_hi16(f(a, 0), f(b, 0)), pack_hi16(f(a, 1), f(b, 1)), pack_hi16(f(a, 2), f(b, 2)),
                      pack_hi16(f(a, 3), f(b, 3)));
}

// What a wave stages per weight row, in 16-byte pieces: kC bytes of codes per two sub-blocks
// (at kCOff of the super-block), kX: 16 bytes per kX sub-blocks (high bits, or fp32 scales), and 16
// bytes per super-block (kHOff; scales, header).  kOff: the code offset; kSums: kind of the sums
// read.
template <int F> struct TQ;
template <> struct TQ<FMT_Q8_0> {
    static constexpr int kC = 64, kCOff = 0, kX = 0, kXOff = 0, kSums = 0;
    static constexpr bool kH = true, kHD = true, kD = false, kXD = false;
    static constexpr float kOff = 0.0f;
};
template <> struct TQ<FMT_SQ8> {
    static constexpr int kC = 64, kCOff = 0, kX = 4, kXOff = 0, kSums = 0;
    static constexpr bool kH = false, kHD = false, kD = false, kXD = true;
    static constexpr float kOff = 0.0f;
};
template <> struct TQ<FMT_Q4_0> {
    static constexpr int kC = 32, kCOff = 0, kX = 0, kXOff = 0, kSums = 1;
    static constexpr bool kH = true, kHD = true, kD = false, kXD = false;
    static constexpr float kOff = 24.0f;
};
template <> struct TQ<FMT_SQ4> {
    static constexpr int kC = 32, kCOff = 0, kX = 4, kXOff = 0, kSums = 1;
    static constexpr bool kH = false, kHD = false, kD = false, kXD = true;
    static constexpr float kOff = 24.0f;
};
template <> struct TQ<FMT_Q4_K> {
    static constexpr int kC = 32, kCOff = 16, kX = 0, kXOff = 0, kSums = 1;
    static constexpr bool kH = true, kHD = false, kD = false, kXD = false;
    static constexpr float kOff = 16.0f;
};
template <> struct TQ<FMT_Q5_K> {
    static constexpr int kC = 32, kCOff = 48, kX = 4, kXOff = 16, kSums = 1;
    static constexpr bool kH = true, kHD = false, kD = false, kXD = false;
    static constexpr float kOff = 48.0f;
};
template <> struct TQ<FMT_Q6_K> {
    static constexpr int kC = 32, kCOff = 0, kX = 2, kXOff = 128, kSums = 2;
    static constexpr bool kH = true, kHD = false, kD = true, kXD = false;
    static constexpr float kOff = 96.0f;
};
constexpr int tile_hoff(int f) { return f == FMT_Q6_K ? 192 : 0; }

__device__ __forceinline__ uint32_t word(const uint4 &v, int i) { return i == 0 ? v.x : i == 1 ? v.y : i == 2 ? v.z : v.w; }

// Scales of sub-block j: sc (first 16 elements) and sc2 (second 16; the same except in Q6_K), and the
// min m.
struct TScl {
    float sc, sc2, m;
};

// Tile order: workgroup i runs tile (i % 8) * chunk + i / 8 of a panel-major order (panels of G
// token groups, the G groups fastest within a panel), so that each XCD works through one
// contiguous chunk in which G neighbouring workgroups share their weights and the row groups of
// a panel share its activation parts in the XCD's L2.  A bijection onto the R * T tiles.
struct TileOrder {
    uint32_t R, T, G, chunk;
};

// The loads of a workgroup's ring and the waits for them.  Step i (mod 8) multiplies sub-block i with
// codes and first-tile parts that the step before it fetched from LDS, and fetches those of
// sub-block u = i + 1.  It requests, in this order, the parts of sub-block i + D, every weight stream
// whose period starts at u (its group after next: codes every 2 sub-blocks, X every kX, headers
// every 8) and, at i = 0, the super-block's sums.  wait(i): how many of the wave's youngest loads may
// still be in flight when step i begins, i.e. the number of loads issued after the youngest one
// that the step fetches.
template <int F, int NPW, int D, int NSW> struct TileLoads {
    using Q = TQ<F>;
    static constexpr int KX = Q::kX ? Q::kX : 8;
    static constexpr int streams(int j)
    {
        const int u = ((j + 1) % 8 + 8) % 8;
        int n = u % 2 == 0 ? Q::kC / 16 : 0;
        if (Q::kX && u % KX == 0) n += 1;
        if (u == 0) n += (Q::kH ? 1 : 0) + (Q::kD ? 1 : 0);
        return n;
    }
    static constexpr int sums(int j) { return (j % 8 + 8) % 8 == 0 ? NSW : 0; }
    static constexpr int after(int i, int back)   // loads of the steps i - back + 1 .. i - 1
    {
        int n = 0;
        for (int k = i - back + 1; k < i; k++) n += NPW + streams(k) + sums(k);
        return n;
    }
    static constexpr int wait(int i)
    {
        int n = after(i, D - 1) + streams(i + 1 - D) + sums(i + 1 - D);   // the parts of sub-block i + 1
        const int u = (i + 1) % 8;
        for (int p = 2; p <= 8; p++) {
            const bool use = (p == 2 && u % 2 == 0) || (Q::kX && p == KX && u % KX == 0) || (p == 8 && u == 0);
            const int a = after(i, p) + sums(i - p);
            if (use && a < n) n = a;
        }
        if (i == 7 && NSW && after(7, 7) < n) n = after(7, 7);   // the sums, requested at step 0
        return n < 63 ? n : 63;
    }
};

template <int F, int WR, int WK, int TT, int D>
__global__ __launch_bounds__(64 * WR * WK, 2) void k_qgemm_tile(QgemmArgs a, TileOrder to)
{
    using Q = TQ<F>;
    constexpr int kB = fmt_kquant(F) ? fmt_main_bytes(F) : 8 * fmt_main_bytes(F);   // row bytes per super-block
    constexpr int T16 = 2 * TT;                       // 16-token tiles
    constexpr int NB = 3 * T16;                       // 1 KB part blocks per sub-block
    constexpr int NPW = NB / WR;                      // ... per wave
    constexpr int SL = D + 1;                         // part slots
    constexpr int NS = Q::kSums;
    constexpr int SUMB = NS * 768 * T16;              // sum bytes of a super-block (all tokens)
    constexpr int NSW = (SUMB / 16 + 64 * WR - 1) / (64 * WR);   // sum loads per wave and super-block
    using Ld = TileLoads<F, NPW, D, NSW>;
    static_assert(NB % WR == 0 && D >= 2, "work split; parts are read one step ahead");
    struct WaveW {
        uint8_t c[2][64 * Q::kC];
        uint8_t x[Q::kX ? 2 : 0][1024];
        uint8_t h[Q::kH ? 2 : 0][1024];
        uint32_t d[Q::kD ? 2 : 0][64];
    };
    struct Lds {
        uint4 part[WK][SL][NB][64];
        uint8_t sum[WK][NSW * WR * 1024];
        WaveW w[WR * WK];
    };
    struct Red {
        f32x16 t[WK > 1 ? WK - 1 : 1][WR][2][TT][64];
    };
    __shared__ __align__(16) uint8_t s_mem[sizeof(Lds) > sizeof(Red) || WK == 1 ? sizeof(Lds) : sizeof(Red)];
    Lds &L = *(Lds *)s_mem;
    Red &R = *(Red *)s_mem;   // reuses the ring once the last step is done
    const WView &w = a.w;
    const int M = a.M;
    const int wv = wave_id();
    const int wr = wv % WR, kg = wv / WR;
    const int lane = lane_id();
    const int h = lane >> 5, li = lane & 31;
    const uint32_t N = (uint32_t)w.rows;
    const int nsb = (int)(w.cols >> 5), nsup = nsb >> 3;
    const int ntt = (M + 15) >> 4;
    uint32_t bx, by;
    {
        const uint32_t i = blockIdx.x, t = (i & 7u) * to.chunk + (i >> 3);
        if (t >= to.R * to.T) return;   // the whole workgroup
        const uint32_t pt = to.R * to.G, panel = t / pt, rem = t - panel * pt;
        const uint32_t gp = min(to.G, to.T - panel * to.G);
        bx = rem / gp;
        by = panel * to.G + (rem - bx * gp);
    }
    const uint32_t row0 = (bx * WR + (uint32_t)wr) * 64u;   // this wave's rows
    const int tt0 = (int)by * T16;                           // this workgroup's first 16-token tile
    const int per = (nsup + WK - 1) / WK;
    const int sup0 = kg * per, sup1 = min(sup0 + per, nsup);
    const uint32_t row_bytes = (uint32_t)nsup * kB;
    WaveW &W = L.w[wv];

    // Byte offsets of this lane's 16-byte pieces of the codes of two sub-blocks: slot i = 64 k + lane
    // holds row i / P, piece (i % P) ^ swizzle (P pieces per row), so that reads of one piece over
    // neighbouring rows fall on distinct banks.
    constexpr int NC = Q::kC / 16;
    uint32_t coff[NC];
#pragma unroll
    for (int k = 0; k < NC; k++) {
        const uint32_t i = 64u * k + (uint32_t)lane, r = i / NC, p = (i % NC) ^ (NC == 4 ? (r >> 2) & 3u : (r >> 3) & 1u);
        coff[k] = min(row0 + r, N - 1) * row_bytes + Q::kCOff + 16u * p;
    }
    const uint32_t rl = min(row0 + (uint32_t)lane, N - 1);   // row of the one-piece-per-row streams
    // requests the groups that follow those starting at sub-block u (0 .. 8) of super-block sup
    auto issue_w = [&](int sup, int u) {
        {
            const int e = u + 2, cs = min(sup + (e >> 3), nsup - 1), cg = (e & 7) >> 1;
            const uint8_t *b = w.q + (uint32_t)cs * kB + (uint32_t)cg * Q::kC;
#pragma unroll
            for (int k = 0; k < NC; k++) lds_dma16s(b, coff[k], W.c[cg & 1] + 1024 * k);
        }
        if constexpr (Q::kX > 0) {
            if (u % Q::kX == 0) {
                const int e = u + Q::kX, xs = min(sup + (e >> 3), nsup - 1), xg = (e & 7) / Q::kX;
                if constexpr (Q::kXD)   // 4 fp32 scales per row
                    lds_dma16s((const uint8_t *)w.d + (uint32_t)xs * 32u + 16u * xg, rl * (uint32_t)nsup * 32u, W.x[xg & 1]);
                else
                    lds_dma16s(w.q + (uint32_t)xs * kB + Q::kXOff + 16u * xg, rl * row_bytes, W.x[xg & 1]);
            }
        }
        if (u % 8 == 0) {
            const int nx = sup + (u >> 3) + 1, hs = min(nx, nsup - 1), sl = nx & 1;
            if constexpr (Q::kH) {
                if constexpr (Q::kHD) lds_dma16s((const uint8_t *)w.d + (uint32_t)hs * 16u, rl * (uint32_t)nsup * 16u, W.h[sl]);
                else lds_dma16s(w.q + (uint32_t)hs * kB + tile_hoff(F), rl * row_bytes, W.h[sl]);
            }
            if constexpr (Q::kD)   // the aligned word that holds the row's fp16 d
                lds_dma4s((const uint8_t *)w.d, ((rl * (uint32_t)nsup + (uint32_t)hs) * 2u) & ~3u, W.d[sl]);
        }
    };
    auto issue_x = [&](int s, int slot) {
        const int sc = min(s, nsb - 1);
#pragma unroll
        for (int k = 0; k < NPW; k++) {
            const int c = wr * NPW + k, tt = min(tt0 + c / 3, ntt - 1);
            lds_dma16s(a.xp + ((size_t)tt * nsb + sc) * 3072u + 1024u * (c % 3), (uint32_t)lane * 16u,
                       &L.part[kg][slot][c][0]);
        }
    };
    // sums of super-block sup: 48 NS pieces of 16 bytes per token tile
    auto issue_s = [&](int sup) {
        if constexpr (NS > 0) {
            const uint8_t *sums = a.xp + (size_t)ntt * nsb * 3072u + (size_t)sup * (768u * NS);
#pragma unroll
            for (int k = 0; k < NSW; k++) {
                const int i = (wr * NSW + k) * 64 + lane;
                const int tt = min(tt0 + min(i / (48 * NS), T16 - 1), ntt - 1), pc = i % (48 * NS);
                lds_dma16s(sums, (uint32_t)tt * (uint32_t)nsup * (768u * NS) + 16u * (uint32_t)pc,
                           &L.sum[kg][(wr * NSW + k) * 1024]);
            }
        }
    };

    uint32_t wrow[2];
#pragma unroll
    for (int r = 0; r < 2; r++) wrow[r] = min(row0 + 32u * r + (uint32_t)li, N - 1);
    f32x16 acc[2][TT];
#pragma unroll
    for (int r = 0; r < 2; r++)
#pragma unroll
        for (int t = 0; t < TT; t++)
#pragma unroll
            for (int i = 0; i < 16; i++) acc[r][t][i] = 0.0f;

    // the 8 codes of (row tile r, sub-block j, product mf), in bf16
    auto codes = [&](int r, int j, int mf) {
        const int row = 32 * r + li, js = j & 1, g = 2 * mf + h;
        const uint8_t *c = W.c[(j >> 1) & 1] + row * Q::kC;
        if constexpr (Q::kC == 64) {
            const uint2 v = *(const uint2 *)(c + 16 * ((2 * js + mf) ^ ((row >> 2) & 3)) + 8 * h);
            return codes8(v.x, v.y);
        } else {
            const uint32_t v = *(const uint32_t *)(c + 16 * (js ^ ((row >> 3) & 1)) + 8 * mf + 4 * h);
            if constexpr (F == FMT_Q4_0 || F == FMT_SQ4) {
                return codes4(v ^ 0x88888888u);
            } else if constexpr (F == FMT_Q4_K) {
                return codes4(v);
            } else if constexpr (F == FMT_Q5_K) {
                // 5-bit codes of the even / odd elements in bits 2-6 of each byte (the high-bit
                // layout is QW<FMT_Q5_K>'s); 32 + q = bf16 0x4200 | q << 2
                const uint32_t H = *(const uint32_t *)(W.x[(j >> 2) & 1] + 16 * row + 4 * (j & 3));
                const uint32_t hg = H >> (2 * g);
                const uint32_t e0 = bfi(0x3C3C3C3Cu, v << 2, hg << 6), e1 = bfi(0x3C3C3C3Cu, v >> 2, hg << 5);
                return make_uint4(or_and(e0, 0x007C007Cu, 0x42004200u), or_and(e1, 0x007C007Cu, 0x42004200u),
                                  or_and(e0 >> 8, 0x007C007Cu, 0x42004200u), or_and(e1 >> 8, 0x007C007Cu, 0x42004200u));
            } else {
                // 6-bit codes in bits 1-6; 64 + q = bf16 0x4280 | q << 1
                const uint2 H = *(const uint2 *)(W.x[(j >> 1) & 1] + 16 * row + 8 * js);
                const uint32_t e0 = bfi(0x1E1E1E1Eu, v << 1, (H.x >> (2 * g)) << 5);
                const uint32_t e1 = bfi(0x1E1E1E1Eu, v >> 3, (H.y >> (2 * g)) << 5);
                return make_uint4(or_and(e0, 0x007E007Eu, 0x42804280u), or_and(e1, 0x007E007Eu, 0x42804280u),
                                  or_and(e0 >> 8, 0x007E007Eu, 0x42804280u), or_and(e1 >> 8, 0x007E007Eu, 0x42804280u));
            }
        }
    };
    // scales of sub-block j from the row's header words
    auto scale = [&](const uint4 &hd, uint32_t d, int j) -> TScl {
        if constexpr (F == FMT_Q8_0 || F == FMT_Q4_0) {
            const float s = h2f((word(hd, j >> 1) >> (16 * (j & 1))) & 0xFFFFu);
            return {s, s, 0.0f};
        } else if constexpr (F == FMT_SQ8 || F == FMT_SQ4) {
            const float s = __uint_as_float(d);
            return {s, s, 0.0f};
        } else if constexpr (F == FMT_Q6_K) {
            const float df = h2f(d);
            const uint32_t p = word(hd, j >> 1) >> (16 * (j & 1));
            return {df * (float)(int8_t)(p & 0xFFu), df * (float)(int8_t)((p >> 8) & 0xFFu), 0.0f};
        } else {
            const float s = h2f(hd.x & 0xFFFFu) * (float)kq_scale6(hd.y, hd.z, hd.w, j, 0);
            return {s, s, h2f(hd.x >> 16) * (float)kq_scale6(hd.y, hd.z, hd.w, j, 1)};
        }
    };

    uint4 hd[2];
    uint32_t hdd[2] = {0, 0};
    // b operands of the sum products: bf16 parts of b = -(sc * offset + m) over the 8 sub-blocks,
    // arranged for this lane half (see add_sums)
    uint4 bs[2][NS > 0 ? 3 * NS : 1];
    float bv[2][NS == 1 ? 8 : 1];   // kind 1: b of each sub-block

    // Operands fetched one step ahead: codes and scales of the next sub-block, parts of its first
    // token tile.
    uint4 wc[2][2], xa[2][3];
    TScl sc[2];
    auto fetch_w = [&](int j, uint4 (*c)[2], TScl *z) {   // sub-block j of the super-block whose header is in hd
#pragma unroll
        for (int r = 0; r < 2; r++) {
            uint32_t d = hdd[r];
            if constexpr (Q::kXD) d = *(const uint32_t *)(W.x[(j >> 2) & 1] + 16 * (32 * r + li) + 4 * (j & 3));
            z[r] = scale(hd[r], d, j);
            if constexpr (NS == 1) bv[r][j] = -__builtin_fmaf(z[r].sc, Q::kOff, z[r].m);
#pragma unroll
            for (int mf = 0; mf < 2; mf++) c[r][mf] = codes(r, j, mf);
        }
    };
    auto fetch_x = [&](int slot, int t, uint4 (*x)[3]) {
#pragma unroll
        for (int mf = 0; mf < 2; mf++)
#pragma unroll
            for (int p = 0; p < 3; p++) x[mf][p] = L.part[kg][slot][3 * (2 * t + (li >> 4)) + p][16 * (2 * mf + h) + (li & 15)];
    };
    auto fetch_hdr = [&](int sup) {
#pragma unroll
        for (int r = 0; r < 2; r++) {
            if constexpr (Q::kH) hd[r] = *(const uint4 *)(W.h[sup & 1] + 16 * (32 * r + li));
            if constexpr (Q::kD) {
                const uint32_t odd = (wrow[r] * (uint32_t)nsup + (uint32_t)sup) & 1u;
                hdd[r] = (W.d[sup & 1][32 * r + li] >> (16u * odd)) & 0xFFFFu;
            }
        }
    };
    // Products of one chain: the two row tiles' products alternate.  A chain's scale step (acc += s *
    // d) runs while the matrix core works on the next chain.
    constexpr int CH = F == FMT_Q6_K ? 2 : 1;   // chains per token tile: one per scale of the sub-block
    f32x16 dp[2];
    float sp[2] = {0.0f, 0.0f};
#pragma unroll
    for (int r = 0; r < 2; r++)
#pragma unroll
        for (int i = 0; i < 16; i++) dp[r][i] = 0.0f;
    auto chain = [&](const uint4 (*x)[3], int q, f32x16 *d) {
#pragma unroll
        for (int r = 0; r < 2; r++)
#pragma unroll
            for (int i = 0; i < 16; i++) d[r][i] = 0.0f;
#pragma unroll
        for (int mf = CH == 2 ? q : 0; mf < (CH == 2 ? q + 1 : 2); mf++)
#pragma unroll
            for (int p = 0; p < 3; p++)
#pragma unroll
                for (int r = 0; r < 2; r++) d[r] = mfma32(x[mf][p], wc[r][mf], d[r]);
    };
    auto scale_prev = [&](int t) {
#pragma unroll
        for (int r = 0; r < 2; r++)
#pragma unroll
            for (int i = 0; i < 16; i++) acc[r][t][i] = __builtin_fmaf(sp[r], dp[r][i], acc[r][t][i]);
    };
    // acc += sum_j b_j sx_j of the super-block: with b = bh + bm + bl and sx = sh + sm + sl, the six
    // products bh sh, bm sh, bh sm, bl sh, bm sm, bh sl.  Kind 1: 8 terms, two products per
    // instruction (k half h of the operand): {bh | bm} {sh | sh}, {bh | bl} {sm | sh}, {bm | bh} {sm | sl}.
    // Kind 2: 16 terms, one product per instruction, half h = the sub-blocks' 16-element half.
    auto add_sums = [&]() {
        if constexpr (NS > 0) {
#pragma unroll
            for (int r = 0; r < 2; r++) {
                uint4 bp[3];
                uint32_t q[3][4];
#pragma unroll
                for (int k = 0; k < 4; k++) {
                    float x0, x1;
                    if constexpr (NS == 1) {
                        x0 = bv[r][2 * k];
                        x1 = bv[r][2 * k + 1];
                    } else {   // the scales of this lane half's 16 elements, from the header once more
                        const TScl s0 = scale(hd[r], hdd[r], 2 * k), s1 = scale(hd[r], hdd[r], 2 * k + 1);
                        x0 = -((h ? s0.sc2 : s0.sc) * Q::kOff);
                        x1 = -((h ? s1.sc2 : s1.sc) * Q::kOff);
                    }
#pragma unroll
                    for (int p = 0; p < 3; p++) {
                        q[p][k] = bf16_pair(x0, x1);
                        x0 -= __uint_as_float(q[p][k] << 16);
                        x1 -= __uint_as_float(q[p][k] & 0xFFFF0000u);
                    }
                }
#pragma unroll
                for (int p = 0; p < 3; p++) bp[p] = make_uint4(q[p][0], q[p][1], q[p][2], q[p][3]);
                auto sel = [&](const uint4 &x, const uint4 &y) {
                    return make_uint4(h ? y.x : x.x, h ? y.y : x.y, h ? y.z : x.z, h ? y.w : x.w);
                };
                if constexpr (NS == 1) {
                    bs[r][0] = sel(bp[0], bp[1]);
                    bs[r][1] = sel(bp[0], bp[2]);
                    bs[r][2] = sel(bp[1], bp[0]);
                } else {
                    bs[r][0] = bp[0]; bs[r][1] = bp[1]; bs[r][2] = bp[2];
                }
            }
#pragma unroll
            for (int t = 0; t < TT; t++) {
                const uint8_t *s = &L.sum[kg][0] + (2 * t + (li >> 4)) * (768 * NS) + (li & 15) * 16;
                if constexpr (NS == 1) {
                    const uint4 s0 = *(const uint4 *)s;
                    const uint4 s1 = *(const uint4 *)(s + (h ? 0 : 256));
                    const uint4 s2 = *(const uint4 *)(s + (h ? 512 : 256));
#pragma unroll
                    for (int r = 0; r < 2; r++) {
                        acc[r][t] = mfma32(s0, bs[r][0], acc[r][t]);
                        acc[r][t] = mfma32(s1, bs[r][1], acc[r][t]);
                        acc[r][t] = mfma32(s2, bs[r][2], acc[r][t]);
                    }
                } else {
                    uint4 sp[3];
#pragma unroll
                    for (int p = 0; p < 3; p++) sp[p] = *(const uint4 *)(s + 512 * p + 256 * h);
#pragma unroll
                    for (int p = 0; p < 3; p++)
#pragma unroll
                        for (int q = 0; q + p < 3; q++)
#pragma unroll
                            for (int r = 0; r < 2; r++) acc[r][t] = mfma32(sp[p], bs[r][q], acc[r][t]);
                }
            }
        }
    };

    // The wait of a step leaves in flight what later steps need; the barrier makes every wave's parts
    // visible and says that every wave has finished reading the slot that is filled next.  Past the
    // end of the range the loads repeat valid ones into slots whose contents are no longer used, so
    // the counts hold to the end.  K groups without super-blocks only take part in the barriers.
    const bool any = sup0 < sup1;
    if (any) {
        issue_w(sup0 - 1, 6);   // codes of sub-blocks 0, 1
        if constexpr (Q::kX > 0) {
            if constexpr (Q::kXD) lds_dma16s((const uint8_t *)w.d + (uint32_t)sup0 * 32u, rl * (uint32_t)nsup * 32u, W.x[0]);
            else lds_dma16s(w.q + (uint32_t)sup0 * kB + Q::kXOff, rl * row_bytes, W.x[0]);
        }
        if constexpr (Q::kH) {
            if constexpr (Q::kHD) lds_dma16s((const uint8_t *)w.d + (uint32_t)sup0 * 16u, rl * (uint32_t)nsup * 16u, W.h[sup0 & 1]);
            else lds_dma16s(w.q + (uint32_t)sup0 * kB + tile_hoff(F), rl * row_bytes, W.h[sup0 & 1]);
        }
        if constexpr (Q::kD) lds_dma4s((const uint8_t *)w.d, ((rl * (uint32_t)nsup + (uint32_t)sup0) * 2u) & ~3u, W.d[sup0 & 1]);
#pragma unroll
        for (int i = 0; i < D; i++) issue_x(sup0 * 8 + i, i);
        issue_w(sup0, 0);
    }
    wait_vm_lds<0>();
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    if (any) {
        fetch_hdr(sup0);
        fetch_w(0, wc, sc);
        fetch_x(0, 0, xa);
    }
    int slot = 0;   // part slot of the current step
    for (int it = 0; it < per; it++) {
        const int sup = sup0 + it;
        const bool live = sup < sup1;
        auto step = [&](auto jc) {
            constexpr int j = decltype(jc)::value;
            asm volatile("" ::: "memory");
            wait_vm_lds<Ld::wait(j)>();
            __builtin_amdgcn_s_barrier();
            asm volatile("" ::: "memory");
            if (!live) return;
            const int next = slot == SL - 1 ? 0 : slot + 1;
            uint4 xt[2][3];
            f32x16 d[2];
#pragma unroll
            for (int t = 0; t < TT; t++) {
                if (t > 0) fetch_x(slot, t, xt);
#pragma unroll
                for (int q = 0; q < CH; q++) {
                    chain(t == 0 ? xa : xt, q, d);
                    // the previous chain's scale step: the last chain of the step before, or of this step
                    scale_prev(q > 0 ? t : t > 0 ? t - 1 : TT - 1);
#pragma unroll
                    for (int r = 0; r < 2; r++) {
                        dp[r] = d[r];
                        sp[r] = CH == 2 && q == 1 ? sc[r].sc2 : sc[r].sc;
                    }
                    if (t == 0 && q == 0) {
                        issue_x(sup * 8 + j + D, slot == 0 ? SL - 1 : slot - 1);
                        if constexpr (j % 2 == 1) issue_w(sup, j + 1);
                        if constexpr (j == 0) issue_s(sup);
                    }
                }
            }
            if constexpr (j == 7) {
                add_sums();
                fetch_hdr(sup + 1);
            }
            fetch_w((j + 1) & 7, wc, sc);
            fetch_x(next, 0, xa);
            slot = next;
        };
        step(ic<0>{}); step(ic<1>{}); step(ic<2>{}); step(ic<3>{});
        step(ic<4>{}); step(ic<5>{}); step(ic<6>{}); step(ic<7>{});
    }
    scale_prev(TT - 1);
    wait_vm_lds<0>();   // no load into LDS outlives the ring

    // the K groups' tiles are added in order; group 0 applies the epilogue
    if constexpr (WK > 1) {
        __syncthreads();   // the ring is no longer read
        if (kg > 0) {
#pragma unroll
            for (int r = 0; r < 2; r++)
#pragma unroll
                for (int t = 0; t < TT; t++) R.t[kg - 1][wr][r][t][lane] = acc[r][t];
        }
        __syncthreads();
        if (kg > 0) return;
#pragma unroll
        for (int k = 0; k < WK - 1; k++)
#pragma unroll
            for (int r = 0; r < 2; r++)
#pragma unroll
                for (int t = 0; t < TT; t++) {
                    const f32x16 o = R.t[k][wr][r][t][lane];
#pragma unroll
                    for (int i = 0; i < 16; i++) acc[r][t][i] += o[i];
                }
    }
    if (row0 >= N) return;
#pragma unroll
    for (int t = 0; t < TT; t++)
#pragma unroll
        for (int i = 0; i < 16; i++) {
            // opaque: the addresses of one token at a time, not of all 16 in registers
            int tok = (tt0 + 2 * t) * 16 + 8 * (i >> 2) + 4 * h + (i & 3);
            asm volatile("" : "+v"(tok));
            float y[2];
#pragma unroll
            for (int r = 0; r < 2; r++)
                y[r] = qgemm_epilogue(a, acc[r][t][i], row0 + 32u * r + (uint32_t)li, tok, true);
            if (a.yp_sums) {   // sums of the next GEMM's activations: 32 rows (GELU) or 64 (SwiGLU) per sub-block
                const int nsb_o = (int)(N >> (a.epi == EPI_SILU ? 6 : 5));
                float s[2];
#pragma unroll
                for (int r = 0; r < 2; r++) s[r] = row16_sum(y[r]);
                const bool live = tok < M;
                if (a.epi == EPI_SILU) {   // y is 0 in the odd (up) rows
#pragma unroll
                    for (int r = 0; r < 2; r++) s[r] += swap16_other(s[r]);
                    if (li == 0 && live) xp_sums(a.yp, a.yp_sums, M, nsb_o, tok, (int)(row0 >> 6), s[0], s[1]);
                } else {
#pragma unroll
                    for (int r = 0; r < 2; r++) {
                        const float o = swap16_other(s[r]);
                        if (li == 0 && live && row0 + 32u * r < N)
                            xp_sums(a.yp, a.yp_sums, M, nsb_o, tok, (int)(row0 >> 5) + r, s[r], o);
                    }
                }
            }
        }
}

template <int F, int WR, int WK, int TT, int D>
hipError_t launch_tile(const QgemmArgs &a, hipStream_t s)
{
    TileOrder to{};
    to.R = (uint32_t)((a.w.rows + 64 * WR - 1) / (64 * WR));
    to.T = (uint32_t)((a.M + 32 * TT - 1) / (32 * TT));
    to.G = std::min<uint32_t>(to.T, 8);
    to.chunk = (to.R * to.T + 7) / 8;
    hipLaunchKernelGGL((k_qgemm_tile<F, WR, WK, TT, D>), dim3(8 * to.chunk), dim3(64 * WR * WK), 0, s, a, to);
    return hipGetLastError();
}

}  // namespace

#define SMX_CAT2(a, b) a##b
#define SMX_CAT(a, b) SMX_CAT2(a, b)

// Shapes by the workgroups of 128 rows x 32 tokens (G), measured (microseconds with k_qprep_tokens, Q8_0 /
// Q4_K):
//  - G >= 1024, and where these make exactly one workgroup per CU: four waves of 64 x 64 sharing their parts:
//    11264 x 2048 at 511 tokens 104 / 106 (G 1408; 64 x 32 tiles 112 / 117), 2048 x 5632 at 2048 tokens 175 / 176
//    (199 / 200);
//  - 512 < G < 1024, two waves of 64 x 32, all in one round: 2560 x 2048 at 1024 tokens 64 / 68 (K split in two
//    69 / 72, 64 x 64 tiles 73 / 79), 11264 x 2048 at 352 tokens Q4_K 76 (64 x 64 tiles, 264 workgroups, 94);
//  - fewer, 64 x 32 tiles with K split in two, two workgroups per CU (2048 x 5632 at 1024 tokens 108 / 107;
//    unsplit 133 / 143; 11264 x 2048 at 160 tokens Q4_K 45, unsplit 58), and in four at up to 256 64 x 64 tiles
//    when every part has two super-blocks (2048 x 8192 at 511 tokens 84 / 90; in two 91 / 97).
hipError_t SMX_CAT(launch_qgemm_tile_f, SMX_TILE_FMT)(const QgemmArgs &a, hipStream_t s)
{
    constexpr int F = SMX_TILE_FMT;
    const int64_t G = qgemm_tile_groups(a.w, a.M);
    if (G >= 1024 || ((a.w.rows + 255) / 256) * ((a.M + 63) / 64) == 256) return launch_tile<F, 4, 1, 2, 2>(a, s);
    if (G > 512) return launch_tile<F, 2, 1, 1, 2>(a, s);
    if (qgemm_tiles(a.w, a.M) <= 256 && a.w.cols >= 2048) return launch_tile<F, 2, 4, 1, 2>(a, s);
    return launch_tile<F, 2, 2, 1, 2>(a, s);
}

}  // namespace smx

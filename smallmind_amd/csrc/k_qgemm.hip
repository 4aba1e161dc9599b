// k_qgemm.hip -- quantized GEMM Y[M][N] = X[M][K] . W[N][K]^T on the bf16 matrix cores, for
// several activation rows at once (batched decode of many sessions, short prompts,
// IWeightTensor.MatMul with m > 1; NeuralNet.cs:145-298, MatMulF32Q8.cs:23-80), the preparation of
// its activation parts, and the dispatch between these kernels and the tile kernel for longer
// prompts (k_qgemm_tile.hip, qgemm_tiled).
//
// Exactness.  The MFMA inputs are bf16, the reference computes in fp32.  Both sides are made
// exact:
//   * weights enter as their integer codes, which bf16 represents exactly: 128 + q is built
//     with one and-or per pair of codes (bf16 0x4300 | q; Q8_0 codes go through a conversion),
//     and the block scales are applied to the fp32 result of each 32-element sub-block;
//   * activations enter as three bf16 parts, x = hi + mid + lo (8 + 8 + 8 significant bits),
//     so every product code x part is exact and the MFMA accumulates in fp32.
// A fourth product with an all-ones weight operand gives sum(x) per sub-block, which removes
// the +128 code offset and supplies the min term of Q4_K/Q5_K:
//   y += sc * (C - off * sum x) - m * sum x        (C = sum (128 + q) x over the sub-block).
//
// MFMA v_mfma_f32_16x16x32_bf16: A = activation parts (16 tokens x 32 k), B = weight codes
// (32 k x 16 weight rows), D[token][row].  Lane l supplies token / weight row l % 16 and the
// 8 k-values of group l / 16; D lane l holds tokens 4*(l/16)+0..3 of weight row l % 16.  The
// order of the 8 k-values inside a group is free as long as A and B agree; both use
// element order {0,4,1,5,2,6,3,7}, the order in which ((v >> 4p) & 0x000F000F) lays out two
// nibble codes per 32-bit pair.
//
// Work decomposition: a workgroup is 4 waves that split the sub-blocks of K between them
// (wave w takes sub-blocks w, w+4, ...) for RT row tiles of 16 weight rows and TT token tiles
// of 16 tokens; the four partial tiles are summed in LDS in a fixed order.
//
// Activation parts come from k_qprep: Xp[tt][s][p][g][t][8 bf16] (1 KB per (token tile,
// sub-block, part), lane l reads 16 bytes at l*16).
#include <algorithm>
#include <type_traits>

#include "smx_qgemm.h"

namespace smx {

hipError_t launch_qgemm_tile(const QgemmArgs &a, hipStream_t s);

namespace {

template <int F, int RT, int TT, int NW, int SB>
__global__ __launch_bounds__(64 * NW) void k_qgemm(QgemmArgs a)
{
    using Q = QW<F>;
    const WView &w = a.w;
    const uint8_t *__restrict__ xp = a.xp;
    const int M = a.M;
    __shared__ f32x4 s_part[NW - 1][RT * TT][64];
    const int wv = wave_id();
    const int lane = lane_id();
    const int g = lane >> 4, li = lane & 15;
    const uint32_t lane16 = (uint32_t)lane * 16u;
    const uint32_t N = (uint32_t)w.rows;
    const int nsb = (int)(w.cols >> 5);
    const uint32_t row_base = blockIdx.x * (16 * RT);
    const int tt0 = blockIdx.y * TT;
    const int ntt = (M + 15) >> 4;

    f32x4 acc[RT][TT];
#pragma unroll
    for (int r = 0; r < RT; r++)
#pragma unroll
        for (int t = 0; t < TT; t++) acc[r][t] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};

    // weight rows of this lane (B operand column l % 16), clamped to the matrix
    uint32_t wrow[RT];
#pragma unroll
    for (int r = 0; r < RT; r++) {
        const uint32_t rr = row_base + 16 * r + li;
        wrow[r] = rr < N ? rr : N - 1;
    }
    const uint4 ones_a = Q::kHalves ? (g < 2 ? make_uint4(kOnes, kOnes, kOnes, kOnes) : kZero4)
                                    : make_uint4(kOnes, kOnes, kOnes, kOnes);
    const uint4 ones_b = g >= 2 ? make_uint4(kOnes, kOnes, kOnes, kOnes) : kZero4;

    // Wave wv takes sub-blocks wv, wv + NW, ...; SB of them at a time, all of whose loads (raw
    // weight words and activation parts) are issued before any is consumed.
    for (int s0 = wv; s0 < nsb; s0 += NW * SB) {
        RawQ raw[SB][RT];
        uint4 xa[SB][TT][3];
#pragma unroll
        for (int u = 0; u < SB; u++) {
            const int s = s0 + u * NW < nsb ? s0 + u * NW : nsb - 1;
#pragma unroll
            for (int t = 0; t < TT; t++) {
                const int tt = tt0 + t < ntt ? tt0 + t : ntt - 1;
#pragma unroll
                for (int p = 0; p < 3; p++)
                    xa[u][t][p] = ld_part(xp, tt, nsb, s, p, lane16);
            }
#pragma unroll
            for (int r = 0; r < RT; r++) raw[u][r] = Q::load(w, wrow[r], s, g);
        }
        // keep the whole batch of loads ahead of the first use
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int u = 0; u < SB; u++) {
            const int s = s0 + u * NW;
            const float ok = s < nsb ? 1.0f : 0.0f;   // past the end: clamped duplicate, adds 0
            uint4 wc[RT];
            Scl sc[RT];
#pragma unroll
            for (int r = 0; r < RT; r++) {
                wc[r] = Q::codes(raw[u][r], g);
                sc[r] = Q::scale(raw[u][r], s);
            }
            // sum(x) per token (and per half for Q6_K): the same for every weight row
#pragma unroll
            for (int t = 0; t < TT; t++) {
                f32x4 sa = {0.0f, 0.0f, 0.0f, 0.0f}, sb = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
                for (int p = 0; p < 3; p++) {
                    sa = mfma(xa[u][t][p], ones_a, sa);
                    if constexpr (Q::kHalves) sb = mfma(xa[u][t][p], ones_b, sb);
                }
#pragma unroll
                for (int r = 0; r < RT; r++) {
                    if constexpr (Q::kHalves) {
                        const uint4 ca = g < 2 ? wc[r] : kZero4, cb = g >= 2 ? wc[r] : kZero4;
                        f32x4 da = {0.0f, 0.0f, 0.0f, 0.0f}, db = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
                        for (int p = 0; p < 3; p++) {
                            da = mfma(xa[u][t][p], ca, da);
                            db = mfma(xa[u][t][p], cb, db);
                        }
#pragma unroll
                        for (int i = 0; i < 4; i++)
                            acc[r][t][i] = accumulate2(acc[r][t][i], ok * sc[r].sc, ok * sc[r].sc2, da[i], db[i], sa[i], sb[i],
                                                       Q::kOff);
                    } else {
                        f32x4 dc = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
                        for (int p = 0; p < 3; p++) dc = mfma(xa[u][t][p], wc[r], dc);
                        const float c = ok * sc[r].sc, cs = ok * (sc[r].sc * Q::kOff + sc[r].m);
#pragma unroll
                        for (int i = 0; i < 4; i++) acc[r][t][i] = accumulate1(acc[r][t][i], c, cs, dc[i], sa[i]);
                    }
                }
            }
        }
    }

    // sum the NW waves' partial tiles in a fixed order; wave 0 stores
    if (wv > 0) {
#pragma unroll
        for (int r = 0; r < RT; r++)
#pragma unroll
            for (int t = 0; t < TT; t++) s_part[wv - 1][r * TT + t][lane] = acc[r][t];
    }
    __syncthreads();
    if (wv != 0) return;
#pragma unroll
    for (int r = 0; r < RT; r++)
#pragma unroll
        for (int t = 0; t < TT; t++) {
            f32x4 v = acc[r][t];
#pragma unroll
            for (int k = 0; k < NW - 1; k++) {
                const f32x4 o = s_part[k][r * TT + t][lane];
#pragma unroll
                for (int i = 0; i < 4; i++) v[i] += o[i];
            }
            const uint32_t row = row_base + 16 * r + li;
#pragma unroll
            for (int i = 0; i < 4; i++) qgemm_epilogue(a, v[i], row, (tt0 + t) * 16 + 4 * g + i, true);
        }
}

// ---- unquantized weights (F16 / F32) --------------------------------------------------------
// The FP32 Linear on F16 / F32 matrices (NeuralNet.cs:233-298, F32WeightTensor.cs:9-60).  The
// weights have no block scale to factor out, so they enter as bf16 parts of their own, exactly:
// an fp16 value (11 significant bits) is hi + lo, an fp32 value hi + mid + lo (8 + 8 + 8), each
// part a round-to-nearest-even bf16 of the remainder.  Every product of a weight part and an
// activation part is exact in fp32; the MFMA sums them (6 products per element for F16, 9 for
// F32).  Same operand layout, work split and epilogue as k_qgemm; no sum(x) term.
template <int F> struct DW {
    static constexpr int kParts = F == FMT_F16 ? 2 : 3;
    // the 8 weights of (row, sub-block s, k-group g) as fp32, element order 0..7
    __device__ __forceinline__ static void load(const WView &w, uint32_t row, int s, int g, float *v)
    {
        const uint8_t *p = w.q + ((size_t)row * (uint32_t)w.nb + (uint32_t)s) * fmt_main_bytes(F);
        if constexpr (F == FMT_F16) {
            const uint4 h = *(const uint4 *)(p + 16 * g);
            const uint32_t u[4] = {h.x, h.y, h.z, h.w};
#pragma unroll
            for (int i = 0; i < 4; i++) {
                v[2 * i] = h2f(u[i] & 0xFFFFu);
                v[2 * i + 1] = h2f(u[i] >> 16);
            }
        } else {
            const float4 a = *(const float4 *)(p + 32 * g), b = *(const float4 *)(p + 32 * g + 16);
            v[0] = a.x; v[1] = a.y; v[2] = a.z; v[3] = a.w; v[4] = b.x; v[5] = b.y; v[6] = b.z; v[7] = b.w;
        }
    }
    // bf16 parts in the operand order (pair q = element q, element q + 4)
    __device__ __forceinline__ static void parts(const float *v, uint4 *o)
    {
        uint32_t pt[3][8];
#pragma unroll
        for (int k = 0; k < 8; k++) {
            const uint32_t h = bf16_rne(v[k]);
            const float r1 = v[k] - __uint_as_float(h << 16);
            const uint32_t m = bf16_rne(r1);
            pt[0][k] = h;
            pt[1][k] = m;
            if constexpr (kParts == 3) pt[2][k] = bf16_rne(r1 - __uint_as_float(m << 16));
        }
#pragma unroll
        for (int p = 0; p < kParts; p++)
            o[p] = make_uint4(pt[p][0] | (pt[p][4] << 16), pt[p][1] | (pt[p][5] << 16), pt[p][2] | (pt[p][6] << 16),
                              pt[p][3] | (pt[p][7] << 16));
    }
};

template <int F, int RT, int TT, int NW, int SB>
__global__ __launch_bounds__(64 * NW) void k_dgemm(QgemmArgs a)
{
    using D = DW<F>;
    constexpr int NP = D::kParts;
    const WView &w = a.w;
    const uint8_t *__restrict__ xp = a.xp;
    const int M = a.M;
    __shared__ f32x4 s_part[NW - 1][RT * TT][64];
    const int wv = wave_id();
    const int lane = lane_id();
    const int g = lane >> 4, li = lane & 15;
    const uint32_t lane16 = (uint32_t)lane * 16u;
    const uint32_t N = (uint32_t)w.rows;
    const int nsb = (int)(w.cols >> 5);
    const uint32_t row_base = blockIdx.x * (16 * RT);
    const int tt0 = blockIdx.y * TT;
    const int ntt = (M + 15) >> 4;

    f32x4 acc[RT][TT];
#pragma unroll
    for (int r = 0; r < RT; r++)
#pragma unroll
        for (int t = 0; t < TT; t++) acc[r][t] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
    uint32_t wrow[RT];
#pragma unroll
    for (int r = 0; r < RT; r++) {
        const uint32_t rr = row_base + 16 * r + li;
        wrow[r] = rr < N ? rr : N - 1;
    }

    for (int s0 = wv; s0 < nsb; s0 += NW * SB) {
        float wf[SB][RT][8];
        uint4 xa[SB][TT][3];
#pragma unroll
        for (int u = 0; u < SB; u++) {
            const int s = s0 + u * NW < nsb ? s0 + u * NW : nsb - 1;
#pragma unroll
            for (int t = 0; t < TT; t++) {
                const int tt = tt0 + t < ntt ? tt0 + t : ntt - 1;
#pragma unroll
                for (int p = 0; p < 3; p++) xa[u][t][p] = ld_part(xp, tt, nsb, s, p, lane16);
            }
#pragma unroll
            for (int r = 0; r < RT; r++) D::load(w, wrow[r], s, g, wf[u][r]);
        }
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int u = 0; u < SB; u++) {
            if (s0 + u * NW >= nsb) break;   // wave-uniform: past the end of K
#pragma unroll
            for (int r = 0; r < RT; r++) {
                uint4 wp[NP];
                D::parts(wf[u][r], wp);
#pragma unroll
                for (int t = 0; t < TT; t++)
#pragma unroll
                    for (int q = 0; q < NP; q++)
#pragma unroll
                        for (int p = 0; p < 3; p++) acc[r][t] = mfma(xa[u][t][p], wp[q], acc[r][t]);
            }
        }
    }

    if (wv > 0) {
#pragma unroll
        for (int r = 0; r < RT; r++)
#pragma unroll
            for (int t = 0; t < TT; t++) s_part[wv - 1][r * TT + t][lane] = acc[r][t];
    }
    __syncthreads();
    if (wv != 0) return;
#pragma unroll
    for (int r = 0; r < RT; r++)
#pragma unroll
        for (int t = 0; t < TT; t++) {
            f32x4 v = acc[r][t];
#pragma unroll
            for (int k = 0; k < NW - 1; k++) {
                const f32x4 o = s_part[k][r * TT + t][lane];
#pragma unroll
                for (int i = 0; i < 4; i++) v[i] += o[i];
            }
            const uint32_t row = row_base + 16 * r + li;
#pragma unroll
            for (int i = 0; i < 4; i++) qgemm_epilogue(a, v[i], row, (tt0 + t) * 16 + 4 * g + i, true);
        }
}

// ---- LDS-staged variant --------------------------------------------------------------------
// The lane-per-(row, k-group) operand layout makes direct weight loads touch 16 rows (16 cache
// lines) per instruction for 4 useful bytes each.  Here every wave copies its weight tile --
// 16*RT rows x one 256-element super-block -- into its own LDS region with coalesced 16-byte
// loads (the next super-block's copy in flight while the current one is multiplied), and reads
// the operand dwords from LDS.  RT row tiles per wave share each activation-part load.
// Waves of a workgroup take contiguous super-block ranges of K.
// kBytes: main-stream bytes per row and super-block; kDW: dwords of the d stream per row and
// super-block (8 fp16 scales, one fp16 scale, or 8 fp32 scales).
template <int F> struct Stage;
template <> struct Stage<FMT_Q4_0> { static constexpr int kBytes = 128, kDW = 4; };
template <> struct Stage<FMT_Q8_0> { static constexpr int kBytes = 256, kDW = 4; };
template <> struct Stage<FMT_Q4_K> { static constexpr int kBytes = 144, kDW = 0; };
template <> struct Stage<FMT_Q5_K> { static constexpr int kBytes = 176, kDW = 0; };
template <> struct Stage<FMT_Q6_K> { static constexpr int kBytes = 208, kDW = 1; };
template <> struct Stage<FMT_SQ4> { static constexpr int kBytes = 128, kDW = 8; };
template <> struct Stage<FMT_SQ8> { static constexpr int kBytes = 256, kDW = 8; };

__device__ __forceinline__ uint32_t lds_u32(const uint8_t *p) { return *(const uint32_t *)p; }

// Raw operand words of (tile row, sub-block j of the staged super-block, k-group g) from LDS:
// `row` points at the row's staged main bytes, `dr` at its staged fp16 scales (packed in
// dwords).  Staged data is written and read as 32-bit words only, so the compiler cannot
// treat a narrower read as independent of the staging stores and move it above them.
template <int F>
__device__ __forceinline__ RawQ stage_raw(const uint8_t *row, const uint32_t *dr, int j, int g)
{
    RawQ r{};
    if constexpr (F == FMT_Q4_0) {
        r.v = lds_u32(row + 16 * j + 4 * g);
        r.d = (dr[j >> 1] >> (16 * (j & 1))) & 0xFFFFu;
    } else if constexpr (F == FMT_SQ4) {
        r.v = lds_u32(row + 16 * j + 4 * g);
        r.d = dr[j];
    } else if constexpr (F == FMT_SQ8) {
        r.v = lds_u32(row + 32 * j + 8 * g);
        r.v2 = lds_u32(row + 32 * j + 8 * g + 4);
        r.d = dr[j];
    } else if constexpr (F == FMT_Q8_0) {
        r.v = lds_u32(row + 32 * j + 8 * g);
        r.v2 = lds_u32(row + 32 * j + 8 * g + 4);
        r.d = (dr[j >> 1] >> (16 * (j & 1))) & 0xFFFFu;
    } else if constexpr (F == FMT_Q4_K) {
        r.h = make_uint4(lds_u32(row), lds_u32(row + 4), lds_u32(row + 8), lds_u32(row + 12));
        r.v = lds_u32(row + 16 + 16 * j + 4 * g);
    } else if constexpr (F == FMT_Q5_K) {
        r.h = make_uint4(lds_u32(row), lds_u32(row + 4), lds_u32(row + 8), lds_u32(row + 12));
        r.v = lds_u32(row + 48 + 16 * j + 4 * g);
        r.H = lds_u32(row + 16 + 4 * j);
    } else {
        r.v = lds_u32(row + 16 * j + 4 * g);
        r.H = lds_u32(row + 128 + 8 * j);
        r.H2 = lds_u32(row + 128 + 8 * j + 4);
        const uint32_t scw = (lds_u32(row + 192 + 4 * (j >> 1)) >> (16 * (j & 1))) & 0xFFFFu;
        r.d = (dr[0] & 0xFFFFu) | (scw << 16);
    }
    return r;
}

// TS > 1 (one token tile only): the tile's 16 tokens are split over TS workgroups of 16 / TS
// tokens each (grid y).  Each workgroup still multiplies whole 16 x 16 MFMA tiles, but it loads
// the activation parts of its own tokens only (the other token lanes repeat them) and stores
// only their outputs: the parts of the whole K, which every workgroup of a row tile reads, are
// most of what a one-token-tile workgroup moves into its CU, and the split also spreads a
// matrix of few row tiles over more CUs.  No partial sums cross workgroups.
template <int F, int RT, int TT, int NW, int TS = 1>
__global__ __launch_bounds__(64 * NW) void k_qgemm_st(QgemmArgs a)
{
    static_assert(TS == 1 || (TT == 1 && (TS == 2 || TS == 4)), "token split of one token tile into 8 or 4");
    using Q = QW<F>;
    using G = Stage<F>;
    constexpr int R16 = 16 * RT;
    constexpr int RS = G::kBytes + 4;                       // row stride: dword pad, odd in dwords
    constexpr int NPC = (R16 * G::kBytes / 16 + 63) / 64;   // 16-byte pieces per lane
    // dword accesses below: the byte array must be dword (here 16-byte) aligned
    __shared__ __align__(16) uint8_t s_w[NW][R16 * RS];
    __shared__ __align__(16) uint32_t s_d[NW][R16][G::kDW > 0 ? G::kDW : 1];
    __shared__ f32x4 s_part[NW - 1][RT * TT][64];
    const WView &w = a.w;
    const uint8_t *__restrict__ xp = a.xp;
    const int M = a.M;
    const int wv = wave_id();
    const int lane = lane_id();
    const int g = lane >> 4, li = lane & 15;
    const uint32_t lane16 = (uint32_t)lane * 16u;
    const uint32_t N = (uint32_t)w.rows;
    const int nsb = (int)(w.cols >> 5), nsup = nsb >> 3;
    const uint32_t bx = blockIdx.x, by = blockIdx.y;
    const uint32_t row_base = bx * R16;
    // token split: this workgroup's tokens are tlo .. tlo + TW - 1 of the single token tile
    constexpr int TW = 16 / TS;
    const int tlo = TS > 1 ? (int)by * TW : 0;
    const int tt0 = TS > 1 ? 0 : (int)by * TT;
    const int ntt = (M + 15) >> 4;
    // lanes whose results are this workgroup's tokens (tokens 4g .. 4g + 3; TW is a multiple of
    // 4).  A lane supplies token li's parts to the MFMA; lanes of the other tokens read those of
    // token tlo + li % TW instead, so the loads touch only this workgroup's tokens' lines and
    // need no mask or select (the duplicated tokens' results are not stored).
    const bool tlive = TS == 1 || (uint32_t)(4 * g - tlo) < (uint32_t)TW;
    const uint32_t xl16 = TS == 1 ? lane16 : (uint32_t)(16 * g + tlo + (li & (TW - 1))) * 16u;
    const uint32_t row_bytes = (uint32_t)nsup * G::kBytes;
    // contiguous super-block range of this wave
    const int per = (nsup + NW - 1) / NW;
    const int sup0 = wv * per, sup1 = sup0 + per < nsup ? sup0 + per : nsup;

    f32x4 acc[RT][TT];
#pragma unroll
    for (int r = 0; r < RT; r++)
#pragma unroll
        for (int t = 0; t < TT; t++) acc[r][t] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
    const uint4 ones_a = Q::kHalves ? (g < 2 ? make_uint4(kOnes, kOnes, kOnes, kOnes) : kZero4)
                                    : make_uint4(kOnes, kOnes, kOnes, kOnes);
    const uint4 ones_b = g >= 2 ? make_uint4(kOnes, kOnes, kOnes, kOnes) : kZero4;

    // Folded RMSNorm (one token tile): the tile sums of x^2 of wave wv's tokens wv + NW*j are
    // requested here and reduced after the main loop.
    constexpr int RJ = TT == 1 ? (16 + NW - 1) / NW : 1, RP = 4;   // tokens per wave, sums per lane
    __shared__ float s_r[16];
    float rl[RJ][RP];
    const bool fold = TT == 1 && a.rss != nullptr;
    if (fold) {
#pragma unroll
        for (int j = 0; j < RJ; j++) {
            const int tk = min(tt0 * 16 + wv + NW * j, M - 1);
#pragma unroll
            for (int q = 0; q < RP; q++) {
                const int p = lane + 64 * q;
                rl[j][q] = p < a.rss_n ? a.rss[(int64_t)p * M + tk] : 0.0f;
            }
        }
    }

    // EPI_RESID with one 16 x 16 tile per wave: wave 0's residual values (and the next norm's
    // gamma) are requested at entry, so the epilogue waits for no load.  EPI_QKV likewise: the
    // positions of wave 0's tokens at entry, their RoPE factors and cache bases (which depend
    // on the positions) right after the main loop, ahead of the cross-wave reduction.
    constexpr bool PRE = TT == 1 && RT == 1;
    const bool pre = PRE && (a.epi == EPI_RESID || a.epi == EPI_QKV);
    const bool preq = PRE && a.epi == EPI_QKV;
    float pres[4] = {0.0f, 0.0f, 0.0f, 0.0f}, pg = 0.0f;
    QkvPre qp[4] = {};
    if (pre && wv == 0 && tlive) {
        const uint32_t rc = min(row_base + (uint32_t)li, N - 1);
        if (preq) {
#pragma unroll
            for (int i = 0; i < 4; i++) qp[i].pos = a.tok_pos[min(tt0 * 16 + 4 * g + i, M - 1)];
        } else {
#pragma unroll
            for (int i = 0; i < 4; i++) pres[i] = a.y[(int64_t)min(tt0 * 16 + 4 * g + i, M - 1) * a.y_stride + rc];
            if (a.np) pg = a.ngamma[rc];
        }
    }

    // staging loads of one super-block: piece p -> (row p / (kBytes/16), 16-byte column)
    uint4 wp[NPC];
    uint4 dp = kZero4, dp2 = kZero4;
    auto issue = [&](int sup) {
#pragma unroll
        for (int k = 0; k < NPC; k++) {
            const int p = lane + 64 * k;
            const int row = p / (G::kBytes / 16), col = p % (G::kBytes / 16);
            uint32_t gr = row_base + (uint32_t)row;
            gr = gr < N ? gr : N - 1;
            wp[k] = p < R16 * G::kBytes / 16
                        ? *(const uint4 *)(w.q + gr * row_bytes + (uint32_t)sup * G::kBytes + 16u * col)
                        : kZero4;
        }
        if constexpr (G::kDW == 4) {
            if (lane < R16) {
                uint32_t gr = row_base + (uint32_t)lane;
                gr = gr < N ? gr : N - 1;
                dp = *(const uint4 *)(w.d + (gr * (uint32_t)nsb + (uint32_t)sup * 8));
            }
        } else if constexpr (G::kDW == 8) {
            if (lane < R16) {
                uint32_t gr = row_base + (uint32_t)lane;
                gr = gr < N ? gr : N - 1;
                const uint4 *dq = (const uint4 *)((const uint32_t *)w.d + (gr * (uint32_t)nsb + (uint32_t)sup * 8));
                dp = dq[0];
                dp2 = dq[1];
            }
        } else if constexpr (G::kDW == 1) {
            if (lane < R16) {
                uint32_t gr = row_base + (uint32_t)lane;
                gr = gr < N ? gr : N - 1;
                dp.x = w.d[gr * (uint32_t)nsup + (uint32_t)sup];
            }
        }
    };
    auto stage = [&]() {
        // the previous super-block's reads of the tile stay above these stores
        asm volatile("" ::: "memory");
        uint8_t *dst = s_w[wv];
#pragma unroll
        for (int k = 0; k < NPC; k++) {
            const int p = lane + 64 * k;
            if (p < R16 * G::kBytes / 16) {
                const int row = p / (G::kBytes / 16), col = p % (G::kBytes / 16);
                uint32_t *o = (uint32_t *)(dst + row * RS + 16 * col);
                o[0] = wp[k].x;
                o[1] = wp[k].y;
                o[2] = wp[k].z;
                o[3] = wp[k].w;
            }
        }
        if constexpr (G::kDW == 4 || G::kDW == 8) {
            if (lane < R16) {
                uint32_t *o = s_d[wv][lane];
                o[0] = dp.x; o[1] = dp.y; o[2] = dp.z; o[3] = dp.w;
                if constexpr (G::kDW == 8) { o[4] = dp2.x; o[5] = dp2.y; o[6] = dp2.z; o[7] = dp2.w; }
            }
        } else if constexpr (G::kDW == 1) {
            if (lane < R16) s_d[wv][lane][0] = dp.x;
        }
        // keep every read of the staged tile below these stores
        asm volatile("" ::: "memory");
    };

    if (sup0 < sup1) issue(sup0);
    for (int sup = sup0; sup < sup1; sup++) {
        stage();                               // this wave's LDS region only: in-order LDS ops
        if (sup + 1 < sup1) issue(sup + 1);    // next super-block in flight
        // XU sub-blocks of activation parts in flight at once (fewer with more token tiles, and
        // two for the 16-wave SMQ Q8 tile, whose two staged scale words per sub-block would
        // otherwise push it past the 128 registers of a 1024-thread workgroup)
        constexpr int XU = TT == 1 ? (F == FMT_SQ8 && NW == 16 ? 2 : 4) : 1;
#pragma unroll
        for (int h = 0; h < 8 / XU; h++) {
            uint4 xa[XU][TT][3];
#pragma unroll
            for (int u = 0; u < XU; u++) {
                const int s = sup * 8 + XU * h + u;
#pragma unroll
                for (int t = 0; t < TT; t++) {
                    const int tt = tt0 + t < ntt ? tt0 + t : ntt - 1;
#pragma unroll
                    for (int p = 0; p < 3; p++)
                        xa[u][t][p] = ld_part(xp, tt, nsb, s, p, xl16);
                }
            }
#pragma unroll
            for (int u = 0; u < XU; u++) {
                const int j = XU * h + u;
                uint4 wc[RT];
                Scl sc[RT];
#pragma unroll
                for (int r = 0; r < RT; r++) {
                    const int row = 16 * r + li;
                    const RawQ raw = stage_raw<F>(s_w[wv] + row * RS, s_d[wv][row], j, g);
                    wc[r] = Q::codes(raw, g);
                    sc[r] = Q::scale(raw, j);
                }
#pragma unroll
                for (int t = 0; t < TT; t++) {
                    f32x4 sa = {0.0f, 0.0f, 0.0f, 0.0f}, sb = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
                    for (int p = 0; p < 3; p++) {
                        sa = mfma(xa[u][t][p], ones_a, sa);
                        if constexpr (Q::kHalves) sb = mfma(xa[u][t][p], ones_b, sb);
                    }
#pragma unroll
                    for (int r = 0; r < RT; r++) {
                        if constexpr (Q::kHalves) {
                            const uint4 ca = g < 2 ? wc[r] : kZero4, cb = g >= 2 ? wc[r] : kZero4;
                            f32x4 da = {0.0f, 0.0f, 0.0f, 0.0f}, db = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
                            for (int p = 0; p < 3; p++) {
                                da = mfma(xa[u][t][p], ca, da);
                                db = mfma(xa[u][t][p], cb, db);
                            }
#pragma unroll
                            for (int i = 0; i < 4; i++)
                                acc[r][t][i] = accumulate2(acc[r][t][i], sc[r].sc, sc[r].sc2, da[i], db[i], sa[i], sb[i],
                                                           Q::kOff);
                        } else {
                            f32x4 dc = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
                            for (int p = 0; p < 3; p++) dc = mfma(xa[u][t][p], wc[r], dc);
                            const float c = sc[r].sc, cs = sc[r].sc * Q::kOff + sc[r].m;
#pragma unroll
                            for (int i = 0; i < 4; i++) acc[r][t][i] = accumulate1(acc[r][t][i], c, cs, dc[i], sa[i]);
                        }
                    }
                }
            }
        }
    }

    if (preq && wv == 0 && tlive) {
        const int d = a.d_model, kv = a.kv_dim, hd = a.head_dim, half = hd / 2;
        const int r = (int)min(row_base + (uint32_t)li, N - 1);
        const int pair = ((r < d ? r : r - d) % hd) / 2;
        const bool rot = a.use_rope && r < d + kv && !(r & 1);
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const int tk = min(tt0 * 16 + 4 * g + i, M - 1);
            qp[i].c = rot ? a.rope_cos[(int64_t)qp[i].pos * half + pair] : 0.0f;
            qp[i].sn = rot ? a.rope_sin[(int64_t)qp[i].pos * half + pair] : 0.0f;
            qp[i].cache = r < d ? nullptr : (r < d + kv ? a.kc_tok[tk] : a.vc_tok[tk]);
        }
    }
    if (fold) {   // r = 1 / sqrt(sum x^2 / K + eps) (RMSNormOps.cs:114)
#pragma unroll
        for (int j = 0; j < RJ; j++) {
            float t = rl[j][0];
#pragma unroll
            for (int q = 1; q < RP; q++) t += rl[j][q];
            t = wave_sum_uniform(t);
            if (lane == 0 && wv + NW * j < 16) s_r[wv + NW * j] = 1.0f / sqrtf(t / (float)w.cols + a.r_eps);
        }
    }
    // sum the NW waves' partial tiles in a fixed order; wave 0 applies the epilogue
    if (wv > 0) {
#pragma unroll
        for (int r = 0; r < RT; r++)
#pragma unroll
            for (int t = 0; t < TT; t++) s_part[wv - 1][r * TT + t][lane] = acc[r][t];
    }
    __syncthreads();
    if (wv != 0) return;
    float rs[4] = {1.0f, 1.0f, 1.0f, 1.0f};
    if (fold) {
#pragma unroll
        for (int i = 0; i < 4; i++) rs[i] = s_r[4 * g + i];
    }
    const bool emit = TT == 1 && a.np != nullptr;   // producer of a folded norm
#pragma unroll
    for (int r = 0; r < RT; r++) {
        float sq[TT][4];
#pragma unroll
        for (int t = 0; t < TT; t++) {
            f32x4 v = acc[r][t];
#pragma unroll
            for (int k = 0; k < NW - 1; k++) {
                const f32x4 o = s_part[k][r * TT + t][lane];
#pragma unroll
                for (int i = 0; i < 4; i++) v[i] += o[i];
            }
            const uint32_t row = row_base + 16 * r + li;
#pragma unroll
            for (int i = 0; i < 4; i++) {
                const float xn = qgemm_epilogue(a, v[i] * rs[i], row, (tt0 + t) * 16 + 4 * g + i, tlive, pre, pres[i],
                                                pg, qp[i]);
                sq[t][i] = xn * xn;
            }
        }
        if (emit) {   // x^2 summed over the tile's 16 rows (the 16 lanes of a row of lanes)
#pragma unroll
            for (int i = 0; i < 4; i++) {
                const float t = row16_sum(sq[0][i]);
                const int tok = tt0 * 16 + 4 * g + i;
                if (li == 0 && tok < M && tlive) a.nss[(int64_t)(row_base / 16 + r) * M + tok] = t;
            }
        }
    }
}

// ---- row-split variant for one token tile ---------------------------------------------------
// Up to 16 tokens, the K-split workgroups above each read the activation parts of the whole K
// for their own 16-32 rows (6 bytes per token and k against 0.69 bytes per Q5_K weight), and
// a wave can only hold a few sub-blocks of them in registers, so its part loads queue behind
// its weight loads.  Here a workgroup of NW = NR * NKH waves owns NR row tiles (16 rows each)
// and the whole K: wave (r, h) multiplies row tile r by the sub-blocks h * 8 / NKH ... of every
// super-block.  Super-block by super-block, a slot of an NS-slot LDS ring receives the
// super-block's activation parts (24 KB, read by every wave) and its NR * 16 rows of weights,
// both loaded straight into LDS (global_load_lds_dwordx4, no registers) NS - 1 super-blocks
// ahead of use; one barrier per super-block publishes a slot.  Each wave issues the same
// number of loads per super-block (every one with at least one active lane), so the wait for
// a slot is a fixed vector-memory count.  The loads into LDS are issued by inline assembly:
// through the builtin, the compiler cannot tell the slots apart in this kernel and waits for
// every load into LDS in flight before each LDS read, which leaves no load in flight across a
// super-block's multiplications.  The explicit wait before each barrier is what orders a
// slot's reads after its loads.
template <int F, int NR> struct RsSlot {
    uint4 xp[24][64];                  // [sub-block][part] x (64 lanes x 16 bytes)
    uint4 w[NR * Stage<F>::kBytes];    // NR * 16 rows x kBytes, row-major, in 16-byte pieces
};


template <int N> using ic = std::integral_constant<int, N>;

template <int F, int NR, int NKH, int NS>
__global__ __launch_bounds__(64 * NR * NKH) void k_qgemm_rs(QgemmArgs a)
{
    using Q = QW<F>;
    constexpr int kB = Stage<F>::kBytes;
    constexpr int NW = NR * NKH, JP = 8 / NKH;
    constexpr int WP = NR * kB;            // 16-byte weight pieces per super-block
    constexpr int PPW = WP / NW;           // ... per wave
    constexpr int WI = (PPW + 63) / 64;    // weight loads per wave and super-block
    constexpr int NPW = 24 / NW;           // part loads per wave and super-block
    constexpr int L = WI + NPW;            // vector-memory instructions per wave and super-block
    static_assert(Stage<F>::kDW == 0, "weights without a separate scale stream");
    static_assert(WP % NW == 0 && 24 % NW == 0 && 8 % NKH == 0 && NS >= 2 && NS <= 4, "work split");
    static_assert((NS - 2) * L < 64, "vmcnt range");
    __shared__ RsSlot<F, NR> slot[NS];
    __shared__ f32x4 s_part[NKH > 1 ? NKH - 1 : 1][NR][64];
    __shared__ float s_r[16];
    const WView &w = a.w;
    const int M = a.M;
    const int wv = wave_id();
    const int r = wv % NR, h = wv / NR;
    const int lane = lane_id();
    const int g = lane >> 4, li = lane & 15;
    const uint32_t N = (uint32_t)w.rows;
    const int nsup = (int)(w.cols >> 8);
    const uint32_t row_base = blockIdx.x * (16u * NR);
    const uint32_t row_bytes = (uint32_t)nsup * kB;
    const uint32_t my_row = row_base + 16u * r + (uint32_t)li;

    // loads of super-block sup into a slot: this wave's parts (instructions wv * NPW ...) and
    // its share of the weight pieces (wv * PPW ...)
    auto issue = [&](int sup, auto &S) {
        const uint8_t *xs = a.xp + (size_t)sup * (24u * 1024u) + (uint32_t)lane * 16u;
#pragma unroll
        for (int k = 0; k < NPW; k++) {
            const int c = wv * NPW + k;
            lds_dma16(xs + c * 1024, &S.xp[c][0]);
        }
#pragma unroll
        for (int k = 0; k < WI; k++) {
            const int q = wv * PPW + 64 * k + lane;
            if (64 * k + lane < PPW) {
                const int rw = q / (kB / 16), col = q % (kB / 16);
                const uint32_t gr = min(row_base + (uint32_t)rw, N - 1);
                lds_dma16(w.q + gr * row_bytes + (uint32_t)sup * kB + 16u * col, &S.w[wv * PPW + 64 * k]);
            }
        }
    };
    // the first super-blocks' loads go out before anything else
#pragma unroll
    for (int i = 0; i < NS - 1; i++)
        if (i < nsup) issue(i, slot[i]);

    // Folded RMSNorm: the tile sums of x^2 of wave wv's tokens wv + NW*j, requested here and
    // reduced after the main loop.
    constexpr int RJ = (16 + NW - 1) / NW, RP = 4;
    float rl[RJ][RP];
    const bool fold = a.rss != nullptr;
    if (fold) {
#pragma unroll
        for (int j = 0; j < RJ; j++) {
            const int tk = min(wv + NW * j, M - 1);
#pragma unroll
            for (int q = 0; q < RP; q++) {
                const int p = lane + 64 * q;
                rl[j][q] = p < a.rss_n ? a.rss[(int64_t)p * M + tk] : 0.0f;
            }
        }
    }
    // The epilogue waves' residual values and next-norm gamma (EPI_RESID), or their tokens'
    // positions (EPI_QKV), requested at entry so that the epilogue's stores wait for no load.
    const bool pre = a.epi == EPI_RESID || a.epi == EPI_QKV;
    const bool preq = a.epi == EPI_QKV;
    float pres[4] = {0.0f, 0.0f, 0.0f, 0.0f}, pg = 0.0f;
    QkvPre qp[4] = {};
    if (pre && h == 0) {
        const uint32_t rc = min(my_row, N - 1);
        if (preq) {
#pragma unroll
            for (int i = 0; i < 4; i++) qp[i].pos = a.tok_pos[min(4 * g + i, M - 1)];
        } else {
#pragma unroll
            for (int i = 0; i < 4; i++) pres[i] = a.y[(int64_t)min(4 * g + i, M - 1) * a.y_stride + rc];
            if (a.np) pg = a.ngamma[rc];
        }
    }

    // Publishes the slot of super-block i: this wave's loads of it have landed (the loads of
    // the n_after later super-blocks already issued may still be in flight), then every wave's.
    // The wave's LDS reads of the previous super-block's slot have completed too, so the loads
    // that go into that slot after the barrier cannot overtake them.
    auto sync = [&](int n_after) {
        asm volatile("" ::: "memory");
        if (NS > 3 && n_after >= 2) wait_vm_lds<(NS > 3 ? 2 * L : 0)>();
        else if (NS > 2 && n_after >= 1) wait_vm_lds<(NS > 2 ? L : 0)>();
        else wait_vm_lds<0>();
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
    };

    f32x4 acc = {0.0f, 0.0f, 0.0f, 0.0f};
    const uint4 ones = make_uint4(kOnes, kOnes, kOnes, kOnes);
    auto compute = [&](const auto &S) {
        const uint8_t *wrow = (const uint8_t *)S.w + (16 * r + li) * kB;
        auto body = [&](auto hc) {
            constexpr int H = decltype(hc)::value;
#pragma unroll
            for (int jj = 0; jj < JP; jj++) {
                const int j = H * JP + jj;
                uint4 xa[3];
#pragma unroll
                for (int p = 0; p < 3; p++) xa[p] = S.xp[3 * j + p][lane];
                const RawQ raw = stage_raw<F>(wrow, nullptr, j, g);
                const uint4 wc = Q::codes(raw, g);
                const Scl sc = Q::scale(raw, j);
                f32x4 sa = {0.0f, 0.0f, 0.0f, 0.0f}, dc = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
                for (int p = 0; p < 3; p++) sa = mfma(xa[p], ones, sa);
#pragma unroll
                for (int p = 0; p < 3; p++) dc = mfma(xa[p], wc, dc);
                const float c = sc.sc, cs = sc.sc * Q::kOff + sc.m;
#pragma unroll
                for (int i = 0; i < 4; i++) acc[i] = accumulate1(acc[i], c, cs, dc[i], sa[i]);
            }
        };
        if constexpr (NKH == 1) body(ic<0>{});
        else if constexpr (NKH == 2) { if (h == 0) body(ic<0>{}); else body(ic<1>{}); }
        else if constexpr (NKH == 4) {
            if (h == 0) body(ic<0>{}); else if (h == 1) body(ic<1>{}); else if (h == 2) body(ic<2>{}); else body(ic<3>{});
        } else {
            switch (h) {
            case 0: body(ic<0>{}); break;
            case 1: body(ic<1>{}); break;
            case 2: body(ic<2>{}); break;
            case 3: body(ic<3>{}); break;
            case 4: body(ic<4>{}); break;
            case 5: body(ic<5>{}); break;
            case 6: body(ic<6>{}); break;
            default: body(ic<7>{}); break;
            }
        }
    };
    // super-block i lives in slot i % NS; its loads were issued NS - 1 super-blocks earlier,
    // into the slot that super-block i - 1 used, which every wave finished reading before the
    // barrier of step i
    for (int i = 0; i < nsup; i++) {
        sync(min(NS - 2, nsup - 1 - i));
        if (i + NS - 1 < nsup) issue(i + NS - 1, slot[(i + NS - 1) % NS]);
        compute(slot[i % NS]);
    }

    if (preq && h == 0) {
        const int d = a.d_model, kv = a.kv_dim, hd = a.head_dim, half = hd / 2;
        const int rr = (int)min(my_row, N - 1);
        const int pair = ((rr < d ? rr : rr - d) % hd) / 2;
        const bool rot = a.use_rope && rr < d + kv && !(rr & 1);
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const int tk = min(4 * g + i, M - 1);
            qp[i].c = rot ? a.rope_cos[(int64_t)qp[i].pos * half + pair] : 0.0f;
            qp[i].sn = rot ? a.rope_sin[(int64_t)qp[i].pos * half + pair] : 0.0f;
            qp[i].cache = rr < d ? nullptr : (rr < d + kv ? a.kc_tok[tk] : a.vc_tok[tk]);
        }
    }
    if (fold) {   // r = 1 / sqrt(sum x^2 / K + eps) (RMSNormOps.cs:114)
#pragma unroll
        for (int j = 0; j < RJ; j++) {
            float t = rl[j][0];
#pragma unroll
            for (int q = 1; q < RP; q++) t += rl[j][q];
            t = wave_sum_uniform(t);
            if (lane == 0 && wv + NW * j < 16) s_r[wv + NW * j] = 1.0f / sqrtf(t / (float)w.cols + a.r_eps);
        }
    }
    // sum the NKH partial tiles of each row tile in a fixed order; wave (r, 0) applies the
    // epilogue
    if (NKH > 1 && h > 0) s_part[h - 1][r][lane] = acc;
    __syncthreads();   // s_part, and the folded-norm factors in s_r
    if (h != 0) return;
    float rs[4] = {1.0f, 1.0f, 1.0f, 1.0f};
    if (fold) {
#pragma unroll
        for (int i = 0; i < 4; i++) rs[i] = s_r[4 * g + i];
    }
    f32x4 v = acc;
#pragma unroll
    for (int k = 0; k < NKH - 1; k++) {
        const f32x4 o = s_part[k][r][lane];
#pragma unroll
        for (int i = 0; i < 4; i++) v[i] += o[i];
    }
    float sq[4];
#pragma unroll
    for (int i = 0; i < 4; i++) {
        const float xn = qgemm_epilogue(a, v[i] * rs[i], my_row, 4 * g + i, true, pre, pres[i], pg, qp[i]);
        sq[i] = xn * xn;
    }
    if (a.np != nullptr) {   // producer of a folded norm: x^2 summed over the tile's 16 rows
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const float t = row16_sum(sq[i]);
            const int tok = 4 * g + i;
            if (li == 0 && tok < M) a.nss[(int64_t)(row_base / 16 + r) * M + tok] = t;
        }
    }
}

// Activation parts: token m, sub-block s, part p -> Xp[m/16][s][p][g][m%16][perm] (bf16).
// x = hi + mid + lo with hi = bf16(x), mid = bf16(x - hi), lo = bf16(x - hi - mid), each
// rounded to nearest even (bf16_rne, xp_store); tokens beyond M (tile padding) are zero.

// Parts and stores of one item (8 elements of sub-block s, group g) of token row t of tile tt.
__device__ __forceinline__ void qprep_store(const float *v, uint8_t *__restrict__ xp, int nsb, int tt, int t, int i)
{
    const int s = i >> 2, g = i & 3;
    uint32_t part[3][8];
#pragma unroll
    for (int k = 0; k < 8; k++) {
        const float f = v[k];
        const uint32_t h = bf16_rne(f);
        const float r1 = f - __uint_as_float(h << 16);
        const uint32_t mm = bf16_rne(r1);
        const float r2 = r1 - __uint_as_float(mm << 16);
        part[0][k] = h;
        part[1][k] = mm;
        part[2][k] = bf16_rne(r2);
    }
#pragma unroll
    for (int p = 0; p < 3; p++) {
        // pair q = (element q, element q + 4)
        uint4 o;
        o.x = part[p][0] | (part[p][4] << 16);
        o.y = part[p][1] | (part[p][5] << 16);
        o.z = part[p][2] | (part[p][6] << 16);
        o.w = part[p][3] | (part[p][7] << 16);
        *(uint4 *)(xp + (((size_t)tt * nsb + s) * 3 + p) * 1024 + (g * 16 + t) * 16) = o;
    }
}

__device__ __forceinline__ void unpack8(const float4 &a, const float4 &b, float *v)
{
    v[0] = a.x; v[1] = a.y; v[2] = a.z; v[3] = a.w; v[4] = b.x; v[5] = b.y; v[6] = b.z; v[7] = b.w;
}

// Sub-block sums of the values of item i of token m (the items of a sub-block are four neighbouring lanes).
template <int SUMS>
__device__ __forceinline__ void qprep_sums(const float *v, uint8_t *xp, int nsb, int m, int Mp, int i)
{
    if constexpr (SUMS != 0) {
        float q = ((v[0] + v[1]) + (v[2] + v[3])) + ((v[4] + v[5]) + (v[6] + v[7]));
        q += __shfl_xor(q, 1, 64);
        const float o = __shfl_xor(q, 2, 64);
        if ((i & 3) == 0) xp_sums(xp, SUMS, Mp, nsb, m, i >> 2, q, o);
    }
}

// One workgroup per token (rows M..Mp-1 of the last tile are zero): the norm statistic of the
// row (RMSNorm: RMSNormOps.cs:114; LayerNorm: LayerNormOps.cs:92-119), the normalised value in
// the reference's operation order (gamma * (x * invRms); fma(gamma, (x - mean) * invStd, beta)),
// then its three bf16 parts at Xp[m/16][s][p][g][m%16][perm].  Thread j holds items j + 256 u
// (u < IPT, K <= 2048 * IPT): the row, gamma and beta are loaded in one batch before the
// statistic, so the kernel makes one round trip to memory.  pro: PRO_RMS or PRO_LN.  SUMS: the kind of sub-block sums written (xp_sums).
template <int IPT, int SUMS>
__global__ __launch_bounds__(256) void k_qprep(const float *__restrict__ x, int64_t x_stride, int M, int K,
                                               int pro, const float *__restrict__ gamma,
                                               const float *__restrict__ beta, float eps,
                                               uint8_t *__restrict__ xp)
{
    __shared__ float red[16];
    const int m = blockIdx.x;
    const int nsb = K >> 5, items = K >> 3;   // item = 8 elements (sub-block s, group g)
    const int tt = m >> 4, t = m & 15;
    const float *xr = x + (int64_t)m * x_stride;
    const int tid = threadIdx.x;
    if (m >= M) {   // padding row of the last tile
        float z[8] = {0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f};
        for (int i = tid; i < items; i += 256) {
            qprep_store(z, xp, nsb, tt, t, i);
            qprep_sums<SUMS>(z, xp, nsb, m, (int)gridDim.x, i);
        }
        return;
    }
    float4 xa[IPT][2], ga[IPT][2], ba[IPT][2];
#pragma unroll
    for (int u = 0; u < IPT; u++) {
        const int i = tid + 256 * u;
        if (i < items) {
            xa[u][0] = ((const float4 *)xr)[2 * i];
            xa[u][1] = ((const float4 *)xr)[2 * i + 1];
            ga[u][0] = ((const float4 *)gamma)[2 * i];
            ga[u][1] = ((const float4 *)gamma)[2 * i + 1];
            if (pro == PRO_LN) {
                ba[u][0] = ((const float4 *)beta)[2 * i];
                ba[u][1] = ((const float4 *)beta)[2 * i + 1];
            }
        }
    }
    float sc = 1.0f, mean = 0.0f;
    if (pro == PRO_RMS) {
        float ss = 0.0f;
#pragma unroll
        for (int u = 0; u < IPT; u++)
            if (tid + 256 * u < items) {
                float v[8];
                unpack8(xa[u][0], xa[u][1], v);
#pragma unroll
                for (int k = 0; k < 8; k++) { const float q = v[k] * v[k]; ss += q; }
            }
        ss = block_sum<4>(ss, red);
        sc = 1.0f / sqrtf(ss / (float)K + eps);
    } else {
        float tsum = 0.0f;
#pragma unroll
        for (int u = 0; u < IPT; u++)
            if (tid + 256 * u < items) {
                float v[8];
                unpack8(xa[u][0], xa[u][1], v);
#pragma unroll
                for (int k = 0; k < 8; k++) tsum += v[k];
            }
        mean = block_sum<4>(tsum, red) / (float)K;
        float sq = 0.0f;
#pragma unroll
        for (int u = 0; u < IPT; u++)
            if (tid + 256 * u < items) {
                float v[8];
                unpack8(xa[u][0], xa[u][1], v);
#pragma unroll
                for (int k = 0; k < 8; k++) { const float dd = v[k] - mean; const float q = dd * dd; sq += q; }
            }
        sq = block_sum<4>(sq, red);
        sc = 1.0f / sqrtf(sq / (float)K + eps);
    }
#pragma unroll
    for (int u = 0; u < IPT; u++) {
        const int i = tid + 256 * u;
        if (i >= items) continue;
        float v[8];
        unpack8(xa[u][0], xa[u][1], v);
        if (pro == PRO_RMS) {
            float gg[8];
            unpack8(ga[u][0], ga[u][1], gg);
#pragma unroll
            for (int k = 0; k < 8; k++) v[k] = gg[k] * (v[k] * sc);
        } else {
            float gg[8], be[8];
            unpack8(ga[u][0], ga[u][1], gg);
            unpack8(ba[u][0], ba[u][1], be);
#pragma unroll
            for (int k = 0; k < 8; k++) v[k] = __builtin_fmaf(gg[k], (v[k] - mean) * sc, be[k]);
        }
        qprep_store(v, xp, nsb, tt, t, i);
        qprep_sums<SUMS>(v, xp, nsb, m, (int)gridDim.x, i);
    }
}

// Rows longer than 2048 * 4: the same with the row read twice in loops.
template <int SUMS>
__global__ __launch_bounds__(256) void k_qprep_long(const float *__restrict__ x, int64_t x_stride, int M, int K,
                                                    int pro, const float *__restrict__ gamma,
                                                    const float *__restrict__ beta, float eps,
                                                    uint8_t *__restrict__ xp)
{
    __shared__ float red[16];
    const int m = blockIdx.x;
    const int nsb = K >> 5, items = K >> 3;
    const float *xr = x + (int64_t)m * x_stride;
    const bool live = m < M;
    float sc = 1.0f, mean = 0.0f;
    if (live && pro == PRO_RMS) {
        float ss = 0.0f;
        for (int i = threadIdx.x; i < items; i += 256) {
            float v[8];
            unpack8(((const float4 *)xr)[2 * i], ((const float4 *)xr)[2 * i + 1], v);
#pragma unroll
            for (int k = 0; k < 8; k++) { const float q = v[k] * v[k]; ss += q; }
        }
        ss = block_sum<4>(ss, red);
        sc = 1.0f / sqrtf(ss / (float)K + eps);
    } else if (live && pro == PRO_LN) {
        float tsum = 0.0f;
        for (int i = threadIdx.x; i < items; i += 256) {
            float v[8];
            unpack8(((const float4 *)xr)[2 * i], ((const float4 *)xr)[2 * i + 1], v);
#pragma unroll
            for (int k = 0; k < 8; k++) tsum += v[k];
        }
        mean = block_sum<4>(tsum, red) / (float)K;
        float sq = 0.0f;
        for (int i = threadIdx.x; i < items; i += 256) {
            float v[8];
            unpack8(((const float4 *)xr)[2 * i], ((const float4 *)xr)[2 * i + 1], v);
#pragma unroll
            for (int k = 0; k < 8; k++) { const float dd = v[k] - mean; const float q = dd * dd; sq += q; }
        }
        sq = block_sum<4>(sq, red);
        sc = 1.0f / sqrtf(sq / (float)K + eps);
    }
    const int tt = m >> 4, t = m & 15;
    for (int i = threadIdx.x; i < items; i += 256) {
        float v[8];
        if (live) {
            unpack8(((const float4 *)xr)[2 * i], ((const float4 *)xr)[2 * i + 1], v);
            if (pro == PRO_RMS) {
                float gg[8];
                unpack8(((const float4 *)gamma)[2 * i], ((const float4 *)gamma)[2 * i + 1], gg);
#pragma unroll
                for (int k = 0; k < 8; k++) v[k] = gg[k] * (v[k] * sc);
            } else {
                float gg[8], be[8];
                unpack8(((const float4 *)gamma)[2 * i], ((const float4 *)gamma)[2 * i + 1], gg);
                unpack8(((const float4 *)beta)[2 * i], ((const float4 *)beta)[2 * i + 1], be);
#pragma unroll
                for (int k = 0; k < 8; k++) v[k] = __builtin_fmaf(gg[k], (v[k] - mean) * sc, be[k]);
            }
        } else {
#pragma unroll
            for (int k = 0; k < 8; k++) v[k] = 0.0f;
        }
        qprep_store(v, xp, nsb, tt, t, i);
        qprep_sums<SUMS>(v, xp, nsb, m, (int)gridDim.x, i);
    }
}

// Many tokens (qprep_per_token), or no norm: a workgroup takes 4 tokens (a quarter of a token tile), thread (item lane
// tid / 4, token tid % 4).  Four neighbouring lanes store the same item of four tokens, 64
// contiguous bytes of a part (one token per workgroup stored 16-byte pieces 256 bytes apart, which
// ran at a third of the copy rate).  The rows of a norm are read again from the L1 for the
// second pass instead of being held in registers.  SUMS: the kind of sub-block sums written (xp_sums).
// Without a norm no thread needs the whole row, and the rows are cut into spans of items as well
// (qprep_span): what bounds few tokens is the chain of loads in the few workgroups that four tokens
// each make.
template <int PRO, int SUMS>
__global__ __launch_bounds__(256) void k_qprep_tokens(const float *__restrict__ x, int64_t x_stride, int M, int K,
                                                      const float *__restrict__ gamma,
                                                      const float *__restrict__ beta, float eps,
                                                      uint8_t *__restrict__ xp, int span)
{
    __shared__ float red[4][4];
    const int nsb = K >> 5, items = K >> 3, ntt = (M + 15) >> 4;
    const int tid = threadIdx.x, tq = tid & 3, i0 = tid >> 2;
    const int first = (int)blockIdx.y * span, end = min(items, first + span);   // this workgroup's items
    const int m = blockIdx.x * 4 + tq, tt = m >> 4, t = m & 15;
    const bool live = m < M;
    const float4 *xr = (const float4 *)(x + (int64_t)min(m, M - 1) * x_stride);
    const float4 *g4 = (const float4 *)gamma, *b4 = (const float4 *)beta;
    // sum over the row of this thread's token: lanes of equal tid % 4, then the four waves
    auto row_sum = [&](float v) {
#pragma unroll
        for (int o = 4; o < 64; o <<= 1) v += __shfl_xor(v, o, 64);
        __syncthreads();
        if ((tid & 63) < 4) red[tid >> 6][tq] = v;
        __syncthreads();
        return (red[0][tq] + red[1][tq]) + (red[2][tq] + red[3][tq]);
    };
    float sc = 1.0f, mean = 0.0f;
    if constexpr (PRO == PRO_LN) {
        float s = 0.0f;
#pragma unroll 4
        for (int i = i0; i < items; i += 64) {
            float v[8];
            unpack8(xr[2 * i], xr[2 * i + 1], v);
#pragma unroll
            for (int k = 0; k < 8; k++) s += v[k];
        }
        mean = row_sum(s) / (float)K;
    }
    if constexpr (PRO != PRO_NONE) {
        float s = 0.0f;
#pragma unroll 4
        for (int i = i0; i < items; i += 64) {
            float v[8];
            unpack8(xr[2 * i], xr[2 * i + 1], v);
#pragma unroll
            for (int k = 0; k < 8; k++) { const float dd = PRO == PRO_LN ? v[k] - mean : v[k]; const float q = dd * dd; s += q; }
        }
        sc = 1.0f / sqrtf(row_sum(s) / (float)K + eps);
    }
    uint8_t *xt = xp + (size_t)tt * nsb * 3072u + t * 16;
#pragma unroll 2
    for (int i = first + i0; i < end; i += 64) {
        float v[8];
        unpack8(xr[2 * i], xr[2 * i + 1], v);
        if constexpr (PRO != PRO_NONE) {
            float gg[8];
            unpack8(g4[2 * i], g4[2 * i + 1], gg);
            if constexpr (PRO == PRO_RMS) {
#pragma unroll
                for (int k = 0; k < 8; k++) v[k] = gg[k] * (v[k] * sc);
            } else {
                float be[8];
                unpack8(b4[2 * i], b4[2 * i + 1], be);
#pragma unroll
                for (int k = 0; k < 8; k++) v[k] = __builtin_fmaf(gg[k], (v[k] - mean) * sc, be[k]);
            }
        }
#pragma unroll
        for (int k = 0; k < 8; k++) v[k] = live ? v[k] : 0.0f;   // padding rows of the last tile
        const int s = i >> 2, g = i & 3;
        if constexpr (SUMS != 0) {   // the items of a sub-block are four lanes 4 apart (all active together)
            float q = ((v[0] + v[1]) + (v[2] + v[3])) + ((v[4] + v[5]) + (v[6] + v[7]));
            q += __shfl_xor(q, 4, 64);
            const float o = __shfl_xor(q, 8, 64);
            if (g == 0) xp_sums(xp, SUMS, 16 * ntt, nsb, m, s, q, o);
        }
        uint8_t *p = xt + (size_t)s * 3072u + g * 256;
#pragma unroll
        for (int pt = 0; pt < 3; pt++) {
            uint32_t w[4];
#pragma unroll
            for (int q = 0; q < 4; q++) {   // pair q = (element q, element q + 4)
                w[q] = bf16_pair(v[q], v[q + 4]);
                v[q] -= __uint_as_float(w[q] << 16);
                v[q + 4] -= __uint_as_float(w[q] & 0xFFFF0000u);
            }
            *(uint4 *)(p + 1024 * pt) = make_uint4(w[0], w[1], w[2], w[3]);
        }
    }
}

// Items per workgroup of k_qprep_tokens: the whole row under a norm (its statistic); else one item
// per thread, and more only where that would make over 2048 workgroups (eight per CU).  Per call of the
// operator: 16 tokens of 8192 18.3 us (16 workgroups of whole rows in k_qprep, 5.1 us of it) -> 17.6; from
// 511 tokens on, whole rows and spans are within 1 % of each other.
unsigned qprep_span(unsigned groups, unsigned items, int pro)
{
    if (pro != PRO_NONE) return items;
    const unsigned steps = (items + 63) / 64;   // 64 items at a time
    return 64 * std::max(1u, (groups * steps + 2047) / 2048);
}

template <int F, int RT, int TT, int NW, int SB>
hipError_t launch_frt(const QgemmArgs &a, hipStream_t s)
{
    const dim3 grid((unsigned)((a.w.rows + 16 * RT - 1) / (16 * RT)), (unsigned)(((a.M + 15) / 16 + TT - 1) / TT));
    hipLaunchKernelGGL((k_qgemm<F, RT, TT, NW, SB>), grid, dim3(64 * NW), 0, s, a);
    return hipGetLastError();
}

template <int F, int RT, int TT, int NW, int TS = 1>
hipError_t launch_st(const QgemmArgs &a, hipStream_t s)
{
    const uint32_t R = (uint32_t)((a.w.rows + 16 * RT - 1) / (16 * RT));
    // with a token split, one workgroup per 16 / TS tokens of the (single) token tile
    const uint32_t T = TS > 1 ? (uint32_t)((a.M + 16 / TS - 1) / (16 / TS))
                              : (uint32_t)(((a.M + 15) / 16 + TT - 1) / TT);
    if (TS > 1 && a.M > 16) return hipErrorInvalidValue;
    hipLaunchKernelGGL((k_qgemm_st<F, RT, TT, NW, TS>), dim3(R, T), dim3(64 * NW), 0, s, a);
    return hipGetLastError();
}

template <int F, int NR, int NKH, int NS>
hipError_t launch_rs(const QgemmArgs &a, hipStream_t s)
{
    const dim3 grid((unsigned)((a.w.rows + 16 * NR - 1) / (16 * NR)));
    hipLaunchKernelGGL((k_qgemm_rs<F, NR, NKH, NS>), grid, dim3(64 * NR * NKH), 0, s, a);
    return hipGetLastError();
}

template <int F>
hipError_t launch_f(const QgemmArgs &a, hipStream_t s)
{
    // Rows of whole 256-element super-blocks: LDS-staged weight tiles.  Up to 16 tokens: one
    // token tile per workgroup (16 waves splitting K from 8192 up).  More tokens come here only
    // while they make few tiles (qgemm_tiled): per wave RT x 16 rows by TT x 16 tokens, NW waves
    // splitting K; chosen by measurement at 256- and 512-token chunks:
    //  - K-quants (Q4_K / Q5_K): tall matrices 64 rows x 32 tokens, 4 waves; few rows or long
    //    K (O, down) the same above 320 tokens (Q4_K O 47.8 -> 39.7 us, down 92.0 -> 82.0 at
    //    512), 32 x 64 with 8 waves up to 320; other shapes (QKV) 32 x 32, 4 waves (Q4_K QKV 52.5
    //    -> 45.9 us at 512, Q5_K 52.1 -> 50.4 at 256);
    //  - Q8_0 / Q4_0 / SMQ: 32 x 64, 4 waves; few rows or long K with 8 waves;
    //  - Q6_K: 32 x 64 with 8 waves on few rows or long K, else 16 x 64.
    if (a.w.cols % 256 == 0) {
        const bool tall = a.w.rows >= 8192;
        if (a.M > 16) {
            const bool narrow = a.w.cols > 4096 || a.w.rows <= 2048;
            if constexpr (F == FMT_Q4_K || F == FMT_Q5_K) {
                if (tall || (narrow && a.M > 320)) return launch_st<F, 4, 2, 4>(a, s);
                if (narrow) return launch_st<F, 2, 4, 8>(a, s);
                return launch_st<F, 2, 2, 4>(a, s);
            }
            if constexpr (F == FMT_Q6_K) return narrow ? launch_st<F, 2, 4, 8>(a, s) : launch_st<F, 1, 4, 8>(a, s);
            // (SMQ Q8's two staged scale words per sub-block do not fit 8 waves' registers)
            if constexpr (F != FMT_SQ8)
                if (narrow) return launch_st<F, 2, 4, 8>(a, s);
            return launch_st<F, 2, 4, 4>(a, s);
        }
        // tall K-quant matrices up to one workgroup of 64 rows per CU: the row-split kernel
        // (configs[4] gate/up 16.9 -> 13.6 us); up to 192 rows per CU, 12 row tiles of 16 rows
        // per workgroup, each wave all of K, a two-slot ring (117 KB of LDS: one workgroup per
        // CU in a single round; the 64-row form took three rounds on the 49152-row head, which
        // the K-split kernel's several workgroups per CU beat): configs[4] step 1.536 -> 1.528 ms
        if constexpr (F == FMT_Q4_K || F == FMT_Q5_K) {
            if (tall && a.w.rows <= 256 * 64) return launch_rs<F, 4, 2, 3>(a, s);
            if (tall && a.w.rows <= 256 * 192) return launch_rs<F, 12, 1, 2>(a, s);
        }
        // 16 waves of >= 2 super-blocks (Q6_K and Q4_0 would spill at 128 registers)
        if constexpr (F != FMT_Q6_K && F != FMT_Q4_0)
            if (a.w.cols >= 8192) return a.M > 8 ? launch_st<F, 1, 1, 16, 2>(a, s) : launch_st<F, 1, 1, 16>(a, s);
        return tall ? launch_st<F, 2, 1, 4>(a, s) : launch_st<F, 1, 1, 8>(a, s);
    }
    // Rows of 32-element blocks only (K-quant rows are whole super-blocks).  Up to 16 tokens:
    // one token tile, 16 waves per workgroup splitting K, 4 sub-blocks per wave in flight.  More
    // tokens: 4 token tiles per workgroup (the weight codes are reused across 64 tokens), 4
    // waves, 2 sub-blocks in flight.
    if constexpr (F == FMT_Q4_K || F == FMT_Q5_K || F == FMT_Q6_K) {
        return hipErrorInvalidValue;
    } else {
        if (a.M > 16) return launch_frt<F, 1, 4, 4, 2>(a, s);
        if (a.w.rows >= 16 * 2 * 512) return launch_frt<F, 2, 1, 16, 4>(a, s);
        return launch_frt<F, 1, 1, 16, 4>(a, s);
    }
}

template <int F, int RT, int TT, int NW, int SB>
hipError_t launch_drt(const QgemmArgs &a, hipStream_t s)
{
    const dim3 grid((unsigned)((a.w.rows + 16 * RT - 1) / (16 * RT)), (unsigned)(((a.M + 15) / 16 + TT - 1) / TT));
    hipLaunchKernelGGL((k_dgemm<F, RT, TT, NW, SB>), grid, dim3(64 * NW), 0, s, a);
    return hipGetLastError();
}

// F16 / F32 weights: the decomposition of the unstaged quantized kernel (4 token tiles per
// workgroup above 16 tokens, else one tile and 16 waves splitting K).
template <int F>
hipError_t launch_d(const QgemmArgs &a, hipStream_t s)
{
    constexpr int SB = F == FMT_F32 ? 2 : 4;   // F32 with 4 in flight would spill at 128 registers
    if (a.M > 16) return launch_drt<F, 1, 4, 4, 2>(a, s);
    if (a.w.rows >= 16 * 2 * 512) return launch_drt<F, 2, 1, 16, SB>(a, s);
    return launch_drt<F, 1, 1, 16, SB>(a, s);
}

}  // namespace

size_t qgemm_parts_bytes(int M, int K) { return (size_t)(((int64_t)M + 15) / 16) * (size_t)(K / 32) * 3 * 1024; }

// the parts, then up to two sums of three bf16 parts per token and sub-block (xp_sums): 1/16
size_t qgemm_xp_bytes(int M, int K) { return qgemm_parts_bytes(M, K) / 16 * 17; }

int64_t qgemm_tiles(const WView &w, int M) { return ((w.rows + 63) / 64) * (((int64_t)M + 63) / 64); }
int64_t qgemm_tile_groups(const WView &w, int M) { return ((w.rows + 127) / 128) * (((int64_t)M + 31) / 32); }

// Both kernels' times go in steps, a round of workgroups over the chip each, so neither wins from one size
// on.  S: workgroups of the K-split kernel at 32 rows x 64 tokens; G: those of the tile kernel at 128 x 32.
//  - Q8_0, Q4_0, SMQ, Q6_K: the tile kernel wins as soon as the K-split kernel needs a second round.
//    That is S > 256 with 8 waves on a tile (few rows or long K, and Q6_K: K-split / tile, us, 2048 x 2048 Q8_0
//    256 tokens 28 / 34, 320 44 / 35; 5632 x 5632 64 35 / 47, 65 60 / 49) and S > 512 with 4 (2304 x 768 Q8_0 448
//    24 / 25, 511 28 / 25).  Longer K moves the line down, the products that remove Q4_0's offset move it up.
//  - Q4_K, Q5_K, whose K-split kernel runs larger tiles: by G, except in the first part of a new step of the
//    tile kernel (11264 x 2048 Q4_K at 128 tokens 41 / 42, 160 48 / 45, 192 56 / 60, 256 67 / 64, 352 84 / 76, 384
//    91 / 96, 448 100 / 99, 511 111 / 102; 5632 x 2048 192 35 / 41, 320 47 / 46, 384 55 / 61, 512 67 / 64).
// Where the two are level, the tile kernel (its sums are the more exact).
bool qgemm_tiled(const WView &w, int M)
{
    if (M <= 16 || w.cols % 256 != 0 || fmt_dense(w.fmt)) return false;
    const int64_t N = w.rows, K = w.cols;
    const int64_t G = qgemm_tile_groups(w, M), S = ((N + 31) / 32) * (((int64_t)M + 63) / 64);
    const bool tall = N >= 8192, narrow = N <= 2048 || K > 4096;
    if (w.fmt == FMT_Q4_K || w.fmt == FMT_Q5_K) {
        if (M <= 32) return false;
        if (tall && K < 2048) return G >= 400;
        if (tall) return G >= 390 && !(G > 512 && G <= 640) && !(K < 4096 && G > 1024 && G < 1200);
        if (narrow && M <= 320) return S > 256;
        if (N <= 2048) return G >= (M >= 1024 ? 190 : 400);
        if (G > 512 && G <= (N > 4096 ? 600 : 576)) return false;
        if (K < 2048 && N > 4096) return G >= 600 && !(G > 1024 && G < 1188);
        return G >= (K < 2048 ? 475 : K < 4096 ? 420 : 390);
    }
    if (M >= 1024 && S > 200) return true;
    if (w.fmt == FMT_Q6_K || (narrow && (w.fmt != FMT_SQ8 || K >= 2048))) return S > 256;   // (SQ8: 4 waves)
    if (K >= 4096) return S >= 352;
    const bool offset = w.fmt == FMT_Q4_0 || w.fmt == FMT_SQ4;
    // (fp32 scales cost the tile kernel's first part of a step: 11264 x 2048 SMQ Q4 65 tokens 35 / 37, 161 53 / 59)
    if (w.fmt == FMT_SQ4 && tall && K >= 2048 && ((G > 256 && G <= 352) || (G > 512 && G <= 530))) return false;
    return S > (K >= 2048 ? (tall && offset ? 512 : 352) : offset ? 704 : 512);
}

int qgemm_sums_kind(const WView &w, int M)
{
    if (!qgemm_tiled(w, M) || w.fmt == FMT_Q8_0 || w.fmt == FMT_SQ8) return 0;   // signed codes: no offset, no min
    return w.fmt == FMT_Q6_K ? 2 : 1;
}

hipError_t launch_qgemm_tile_f0(const QgemmArgs &a, hipStream_t s);
hipError_t launch_qgemm_tile_f1(const QgemmArgs &a, hipStream_t s);
hipError_t launch_qgemm_tile_f2(const QgemmArgs &a, hipStream_t s);
hipError_t launch_qgemm_tile_f3(const QgemmArgs &a, hipStream_t s);
hipError_t launch_qgemm_tile_f4(const QgemmArgs &a, hipStream_t s);
hipError_t launch_qgemm_tile_f7(const QgemmArgs &a, hipStream_t s);
hipError_t launch_qgemm_tile_f8(const QgemmArgs &a, hipStream_t s);

hipError_t launch_qgemm_tile(const QgemmArgs &a, hipStream_t s)
{
    switch (a.w.fmt) {
    case FMT_Q4_0: return launch_qgemm_tile_f0(a, s);
    case FMT_Q8_0: return launch_qgemm_tile_f1(a, s);
    case FMT_Q4_K: return launch_qgemm_tile_f2(a, s);
    case FMT_Q5_K: return launch_qgemm_tile_f3(a, s);
    case FMT_Q6_K: return launch_qgemm_tile_f4(a, s);
    case FMT_SQ8: return launch_qgemm_tile_f7(a, s);
    case FMT_SQ4: return launch_qgemm_tile_f8(a, s);
    default: return hipErrorInvalidValue;
    }
}

namespace {

// Under a norm, up to these many tokens a workgroup per token, which holds its row in registers; above, the
// store pattern of k_qprep_tokens counts for more.  Per token / four tokens, us, RMSNorm: K 768 17 tokens
// 2.5 / 3.1, 256 3.4 / 3.4, 320 3.8 / 3.4; K 2048 3.0 / 4.6, 5.0 / 5.1, 5.8 / 5.2; K 5632 4.8 / 8.6, 9.1 / 9.6,
// 11.2 / 10.1.  LayerNorm, which reads the row once more: K 768 17 tokens 3.0 / 3.9, 320 4.2 / 4.2, 384
// 4.5 / 4.3; K 2048 3.5 / 6.1, 6.4 / 6.6, 6.8 / 6.7.
bool qprep_per_token(int M, int pro) { return pro != PRO_NONE && M <= (pro == PRO_LN ? 320 : 256); }

template <int SUMS>
hipError_t launch_qprep_k(const QgemmArgs &a, const float *x, int64_t x_stride, int pro, const float *gamma,
                          const float *beta, float eps, hipStream_t s)
{
    const int K = (int)a.w.cols;
    const unsigned mp = (unsigned)((a.M + 15) / 16 * 16);
    uint8_t *xp = (uint8_t *)a.xp;
    if (qprep_per_token(a.M, pro)) {
        const auto run = [&](auto *kernel) {
            hipLaunchKernelGGL(kernel, dim3(mp), dim3(256), 0, s, x, x_stride, a.M, K, pro, gamma, beta, eps, xp);
        };
        switch ((K / 8 + 255) / 256) {
        case 1: run(k_qprep<1, SUMS>); break;
        case 2: run(k_qprep<2, SUMS>); break;
        case 3: run(k_qprep<3, SUMS>); break;
        case 4: run(k_qprep<4, SUMS>); break;
        default: run(k_qprep_long<SUMS>); break;
        }
    } else {
        const unsigned span = qprep_span(mp / 4, K / 8, pro);
        const auto run = [&](auto *kernel) {
            hipLaunchKernelGGL(kernel, dim3(mp / 4, (K / 8 + span - 1) / span), dim3(256), 0, s, x, x_stride, a.M, K,
                               gamma, beta, eps, xp, (int)span);
        };
        if (pro == PRO_NONE) run(k_qprep_tokens<PRO_NONE, SUMS>);
        else if (pro == PRO_RMS) run(k_qprep_tokens<PRO_RMS, SUMS>);
        else run(k_qprep_tokens<PRO_LN, SUMS>);
    }
    return hipGetLastError();
}

hipError_t launch_qprep(const QgemmArgs &a, const float *x, int64_t x_stride, int pro, const float *gamma,
                        const float *beta, float eps, hipStream_t s)
{
    switch (qgemm_sums_kind(a.w, a.M)) {
    case 0: return launch_qprep_k<0>(a, x, x_stride, pro, gamma, beta, eps, s);
    case 1: return launch_qprep_k<1>(a, x, x_stride, pro, gamma, beta, eps, s);
    default: return launch_qprep_k<2>(a, x, x_stride, pro, gamma, beta, eps, s);
    }
}

}  // namespace

hipError_t launch_qgemm(const QgemmArgs &a, const float *x, int64_t x_stride, int pro,
                        const float *gamma, const float *beta, float eps, hipStream_t s)
{
    if (a.M <= 0 || a.w.cols % 32 != 0 || (pro != PRO_NONE && !gamma) || (pro == PRO_LN && !beta))
        return hipErrorInvalidValue;
    if ((a.epi == EPI_SILU || a.epi == EPI_QKV) && (a.w.rows & 1)) return hipErrorInvalidValue;
    if ((uint64_t)a.w.rows * (uint64_t)a.w.nb * (uint64_t)fmt_main_bytes(a.w.fmt) >= (1ull << 32))
        return hipErrorInvalidValue;
    const int K = (int)a.w.cols;
    if ((!x && pro != PRO_NONE) || (a.yp && (a.epi == EPI_SILU ? a.w.rows % 64 : a.w.rows % 32)) ||
        (a.yp && a.epi != EPI_SILU && a.epi != EPI_GELU))
        return hipErrorInvalidValue;
    // folded RMSNorm: one token tile on the staged path (block formats only)
    if ((a.rss || a.np) && (a.M > 16 || K % 256 != 0 || fmt_dense(a.w.fmt))) return hipErrorInvalidValue;
    if (a.rss && (x || pro != PRO_NONE || a.rss_n < 1 || a.rss_n > 256)) return hipErrorInvalidValue;
    if (a.np && (a.epi != EPI_RESID || a.w.rows % 32 != 0 || !a.ngamma || !a.nss)) return hipErrorInvalidValue;
    if (x) {   // (else the parts are already in a.xp, written by the producing kernel)
        const hipError_t e = launch_qprep(a, x, x_stride, pro, gamma, beta, eps, s);
        if (e != hipSuccess) return e;
    }
    if (qgemm_tiled(a.w, a.M)) return launch_qgemm_tile(a, s);
    switch (a.w.fmt) {
    case FMT_Q4_0: return launch_f<FMT_Q4_0>(a, s);
    case FMT_Q8_0: return launch_f<FMT_Q8_0>(a, s);
    case FMT_SQ4: return launch_f<FMT_SQ4>(a, s);
    case FMT_SQ8: return launch_f<FMT_SQ8>(a, s);
    case FMT_Q4_K: return launch_f<FMT_Q4_K>(a, s);
    case FMT_Q5_K: return launch_f<FMT_Q5_K>(a, s);
    case FMT_Q6_K: return launch_f<FMT_Q6_K>(a, s);
    case FMT_F16: return launch_d<FMT_F16>(a, s);
    case FMT_F32: return launch_d<FMT_F32>(a, s);
    default: return hipErrorInvalidValue;
    }
}

}  // namespace smx

// k_attn_prefill.hip -- causal attention of a run of consecutive tokens of one session over its
// KV cache, on the bf16 matrix cores at fp32 accuracy (prefill chunks).
//
// Reference: MultiHeadAttention.Forward with T > 1 tokens over the KV cache
// (MultiHeadAttention.cs:206-297): scores Q.K^T per head (ComputeAttentionScoresInPlace,
// :676-745, MatMulOps.MatMulTransposeB), OptimizedOps.FusedScaleMaskSoftmax
// (OptimizedOps.cs:39-93) -- for query i at position p_first + i: s_j = (q.k_j) * scale for
// j <= p_first + i, max, e_j = FastExp(s_j - max) (MathUtils.cs:20-32), sum, w_j = e_j / sum --
// then out = W.V (ApplyAttentionInPlace, :810-845).
//
// The softmax needs the exact row maximum before any exponential (the Pade FastExp is not
// multiplicative, so flash-style online rescaling would not reproduce the reference), so the
// kernel makes two passes over the keys: pass 1 computes the scores and the row maxima, pass 2
// recomputes the same scores (same instruction sequence, same bits), exponentiates, sums and
// accumulates E.V.  The output is (sum_j e_j v_j) / sum, the reference's sum_j (e_j / sum) v_j
// up to rounding.
//
// What bounds it.  The fp32 matrix instructions run on the vector ALU's datapath: measured, two
// vector instructions beside each v_mfma_f32_16x16x4_f32 take it from 33 to 49 cycles, whatever
// the number of waves, so a kernel of fp32 products (50 % of the time) and FastExp (30 %) cannot
// overlap them.  The bf16 products can (eight vector instructions per product almost free).  Q, K,
// V and E therefore enter as three bf16 parts whose sum is the fp32 value (x = h + m + l), and a
// product is the six leading part products hh, hm, mh, mm, hl, lh (what is left out is below
// 2^-24 of |a| |b|), small ones first.  Then FastExp, at about 28 vector
// instructions per score, bounds pass 2 about as much as the products do.
// 2048 tokens at positions 2048 .. of 32 / 4 heads: 984 us with fp32 products, 502 now (464 GFLOP of
// part products, 920 TFLOP/s; a large bf16 product of the library runs at 1190 here), error against
// 64 bits 4.6e-7 -> 2.9e-7.
//
// Work decomposition.  A workgroup owns 32 RW query rows of one KV head: 32 RW / G tokens x the G
// query heads that share the KV head (GQA); a wave owns 32 rows.  Tiles of 32 keys are split into
// parts once per workgroup and shared through LDS (two slots: the next tile is loaded while the
// current one is multiplied).  KW groups of RW waves take alternate tiles, which halves the chain of
// keys of a workgroup; their maxima, sums and outputs are combined in LDS in a fixed order.  The workgroups
// with most keys start first.  Few rows take another kernel (below).
//
// Operands of v_mfma_f32_32x32x16_bf16 (lane l: li = l % 32, h = l / 32; 8 k-values per lane):
//   S^T = K . Q^T: A = K (key li, dimensions 16 t + 8 h ..), B = Q^T (query li, same dimensions); D
//   lane holds keys 8 (i / 4) + 4 h + i % 4 of query li in register i.
//   O^T = V^T . E^T: B = E^T (query li): the 8 keys of k-step s are registers 8 s .. 8 s + 7 of the
//   scores the lane already holds, i.e. keys 16 s + 8 q + 4 h + r; A = V^T (dimension li + 32 dt, the
//   same keys).  D lane holds dimensions 32 dt + 8 (i / 4) + 4 h + i % 4 of query li.
// Nothing is transposed, and maximum, sum and 1 / sum are the lane's own (two lanes per query).
#include <type_traits>

#include "smx_device.h"
#include "smx_internal.h"

namespace smx {

namespace {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x16 __attribute__((ext_vector_type(16)));

__device__ __forceinline__ f32x16 mma(uint4 a, uint4 b, f32x16 c)
{
    bf16x8 x, y;
    __builtin_memcpy(&x, &a, 16);
    __builtin_memcpy(&y, &b, 16);
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(x, y, c, 0, 0, 0);
}

constexpr int kHD = 64;   // head dimension of this kernel
constexpr int kKeys = 32; // keys per tile

// Value of lane l ^ 32.
__device__ __forceinline__ float half_other(float v)
{
    const float2 p = swap32(v, v);
    return (threadIdx.x & 32) ? p.x : p.y;
}

// FastExp with the quotient formed as the IEEE division does for operands that need no scaling (1/4
// <= den <= 700, |num| <= 700): reciprocal, one Newton step, quotient, residual correction.
__device__ __forceinline__ float fastexp_q(float x)
{
    x = fmaxf(-87.3f, fminf(x, 88.7f));
    const float x2 = x * x, h = x * 0.5f, q = x2 * 0.08333333f;
    const float num = (1.0f + h) + q, den = (1.0f - h) + q;
    float r = __builtin_amdgcn_rcpf(den);
    r = __builtin_fmaf(__builtin_fmaf(-den, r, 1.0f), r, r);
    const float t = num * r;
    return __builtin_fmaf(__builtin_fmaf(-den, t, num), r, t);
}

// Three bf16 parts of eight values, as one operand each.
__device__ __forceinline__ void split8(const float *v, uint4 *o)
{
    float x[8];
#pragma unroll
    for (int i = 0; i < 8; i++) x[i] = v[i];
#pragma unroll
    for (int p = 0; p < 3; p++) {
        uint32_t w[4];
#pragma unroll
        for (int k = 0; k < 4; k++) {
            w[k] = bf16_pair(x[2 * k], x[2 * k + 1]);
            if (p < 2) {
                x[2 * k] -= __uint_as_float(w[k] << 16);
                x[2 * k + 1] -= __uint_as_float(w[k] & 0xFFFF0000u);
            }
        }
        o[p] = make_uint4(w[0], w[1], w[2], w[3]);
    }
}

// Beyond this an element has no finite bf16 part (infinities among them), and its part products would be
// NaN where fp32 arithmetic has a value.
constexpr float kPartMax = 3.38e38f;

// One query of kHD dimensions (scaled) against keys 0 .. n - 1 by one wave, in fp32: the output of
// dimension `lane`.
__device__ __noinline__ float attend_fp32(const float *qr, float scale, const float *K, const float *V, int ctx_stride, int n)
{
    const int lane = threadIdx.x & 63;
    auto score = [&](int j) {
        float s = 0.0f;
        for (int e = 0; e < kHD; e++) s = __builtin_fmaf(qr[e] * scale, K[(int64_t)e * ctx_stride + j], s);
        return s;
    };
    float mx = -INFINITY, sum = 0.0f, acc = 0.0f;
    for (int j = lane; j < n; j += 64) mx = fmaxf(mx, score(j));
    for (int o = 1; o < 64; o <<= 1) mx = fmaxf(mx, __shfl_xor(mx, o, 64));
    for (int j0 = 0; j0 < n; j0 += 64) {
        const float w = j0 + lane < n ? fastexp(score(j0 + lane) - mx) : 0.0f;
        sum += w;
        for (int i = 0; i < min(64, n - j0); i++) acc = __builtin_fmaf(__shfl(w, i, 64), V[(int64_t)(j0 + i) * kHD + lane], acc);
    }
    for (int o = 1; o < 64; o <<= 1) sum += __shfl_xor(sum, o, 64);
    return acc * (1.0f / sum);
}

// With pb.blk set (several sessions' runs of a batch in one launch), a workgroup's rows, cache
// and first position come from the block table instead of the arguments: q, out and tok_off
// move to the block's first batch row, and the block is a run of M <= TT tokens at t0 = 0.
template <int RW, int KW>
__global__ __launch_bounds__(64 * RW * KW, 2) void k_attn_prefill(
    const float *__restrict__ q, int q_stride, const float *__restrict__ kc, const float *__restrict__ vc,
    float *__restrict__ out, int out_stride, int n_head, int n_kv_head, int ctx_stride, int p_first, int M,
    uint8_t *__restrict__ out_parts, int tok_off, XpSums sums, PrefillBlocks pb)
{
    constexpr int IT = 256 / (64 * RW);   // 8-element pieces of a K (V) tile per thread of a key group
    struct Lds {
        uint4 k[KW][2][4][3][2][kKeys];    // [slot][dimensions 16 t ..][part][half][key]
        uint4 v[KW][2][3][2][2][kHD];      // [slot][part][k-step][half][dimension]
        uint4 q[RW][4][3][64];             // the query parts: 48 registers a lane if they were held
        float mx[KW][RW][kKeys], sum[KW][RW][kKeys];
    };
    struct Red {
        float o[KW - 1][RW][2 * 16][64];
    };
    __shared__ __align__(16) uint8_t s_mem[sizeof(Lds)];
    __shared__ int s_large;   // an operand beyond kPartMax
    float large = 0.0f;
    auto note8 = [&](const float *x) {
#pragma unroll
        for (int e = 0; e < 8; e++) large = fmaxf(large, fabsf(x[e]));
    };
    if (threadIdx.x == 0) s_large = 0;   // (read after the loops' barriers)
    static_assert(KW > 1 && sizeof(Red) <= sizeof(uint4) * KW * 2 * 4 * 3 * 2 * kKeys * 2, "outputs reuse the tiles");
    Lds &L = *(Lds *)s_mem;
    Red &R = *(Red *)s_mem;
    const int tid = threadIdx.x, lane = tid & 63, wv = wave_id();
    const int rw = wv % RW, kg = wv / RW;
    const int li = lane & 31, h = lane >> 5;
    const int G = n_head / n_kv_head, TT = 32 * RW / G;
    const int kvh = blockIdx.y;
    int t0 = ((int)gridDim.x - 1 - (int)blockIdx.x) * TT;   // longest rows first
    if (pb.blk) {   // uniform over the workgroup
        const int b = (int)gridDim.x - 1 - (int)blockIdx.x, r0 = pb.blk[2 * b];
        M = pb.blk[2 * b + 1];
        t0 = 0;
        kc = pb.kc_tok[r0] + pb.layer_off;
        vc = pb.vc_tok[r0] + pb.layer_off;
        p_first = pb.pos[r0];
        q += (int64_t)r0 * q_stride;
        out += (int64_t)r0 * out_stride;
        tok_off += r0;
    }
    // MultiHeadAttention.cs:682; a power of two, so scaling q instead of the scores changes no bit
    const float scale = 1.0f / sqrtf((float)kHD);

    // this lane's query: row 32 rw + li of the workgroup
    const int row = 32 * rw + li;
    const int tok = t0 + row / G, head = kvh * G + row % G;
    const int npos = p_first + min(tok, M - 1) + 1;                      // keys the query sees
    if (kg == 0) {
        const float *qr = q + (int64_t)min(tok, M - 1) * q_stride + (int64_t)head * kHD;
#pragma unroll
        for (int t = 0; t < 4; t++) {
            float x[8];
#pragma unroll
            for (int e = 0; e < 8; e++) x[e] = qr[16 * t + 8 * h + e] * scale;   // (scalar loads: q is 4-byte aligned)
            uint4 p[3];
            note8(x);
            split8(x, p);
#pragma unroll
            for (int c = 0; c < 3; c++) L.q[rw][t][c][lane] = p[c];
        }
    }
    const int n_max = p_first + min(t0 + TT, M);   // keys 0 .. n_max-1 are written cache entries
    const int n_tiles = (n_max + kKeys - 1) / kKeys, n_it = (n_tiles + KW - 1) / KW;
    // K and V of one KV head span less than 4 GiB: uniform base + 32-bit offsets
    const float *K = kc + (int64_t)kvh * kHD * ctx_stride;
    const float *V = vc + (int64_t)kvh * ctx_stride * kHD;
    const uint32_t cs = (uint32_t)ctx_stride;
    const int tg = tid - 64 * RW * kg;   // thread of its key group

    // piece i of a K tile: 8 dimensions of one key; of a V tile: 8 keys (the order of a k-step's
    // operand) of one dimension
    float kr[IT][8], vr[IT][8];
    // (keys are clamped into the cache row; a tile wholly inside it needs no per-key clamp)
    const char *Kb = (const char *)K, *Vb = (const char *)V;
    auto load_k = [&](int tile) {
        const int t = min(tile, (ctx_stride - 1) / kKeys), last = ctx_stride - 1 - kKeys * t;
#pragma unroll
        for (int n = 0; n < IT; n++) {
            const int i = tg + 64 * RW * n;
            const uint32_t off = 4u * ((uint32_t)(8 * (i >> 5)) * cs + (uint32_t)min(i & 31, last));
#pragma unroll
            for (int e = 0; e < 8; e++) kr[n][e] = *(const float *)(Kb + 4u * ((uint32_t)e * cs + (uint32_t)(kKeys * t)) + off);
        }
    };
    auto store_k = [&](int slot) {
#pragma unroll
        for (int n = 0; n < IT; n++) {
            const int i = tg + 64 * RW * n, dg = i >> 5;
            uint4 p[3];
            split8(kr[n], p);
#pragma unroll
            for (int c = 0; c < 3; c++) L.k[kg][slot][dg >> 1][c][dg & 1][i & 31] = p[c];
        }
    };
    auto note_k = [&](int tile) {   // (keys past the written ones may hold anything)
#pragma unroll
        for (int n = 0; n < IT; n++) {
            const float was = large;
            note8(kr[n]);
            large = kKeys * tile + ((tg + 64 * RW * n) & 31) < n_max ? large : was;
        }
    };
    auto load_v = [&](int tile) {
        const int t = min(tile, (ctx_stride - 1) / kKeys);
        const char *b = Vb + 4u * (uint32_t)(kKeys * t * kHD);
#pragma unroll
        for (int n = 0; n < IT; n++) {
            const int i = tg + 64 * RW * n, sh = i >> 6;
            const int k0 = 16 * (sh >> 1) + 4 * (sh & 1);
            if (kKeys * (t + 1) <= ctx_stride) {   // uniform
                const uint32_t off = 4u * (uint32_t)(k0 * kHD + (i & 63));
#pragma unroll
                for (int e = 0; e < 8; e++) vr[n][e] = *(const float *)(b + off + 4 * kHD * (8 * (e >> 2) + (e & 3)));
            } else {
#pragma unroll
                for (int e = 0; e < 8; e++) {
                    const int key = min(k0 + 8 * (e >> 2) + (e & 3), ctx_stride - 1 - kKeys * t);
                    vr[n][e] = *(const float *)(b + 4u * (uint32_t)(key * kHD + (i & 63)));
                }
            }
        }
    };
    auto store_v = [&](int slot, int tile, auto tail) {
#pragma unroll
        for (int n = 0; n < IT; n++) {
            const int i = tg + 64 * RW * n, sh = i >> 6;
            // V rows past the written cache entries may hold anything: zero them (0 * NaN)
#pragma unroll
            for (int e = 0; decltype(tail)::value && e < 8; e++) {
                const int key = kKeys * tile + 16 * (sh >> 1) + 8 * (e >> 2) + 4 * (sh & 1) + (e & 3);
                vr[n][e] = key < n_max ? vr[n][e] : 0.0f;
            }
            uint4 p[3];
            note8(vr[n]);
            split8(vr[n], p);
#pragma unroll
            for (int c = 0; c < 3; c++) L.v[kg][slot][c][sh >> 1][sh & 1][i & 63] = p[c];
        }
    };
    // scores of one tile: s[i] = key 8 (i / 4) + 4 h + i % 4 of the tile, query li
    auto scores = [&](int slot, f32x16 &s) {
        int z = 0;   // opaque: the query parts are read at each use and not kept in registers
        asm volatile("" : "+s"(z));
#pragma unroll
        for (int i = 0; i < 16; i++) s[i] = 0.0f;
#pragma unroll
        for (int t = 0; t < 4; t++) {
            const uint4 kh = L.k[kg][slot][t][0][h][li], km = L.k[kg][slot][t][1][h][li], kl = L.k[kg][slot][t][2][h][li];
            const uint4 qh = L.q[rw + z][t][0][lane], qm = L.q[rw + z][t][1][lane], ql = L.q[rw + z][t][2][lane];
            s = mma(kl, qh, s);
            s = mma(kh, ql, s);
            s = mma(km, qm, s);
            s = mma(km, qh, s);
            s = mma(kh, qm, s);
            s = mma(kh, qh, s);
        }
    };

    // Iterations whose tiles (of every key group) hold only keys that all of the workgroup's queries
    // see need no mask.  Tile indices past the last one load clamped keys into slots that are masked
    // or not read.
    const int it_full = min(n_it, max(0, (p_first + min(t0, M - 1) + 1) / kKeys - (KW - 1)) / KW);
    auto seen = [&](int tile, int i) { return kKeys * tile + 8 * (i >> 2) + 4 * h + (i & 3) < npos; };

    // ---- pass 1: row maxima -----------------------------------------------------------------
    // (the next tile is split under the current one's products, the one after it is in flight)
    float mx = -INFINITY;
    load_k(kg);
    note_k(kg);
    store_k(0);
    load_k(kg + KW);
    __syncthreads();
    auto pass1 = [&](int it, auto masked) {
        const int tile = kg + KW * it;
        f32x16 s;
        scores(it & 1, s);
        note_k(tile + KW);
        store_k((it + 1) & 1);
        load_k(tile + 2 * KW);
#pragma unroll
        for (int i = 0; i < 16; i++) {
            if constexpr (decltype(masked)::value) mx = fmaxf(mx, seen(tile, i) ? s[i] : -INFINITY);
            else mx = fmaxf(mx, s[i]);
        }
        __syncthreads();
    };
    int it1 = 0;
    for (; it1 < it_full; it1++) pass1(it1, std::false_type{});
    for (; it1 < n_it; it1++) pass1(it1, std::true_type{});
    mx = fmaxf(mx, half_other(mx));
    if (h == 0) L.mx[kg][rw][li] = mx;

    // ---- pass 2: exponentials, sums and E.V --------------------------------------------------
    // Iteration it multiplies the scores of tile it + 1 while it exponentiates those of tile it, then
    // E.V of tile it while the next tiles are split into the slots read last in iteration it - 1.
    load_k(kg);
    load_v(kg);
    store_k(0);
    store_v(0, kg, std::true_type{});
    load_k(kg + KW);
    load_v(kg + KW);
    __syncthreads();
    f32x16 s0, s1;
    scores(0, s0);
    store_k(1);
    load_k(kg + 2 * KW);
    mx = L.mx[0][rw][li];
#pragma unroll
    for (int k = 1; k < KW; k++) mx = fmaxf(mx, L.mx[k][rw][li]);
    __syncthreads();
    float sum = 0.0f;
    f32x16 oh[2];   // dimensions 32 dt ..
#pragma unroll
    for (int dt = 0; dt < 2; dt++)
#pragma unroll
        for (int i = 0; i < 16; i++) oh[dt][i] = 0.0f;
    // s: scores of tile it in, sn: of tile it + 1 out
    auto pass2 = [&](int it, f32x16 &s, f32x16 &sn, auto masked, auto tail) {
        const int tile = kg + KW * it, slot = it & 1;
        scores(slot ^ 1, sn);
        float sc[16];
#pragma unroll
        for (int i = 0; i < 16; i++) {
            sc[i] = fastexp_q(s[i] - mx);
            if constexpr (decltype(masked)::value) sc[i] = seen(tile, i) ? sc[i] : 0.0f;
        }
        float ts[8];
#pragma unroll
        for (int i = 0; i < 8; i++) ts[i] = sc[i] + sc[8 + i];
        sum += ((ts[0] + ts[1]) + (ts[2] + ts[3])) + ((ts[4] + ts[5]) + (ts[6] + ts[7]));
        uint4 ep[2][3];
        split8(sc, ep[0]);
        split8(sc + 8, ep[1]);
        // the tile's products are summed by themselves and added to the output once, so that the
        // output takes one rounding per tile and not one per part product
#pragma unroll
        for (int dt = 0; dt < 2; dt++) {
            f32x16 d;
#pragma unroll
            for (int i = 0; i < 16; i++) d[i] = 0.0f;
#pragma unroll
            for (int ks = 0; ks < 2; ks++) {
                uint4 vp[3];
#pragma unroll
                for (int p = 0; p < 3; p++) vp[p] = L.v[kg][slot][p][ks][h][32 * dt + li];
                d = mma(vp[2], ep[ks][0], d);
                d = mma(vp[0], ep[ks][2], d);
                d = mma(vp[1], ep[ks][1], d);
                d = mma(vp[1], ep[ks][0], d);
                d = mma(vp[0], ep[ks][1], d);
                d = mma(vp[0], ep[ks][0], d);
            }
#pragma unroll
            for (int i = 0; i < 16; i++) oh[dt][i] += d[i];
        }
        store_k(slot);
        store_v(slot ^ 1, tile + KW, tail);
        load_k(tile + 3 * KW);
        load_v(tile + 2 * KW);
        __syncthreads();
    };
    // pairs of iterations, so that the two score registers trade places without copies
    int it = 0;
    for (; it + 2 < it_full; it += 2) {
        pass2(it, s0, s1, std::false_type{}, std::false_type{});
        pass2(it + 1, s1, s0, std::false_type{}, std::false_type{});
    }
    for (; it < n_it; it += 2) {
        pass2(it, s0, s1, std::true_type{}, std::true_type{});
        if (it + 1 < n_it) pass2(it + 1, s1, s0, std::true_type{}, std::true_type{});
    }
    if (large > kPartMax) s_large = 1;
    __syncthreads();
    if (s_large) {   // uniform: the workgroup's rows again in fp32, a row per wave at a time
        for (int r = wv; r < 32 * RW; r += RW * KW) {
            const int t = t0 + r / G, hd = kvh * G + r % G;
            if (t >= M) break;
            const float o = attend_fp32(q + (int64_t)t * q_stride + (int64_t)hd * kHD, scale, K, V, ctx_stride, p_first + t + 1);
            if (!out_parts) {
                out[(int64_t)t * out_stride + (int64_t)hd * kHD + lane] = o;
                continue;
            }
            const int nsb = n_head * kHD / 32;
            xp_store(out_parts, nsb, tok_off + t, hd * kHD + lane, o);
            if (sums.kind) {
                float a = o;   // sum over 16 dimensions
                for (int x = 1; x < 16; x <<= 1) a += __shfl_xor(a, x, 64);
                const float b = __shfl_xor(a, 16, 64);
                if ((lane & 31) == 0) xp_sums(out_parts, sums.kind, sums.M, nsb, tok_off + t, hd * (kHD / 32) + lane / 32, a, b);
            }
        }
        return;
    }
    sum += half_other(sum);
    // the key groups' sums and outputs, added in order by group 0
    if (h == 0) L.sum[kg][rw][li] = sum;
    if (kg > 0) {
#pragma unroll
        for (int dt = 0; dt < 2; dt++)
#pragma unroll
            for (int i = 0; i < 16; i++) R.o[kg - 1][rw][16 * dt + i][lane] = oh[dt][i];
    }
    __syncthreads();
    if (kg > 0) return;
    sum = L.sum[0][rw][li];
#pragma unroll
    for (int k = 1; k < KW; k++) {
        sum += L.sum[k][rw][li];
#pragma unroll
        for (int dt = 0; dt < 2; dt++)
#pragma unroll
            for (int i = 0; i < 16; i++) oh[dt][i] += R.o[k - 1][rw][16 * dt + i][lane];
    }
    const float inv = 1.0f / sum;
#pragma unroll
    for (int dt = 0; dt < 2; dt++)
#pragma unroll
        for (int i = 0; i < 16; i++) oh[dt][i] *= inv;
    const bool live = tok < M;
    if (!out_parts) {
        if (!live) return;
        float *o = out + (int64_t)tok * out_stride + (int64_t)head * kHD + 4 * h;
#pragma unroll
        for (int dt = 0; dt < 2; dt++)
#pragma unroll
            for (int g = 0; g < 4; g++)
                *(float4 *)(o + 32 * dt + 8 * g) = make_float4(oh[dt][4 * g], oh[dt][4 * g + 1], oh[dt][4 * g + 2], oh[dt][4 * g + 3]);
        return;
    }
    // Activation parts of the O projection: the lanes l and l ^ 32 hold elements r and r + 4 of each
    // group of 8, i.e. the two halves of the pairs a part stores; lane half h stores groups h, h + 2.
    const int nsb = n_head * kHD / 32, m = tok_off + tok;
#pragma unroll
    for (int dt = 0; dt < 2; dt++) {
        const int sb = head * (kHD / 32) + dt;
        uint8_t *p = out_parts + ((size_t)(m >> 4) * nsb + sb) * 3072u + (m & 15) * 16;
#pragma unroll
        for (int gg = 0; gg < 2; gg++) {
            float lo[4], hi[4];
#pragma unroll
            for (int r = 0; r < 4; r++) {
                const float2 e = swap32(oh[dt][8 * gg + r], oh[dt][8 * gg + r]);           // group 2 gg
                const float2 f = swap32(oh[dt][8 * gg + 4 + r], oh[dt][8 * gg + 4 + r]);   // group 2 gg + 1
                lo[r] = h ? f.x : e.x;
                hi[r] = h ? f.y : e.y;
            }
#pragma unroll
            for (int c = 0; c < 3; c++) {
                uint32_t w[4];
#pragma unroll
                for (int r = 0; r < 4; r++) {
                    w[r] = bf16_pair(lo[r], hi[r]);
                    lo[r] -= __uint_as_float(w[r] << 16);
                    hi[r] -= __uint_as_float(w[r] & 0xFFFF0000u);
                }
                if (live) *(uint4 *)(p + 1024 * c + 256 * (2 * gg + h)) = make_uint4(w[0], w[1], w[2], w[3]);
            }
        }
        if (sums.kind) {
            float a = 0.0f, b = 0.0f;   // dimensions 0..15 and 16..31 of the sub-block
#pragma unroll
            for (int i = 0; i < 8; i++) {
                a += oh[dt][i];
                b += oh[dt][8 + i];
            }
            a += half_other(a);
            b += half_other(b);
            if (live && h == 0) xp_sums(out_parts, sums.kind, sums.M, nsb, m, sb, a, b);
        }
    }
}

// ---- few rows ------------------------------------------------------------------------------------
typedef float f32x4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ f32x4 mma4(float a, float b, f32x4 c)
{
    return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}

constexpr int kFewRows = 32;         // query rows per workgroup (two 16-row blocks)
constexpr int kFewWaves = 8;
constexpr int kFewPitch = kHD + 4;   // LDS row pitch of the partial outputs (conflict-free writes)

// Maximum / sum over the four 16-lane rows (lanes l, l^16, l^32, l^48), the same bits in all.
__device__ __forceinline__ float rows_max(float v)
{
    float2 p = swap32(v, v);
    v = fmaxf(p.x, p.y);
    p = swap16(v, v);
    return fmaxf(p.x, p.y);
}
__device__ __forceinline__ float rows_sum(float v)
{
    float2 p = swap32(v, v);
    v = p.x + p.y;
    p = swap16(v, v);
    return p.x + p.y;
}

// The same attention for few rows, where the time is the chain of keys of one workgroup and not
// the products: 32 query rows per workgroup, whose 8 waves split the keys in 16-key tiles (wave w:
// tiles w, w + 8, ...), fp32 products (v_mfma_f32_16x16x4_f32), the same two passes; partial
// maxima, sums and outputs of the waves are combined through LDS in a fixed order.
//   S^T = K . Q^T per (16-key tile, 16-row block): A = K (lane: key l % 16, dimension
//   4j + l / 16 for step j), B = Q^T (lane: query l % 16, same dimension); D lane l holds keys
//   4(l/16) + i of query l % 16.
//   O = E . V per (16-row block, 16-dimension block): A = E (lane: query l % 16, key
//   4(l/16) + j for step j -- exactly the scores lane l already holds), B = V (lane: dimension
//   l % 16, key 4(l/16) + j); D lane l holds queries 4(l/16) + i of dimension l % 16.
__global__ __launch_bounds__(kFewWaves * 64) void k_attn_prefill_few(
    const float *__restrict__ q, int q_stride, const float *__restrict__ kc, const float *__restrict__ vc,
    float *__restrict__ out, int out_stride, int n_head, int n_kv_head, int ctx_stride, int p_first, int M,
    uint8_t *__restrict__ out_parts, int tok_off, XpSums sums, PrefillBlocks pb)
{
    extern __shared__ float s_out[];          // [kFewWaves][kFewRows][kFewPitch]
    __shared__ float s_max[kFewWaves][kFewRows], s_sum[kFewWaves][kFewRows], s_inv[kFewRows];
    const int tid = threadIdx.x, lane = tid & 63, w = wave_id();
    const int li = lane & 15, g = lane >> 4;
    const int G = n_head / n_kv_head, TT = kFewRows / G;
    const int kvh = blockIdx.y;
    int t0 = blockIdx.x * TT;
    if (pb.blk) {   // uniform over the workgroup
        const int r0 = pb.blk[2 * blockIdx.x];
        M = pb.blk[2 * blockIdx.x + 1];
        t0 = 0;
        kc = pb.kc_tok[r0] + pb.layer_off;
        vc = pb.vc_tok[r0] + pb.layer_off;
        p_first = pb.pos[r0];
        q += (int64_t)r0 * q_stride;
        out += (int64_t)r0 * out_stride;
        tok_off += r0;
    }
    const float scale = 1.0f / sqrtf((float)kHD);   // MultiHeadAttention.cs:682

    // this lane's query in row block rb: row 16 rb + li
    int npos[2];
    float qv[2][16];
#pragma unroll
    for (int rb = 0; rb < 2; rb++) {
        const int r = 16 * rb + li;
        const int t = min(t0 + r / G, M - 1), h = kvh * G + r % G;
        npos[rb] = p_first + t + 1;
        const float *qr = q + (int64_t)t * q_stride + (int64_t)h * kHD;
#pragma unroll
        for (int j = 0; j < 16; j++) qv[rb][j] = qr[4 * j + g];
    }
    const int n_max = p_first + min(t0 + TT, M);   // keys 0 .. n_max-1 are written cache entries
    const int n_tiles = (n_max + 15) >> 4;
    // K and V of one KV head span less than 4 GiB: uniform base + 32-bit offsets
    const float *K = kc + (int64_t)kvh * kHD * ctx_stride;
    const float *V = vc + (int64_t)kvh * ctx_stride * kHD;
    const uint32_t cs = (uint32_t)ctx_stride;

    auto load_k = [&](int ti, float *dst) {
        const uint32_t key = (uint32_t)min(16 * ti + li, ctx_stride - 1);
#pragma unroll
        for (int j = 0; j < 16; j++) dst[j] = K[(uint32_t)(4 * j + g) * cs + key];
    };
    auto load_v = [&](int ti, float (*dst)[4]) {
#pragma unroll
        for (int j = 0; j < 4; j++) {
            const uint32_t key = (uint32_t)min(16 * ti + 4 * g + j, ctx_stride - 1);
#pragma unroll
            for (int mb = 0; mb < 4; mb++) dst[j][mb] = V[key * kHD + 16 * mb + li];
        }
    };
    // scores of one tile: s[rb][i] = key 16 ti + 4 g + i, query li of row block rb (scaled)
    auto scores = [&](const float *kv, float (*s)[4]) {
        f32x4 a0 = {0.0f, 0.0f, 0.0f, 0.0f}, a1 = a0;
#pragma unroll
        for (int j = 0; j < 16; j++) {
            a0 = mma4(kv[j], qv[0][j], a0);
            a1 = mma4(kv[j], qv[1][j], a1);
        }
#pragma unroll
        for (int i = 0; i < 4; i++) {
            s[0][i] = a0[i] * scale;
            s[1][i] = a1[i] * scale;
        }
    };

    // ---- pass 1: row maxima -----------------------------------------------------------------
    float mx[2] = {-INFINITY, -INFINITY};
    {
        float kv[16];
        int ti = w;
        for (; ti < n_tiles; ti += kFewWaves) {
            load_k(ti, kv);
            float s[2][4];
            scores(kv, s);
#pragma unroll
            for (int rb = 0; rb < 2; rb++)
#pragma unroll
                for (int i = 0; i < 4; i++)
                    if (16 * ti + 4 * g + i < npos[rb]) mx[rb] = fmaxf(mx[rb], s[rb][i]);
        }
    }
#pragma unroll
    for (int rb = 0; rb < 2; rb++) {
        mx[rb] = rows_max(mx[rb]);
        if (g == 0) s_max[w][16 * rb + li] = mx[rb];
    }
    __syncthreads();
#pragma unroll
    for (int rb = 0; rb < 2; rb++) {
        float m = s_max[0][16 * rb + li];
#pragma unroll
        for (int v = 1; v < kFewWaves; v++) m = fmaxf(m, s_max[v][16 * rb + li]);
        mx[rb] = m;
    }

    // ---- pass 2: exponentials, sums and E.V --------------------------------------------------
    float sum[2] = {0.0f, 0.0f};
    f32x4 o[2][4];
#pragma unroll
    for (int rb = 0; rb < 2; rb++)
#pragma unroll
        for (int mb = 0; mb < 4; mb++) o[rb][mb] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
    {
        float kv[16], vv[4][4];
        int ti = w;
        for (; ti < n_tiles; ti += kFewWaves) {
            load_k(ti, kv);
            load_v(ti, vv);
            float s[2][4];
            scores(kv, s);
#pragma unroll
            for (int rb = 0; rb < 2; rb++)
#pragma unroll
                for (int i = 0; i < 4; i++) {
                    const bool ok = 16 * ti + 4 * g + i < npos[rb];
                    const float e = ok ? fastexp(s[rb][i] - mx[rb]) : 0.0f;
                    s[rb][i] = e;
                    sum[rb] += e;
                }
            // V rows past the written cache entries may hold anything: zero them (0 * NaN)
#pragma unroll
            for (int j = 0; j < 4; j++) {
                const bool ok = 16 * ti + 4 * g + j < n_max;
#pragma unroll
                for (int mb = 0; mb < 4; mb++) {
                    const float vz = ok ? vv[j][mb] : 0.0f;
                    o[0][mb] = mma4(s[0][j], vz, o[0][mb]);
                    o[1][mb] = mma4(s[1][j], vz, o[1][mb]);
                }
            }

        }
    }
    // partial sums and outputs of this wave to LDS
#pragma unroll
    for (int rb = 0; rb < 2; rb++) {
        const float sm = rows_sum(sum[rb]);
        if (g == 0) s_sum[w][16 * rb + li] = sm;
#pragma unroll
        for (int mb = 0; mb < 4; mb++)
#pragma unroll
            for (int i = 0; i < 4; i++)
                s_out[(w * kFewRows + 16 * rb + 4 * g + i) * kFewPitch + 16 * mb + li] = o[rb][mb][i];
    }
    __syncthreads();
    if (tid < kFewRows) {
        float sm = s_sum[0][tid];
#pragma unroll
        for (int v = 1; v < kFewWaves; v++) sm += s_sum[v][tid];
        s_inv[tid] = 1.0f / sm;
    }
    __syncthreads();
    // combine: thread -> (row r, 4 dimensions)
    const int r = tid >> 4, d4 = (tid & 15) * 4;
    float4 acc = *(const float4 *)&s_out[r * kFewPitch + d4];
#pragma unroll
    for (int v = 1; v < kFewWaves; v++) {
        const float4 p = *(const float4 *)&s_out[(v * kFewRows + r) * kFewPitch + d4];
        acc.x += p.x; acc.y += p.y; acc.z += p.z; acc.w += p.w;
    }
    const int t = t0 + r / G;
    if (t < M) {
        const float inv = s_inv[r];
        acc.x *= inv; acc.y *= inv; acc.z *= inv; acc.w *= inv;
        const int h = kvh * G + r % G;
        if (out_parts) {
            const int nsb = n_head * kHD / 32, k = h * kHD + d4;
            xp_store(out_parts, nsb, tok_off + t, k, acc.x);
            xp_store(out_parts, nsb, tok_off + t, k + 1, acc.y);
            xp_store(out_parts, nsb, tok_off + t, k + 2, acc.z);
            xp_store(out_parts, nsb, tok_off + t, k + 3, acc.w);
            if (sums.kind) {   // the 8 threads of a 32-dimension sub-block are neighbouring lanes
                float q = (acc.x + acc.y) + (acc.z + acc.w);
                q += dpp_mov<0xB1>(q);
                q += dpp_mov<0x4E>(q);                    // 16 dimensions
                const float o = dpp_mov<0x141>(q);        // the other quad's
                if ((tid & 7) == 0) xp_sums(out_parts, sums.kind, sums.M, nsb, tok_off + t, k >> 5, q, o);
            }
        } else {
            *(float4 *)(out + (int64_t)t * out_stride + (int64_t)h * kHD + d4) = acc;
        }
    }
}

constexpr int kRW = 4, kKW = 2;      // k_attn_prefill: 128 rows per workgroup, keys split in two

}  // namespace

bool attention_prefill_supported(int n_head, int n_kv_head, int hd)
{
    if (hd != kHD || n_kv_head <= 0 || n_head % n_kv_head) return false;
    const int G = n_head / n_kv_head;
    return G <= 32 && 32 % G == 0;
}

template <bool MANY>
hipError_t launch_prefill(unsigned blocks, const float *q, int q_stride, const float *kc, const float *vc, float *out,
                          int out_stride, int n_head, int n_kv_head, int ctx_stride, int p_first, int M, hipStream_t s,
                          uint8_t *out_parts, int tok_off, XpSums sums, const PrefillBlocks &pb)
{
    const dim3 grid(blocks, (unsigned)n_kv_head);
    if constexpr (MANY) {
        hipLaunchKernelGGL((k_attn_prefill<kRW, kKW>), grid, dim3(64 * kRW * kKW), 0, s, q, q_stride, kc, vc, out,
                           out_stride, n_head, n_kv_head, ctx_stride, p_first, M, out_parts, tok_off, sums, pb);
    } else {
        const size_t lds = (size_t)kFewWaves * kFewRows * kFewPitch * 4;
        const hipError_t e = hipFuncSetAttribute((const void *)k_attn_prefill_few,
                                                 hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
        if (e != hipSuccess) return e;
        hipLaunchKernelGGL(k_attn_prefill_few, grid, dim3(kFewWaves * 64), lds, s, q, q_stride, kc, vc, out, out_stride,
                           n_head, n_kv_head, ctx_stride, p_first, M, out_parts, tok_off, sums, pb);
    }
    return hipGetLastError();
}

// 128-row workgroups where the query rows (tokens x heads) would fill 100 of them and every run is long
// enough that they replace at least twice as many 32-row ones.  With fewer rows the chain of keys of each
// workgroup counts.  Measured (us, 32-row / 128-row): 32 / 4 heads, 511 tokens (128 workgroups) 51 / 41, 32 / 8
// heads, 700 tokens at 500 .. (176) 147 / 90; 32 / 32 heads, 255 tokens (64) 21 / 28; 32 / 4 heads, 40 tokens at
// 1000 .. (10) 49 / 77.  Short runs leave most of a 128-row workgroup empty: 32 / 32 heads, 24 runs of 20 tokens
// 24 / 34 (768 workgroups either way), of 32 30 / 35, of 33 (1536 / 768) 41 / 35; 64 of 16 46 / 89.
PrefillPlan attention_prefill_plan(int n_head, int n_kv_head, const int *counts, int n)
{
    const int few = kFewRows / (n_head / n_kv_head), many = 32 * kRW / (n_head / n_kv_head);
    int64_t tokens = 0, n_few = 0, n_many = 0;
    for (int i = 0; i < n; i++) {
        tokens += counts[i];
        n_few += (counts[i] + few - 1) / few;
        n_many += (counts[i] + many - 1) / many;
    }
    const bool m = tokens * n_head >= 100 * 32 * kRW && n_few >= 2 * n_many;
    return {m, m ? many : few};
}

hipError_t launch_attention_prefill(const float *q, int q_stride, const float *kc, const float *vc, float *out,
                                    int out_stride, int n_head, int n_kv_head, int hd, int ctx_stride,
                                    int p_first, int M, hipStream_t s, uint8_t *out_parts, int tok_off,
                                    XpSums sums)
{
    if (!attention_prefill_supported(n_head, n_kv_head, hd) || M <= 0 || p_first < 0 || ((n_head * hd) & 31) ||
        p_first + M > ctx_stride || (q_stride & 3) || (out_stride & 3) || tok_off < 0)
        return hipErrorInvalidValue;
    const PrefillPlan plan = attention_prefill_plan(n_head, n_kv_head, &M, 1);
    const unsigned blocks = (unsigned)((M + plan.rows - 1) / plan.rows);
    return plan.many
               ? launch_prefill<true>(blocks, q, q_stride, kc, vc, out, out_stride, n_head, n_kv_head, ctx_stride, p_first,
                                      M, s, out_parts, tok_off, sums, PrefillBlocks{})
               : launch_prefill<false>(blocks, q, q_stride, kc, vc, out, out_stride, n_head, n_kv_head, ctx_stride, p_first,
                                       M, s, out_parts, tok_off, sums, PrefillBlocks{});
}

hipError_t launch_attention_prefill_blocks(const float *q, int q_stride, float *out, int out_stride, int n_head,
                                           int n_kv_head, int hd, int ctx_stride, int n_blocks, bool many,
                                           const PrefillBlocks &pb, hipStream_t s, uint8_t *out_parts, XpSums sums)
{
    if (!attention_prefill_supported(n_head, n_kv_head, hd) || n_blocks <= 0 || !pb.blk || !pb.kc_tok ||
        !pb.vc_tok || !pb.pos || ((n_head * hd) & 31) || (q_stride & 3) || (out_stride & 3))
        return hipErrorInvalidValue;
    const unsigned blocks = (unsigned)n_blocks;
    return many
               ? launch_prefill<true>(blocks, q, q_stride, nullptr, nullptr, out, out_stride, n_head, n_kv_head, ctx_stride,
                                      0, 0, s, out_parts, 0, sums, pb)
               : launch_prefill<false>(blocks, q, q_stride, nullptr, nullptr, out, out_stride, n_head, n_kv_head, ctx_stride,
                                       0, 0, s, out_parts, 0, sums, pb);
}

}  // namespace smx

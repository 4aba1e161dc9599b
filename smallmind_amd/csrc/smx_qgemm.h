// smx_qgemm.h -- device code shared by the matrix-core GEMM kernels (k_qgemm.hip: up to 16 tokens, prompts
// of few tiles and rows of 32-element blocks; k_qgemm_tile.hip: the other prompts, qgemm_tiled): the bf16 weight operand of each block
// format, the activation-part loads, the per-value epilogue, and the direct-to-LDS load.
#pragma once

#include "smx_device.h"
#include "smx_formats.h"
#include "smx_internal.h"

namespace smx {

namespace {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ bf16x8 as_bf16x8(uint4 v)
{
    bf16x8 r;
    __builtin_memcpy(&r, &v, 16);
    return r;
}

__device__ __forceinline__ f32x4 mfma(uint4 a, uint4 b, f32x4 c)
{
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(as_bf16x8(a), as_bf16x8(b), c, 0, 0, 0);
}

// bf16 of an fp32 holding an integer of at most 8 significant bits (exact: the low 16 bits are 0)
__device__ __forceinline__ uint32_t pack_hi16(float lo, float hi)
{
    return __builtin_amdgcn_perm(__float_as_uint(hi), __float_as_uint(lo), 0x07060302u);
}

// (a & m) | (b & ~m) and the bf16 pair 128 + (e & m) per 16-bit half, one v_bitop3_b32 each
// (truth-table index = 4 * bit of the first operand + 2 * second + third)
__device__ __forceinline__ uint32_t bfi(uint32_t m, uint32_t a, uint32_t b)
{
    return __builtin_amdgcn_bitop3_b32(a, m, b, 0xE2);   // m ? a : b
}
__device__ __forceinline__ uint32_t code_pair(uint32_t e, uint32_t m)
{
    return __builtin_amdgcn_bitop3_b32(e, m, 0x43004300u, 0xEA);   // (e & m) | 0x43004300
}

// ---- per-format weight operand --------------------------------------------------------------
// load(): the raw words of (row, sub-block s, k-group g) -- codes and scale fields -- issued
// one sub-block ahead of use; codes(): 4 bf16 pairs (element p, element p + 4) of the group's
// 8 codes; scale(): the per-(row, sub-block) scale terms.
struct RawQ {
    uint4 h;          // K-quant super-block header
    uint32_t v, v2;   // code bytes of the group
    uint32_t H, H2;   // high bits (Q5_K: qh'; Q6_K: D0, D1)
    uint32_t d;       // fp16 scale (Q4_0, Q8_0, Q6_K) / Q6_K int8 scale pair in the high half
};
struct Scl {
    float sc, sc2, m;   // Q6_K uses sc (first 16 elements) and sc2 (second 16)
};

template <int F> struct QW;

// Q4_0: block = sub-block of 32; codes n ^ 8 (value = code - 8): offset 128 + 8.
template <> struct QW<FMT_Q4_0> {
    static constexpr float kOff = 136.0f;
    static constexpr bool kHalves = false;
    __device__ __forceinline__ static RawQ load(const WView &w, uint32_t row, int s, int g)
    {
        RawQ r{};
        const uint32_t blk = row * (uint32_t)w.nb + (uint32_t)s;
        r.v = *(const uint32_t *)(w.q + blk * 16u + 4u * g);
        r.d = w.d[blk];
        return r;
    }
    __device__ __forceinline__ static uint4 codes(const RawQ &r, int)
    {
        const uint32_t v = r.v ^ 0x88888888u;
        return make_uint4((v & 0x000F000Fu) | 0x43004300u, ((v >> 4) & 0x000F000Fu) | 0x43004300u,
                          ((v >> 8) & 0x000F000Fu) | 0x43004300u, ((v >> 12) & 0x000F000Fu) | 0x43004300u);
    }
    __device__ __forceinline__ static Scl scale(const RawQ &r, int) { return {h2f(r.d), 0.0f, 0.0f}; }
};

// Q8_0: int8 codes; bf16(b ^ 0x80) = value + 128 (exact integers up to 255).
template <> struct QW<FMT_Q8_0> {
    static constexpr float kOff = 128.0f;
    static constexpr bool kHalves = false;
    __device__ __forceinline__ static RawQ load(const WView &w, uint32_t row, int s, int g)
    {
        RawQ r{};
        const uint32_t blk = row * (uint32_t)w.nb + (uint32_t)s;
        const uint2 v = *(const uint2 *)(w.q + blk * 32u + 8u * g);
        r.v = v.x;
        r.v2 = v.y;
        r.d = w.d[blk];
        return r;
    }
    __device__ __forceinline__ static uint4 codes(const RawQ &r, int)
    {
        const uint32_t a = r.v ^ 0x80808080u, b = r.v2 ^ 0x80808080u;
        // pair p = (element p, element p + 4) = (byte p of a, byte p of b)
        float a0, a1, a2, a3, b0, b1, b2, b3;
        asm("v_cvt_f32_ubyte0 %0, %1" : "=v"(a0) : "v"(a));
        asm("v_cvt_f32_ubyte1 %0, %1" : "=v"(a1) : "v"(a));
        asm("v_cvt_f32_ubyte2 %0, %1" : "=v"(a2) : "v"(a));
        asm("v_cvt_f32_ubyte3 %0, %1" : "=v"(a3) : "v"(a));
        asm("v_cvt_f32_ubyte0 %0, %1" : "=v"(b0) : "v"(b));
        asm("v_cvt_f32_ubyte1 %0, %1" : "=v"(b1) : "v"(b));
        asm("v_cvt_f32_ubyte2 %0, %1" : "=v"(b2) : "v"(b));
        asm("v_cvt_f32_ubyte3 %0, %1" : "=v"(b3) : "v"(b));
        return make_uint4(pack_hi16(a0, b0), pack_hi16(a1, b1), pack_hi16(a2, b2), pack_hi16(a3, b3));
    }
    __device__ __forceinline__ static Scl scale(const RawQ &r, int) { return {h2f(r.d), 0.0f, 0.0f}; }
};

// SMQ blocks (Q8Tensor / Q4Tensor): the Q8_0 / Q4_0 codes with an fp32 scale per 32 elements.
template <> struct QW<FMT_SQ8> {
    static constexpr float kOff = 128.0f;
    static constexpr bool kHalves = false;
    __device__ __forceinline__ static RawQ load(const WView &w, uint32_t row, int s, int g)
    {
        RawQ r{};
        const uint32_t blk = row * (uint32_t)w.nb + (uint32_t)s;
        const uint2 v = *(const uint2 *)(w.q + blk * 32u + 8u * g);
        r.v = v.x;
        r.v2 = v.y;
        r.d = ((const uint32_t *)w.d)[blk];
        return r;
    }
    __device__ __forceinline__ static uint4 codes(const RawQ &r, int g) { return QW<FMT_Q8_0>::codes(r, g); }
    __device__ __forceinline__ static Scl scale(const RawQ &r, int) { return {__uint_as_float(r.d), 0.0f, 0.0f}; }
};

template <> struct QW<FMT_SQ4> {
    static constexpr float kOff = 136.0f;
    static constexpr bool kHalves = false;
    __device__ __forceinline__ static RawQ load(const WView &w, uint32_t row, int s, int g)
    {
        RawQ r{};
        const uint32_t blk = row * (uint32_t)w.nb + (uint32_t)s;
        r.v = *(const uint32_t *)(w.q + blk * 16u + 4u * g);
        r.d = ((const uint32_t *)w.d)[blk];
        return r;
    }
    __device__ __forceinline__ static uint4 codes(const RawQ &r, int g) { return QW<FMT_Q4_0>::codes(r, g); }
    __device__ __forceinline__ static Scl scale(const RawQ &r, int) { return {__uint_as_float(r.d), 0.0f, 0.0f}; }
};

// Q4_K: sub-block s = qs bytes 16 + 16*(s % 8) of super-block s / 8.
template <> struct QW<FMT_Q4_K> {
    static constexpr float kOff = 128.0f;
    static constexpr bool kHalves = false;
    __device__ __forceinline__ static RawQ load(const WView &w, uint32_t row, int s, int g)
    {
        RawQ r{};
        const uint32_t base = (row * (uint32_t)w.nb + ((uint32_t)s >> 3)) * 144u;
        r.h = *(const uint4 *)(w.q + base);
        r.v = *(const uint32_t *)(w.q + base + 16u + 16u * ((uint32_t)s & 7u) + 4u * g);
        return r;
    }
    __device__ __forceinline__ static uint4 codes(const RawQ &r, int)
    {
        const uint32_t v = r.v;
        return make_uint4((v & 0x000F000Fu) | 0x43004300u, ((v >> 4) & 0x000F000Fu) | 0x43004300u,
                          ((v >> 8) & 0x000F000Fu) | 0x43004300u, ((v >> 12) & 0x000F000Fu) | 0x43004300u);
    }
    __device__ __forceinline__ static Scl scale(const RawQ &r, int s)
    {
        const int j = s & 7;
        return {h2f(r.h.x & 0xFFFFu) * (float)kq_scale6(r.h.y, r.h.z, r.h.w, j, 0), 0.0f,
                h2f(r.h.x >> 16) * (float)kq_scale6(r.h.y, r.h.z, r.h.w, j, 1)};
    }
};

// Q5_K: codes = ql nibble | high bit (bit-permuted qh'), value = q - 16: offset 128 + 16.
template <> struct QW<FMT_Q5_K> {
    static constexpr float kOff = 144.0f;
    static constexpr bool kHalves = false;
    __device__ __forceinline__ static RawQ load(const WView &w, uint32_t row, int s, int g)
    {
        RawQ r{};
        const uint32_t base = (row * (uint32_t)w.nb + ((uint32_t)s >> 3)) * 176u;
        const uint32_t j = (uint32_t)s & 7u;
        r.h = *(const uint4 *)(w.q + base);
        r.v = *(const uint32_t *)(w.q + base + 48u + 16u * j + 4u * g);
        r.H = *(const uint32_t *)(w.q + base + 16u + 4u * j);
        return r;
    }
    __device__ __forceinline__ static uint4 codes(const RawQ &r, int g)
    {
        // The high bit of element 8g + 2k + p sits at bit 8k + 2g + p of H, so hg = H >> 2g
        // holds it at bit 8k + p.  e0 / e1 = the 5-bit codes of the even / odd elements
        // 2k / 2k + 1 in bits 0-4 of byte k (bits 5-7 are don't-care); pair q = (element q,
        // element q + 4) is then bytes 0 and 2 of e_{q%2} >> 8(q/2).
        const uint32_t v = r.v, hg = r.H >> (2 * g);
        const uint32_t e0 = bfi(0x0F0F0F0Fu, v, hg << 4), e1 = bfi(0x0F0F0F0Fu, v >> 4, hg << 3);
        return make_uint4(code_pair(e0, 0x001F001Fu), code_pair(e1, 0x001F001Fu), code_pair(e0 >> 8, 0x001F001Fu),
                          code_pair(e1 >> 8, 0x001F001Fu));
    }
    __device__ __forceinline__ static Scl scale(const RawQ &r, int s)
    {
        const int j = s & 7;
        return {h2f(r.h.x & 0xFFFFu) * (float)kq_scale6(r.h.y, r.h.z, r.h.w, j, 0), 0.0f,
                h2f(r.h.x >> 16) * (float)kq_scale6(r.h.y, r.h.z, r.h.w, j, 1)};
    }
};

// Q6_K: 6-bit codes, value = q - 32: offset 128 + 32; two 16-element scales per sub-block.
template <> struct QW<FMT_Q6_K> {
    static constexpr float kOff = 160.0f;
    static constexpr bool kHalves = true;
    __device__ __forceinline__ static RawQ load(const WView &w, uint32_t row, int s, int g)
    {
        RawQ r{};
        const uint32_t sb = row * (uint32_t)w.nb + ((uint32_t)s >> 3);
        const uint32_t base = sb * 208u, cc = (uint32_t)s & 7u;
        r.v = *(const uint32_t *)(w.q + base + 16u * cc + 4u * g);
        const uint2 D = *(const uint2 *)(w.q + base + 128u + 8u * cc);
        r.H = D.x;
        r.H2 = D.y;
        r.d = (uint32_t)w.d[sb] | ((uint32_t)*(const uint16_t *)(w.q + base + 192u + 2u * cc) << 16);
        return r;
    }
    __device__ __forceinline__ static uint4 codes(const RawQ &r, int g)
    {
        // The two high bits of element 8g + 2k + p sit at bits 8k + 2g of D_p, so
        // dp = D_p >> 2g holds them at bits 8k, 8k + 1: e_p = the 6-bit codes of the elements
        // 2k + p in bits 0-5 of byte k, and pair q = bytes 0 and 2 of e_{q%2} >> 8(q/2).
        const uint32_t v = r.v;
        const uint32_t e0 = bfi(0x0F0F0F0Fu, v, (r.H >> (2 * g)) << 4);
        const uint32_t e1 = bfi(0x0F0F0F0Fu, v >> 4, (r.H2 >> (2 * g)) << 4);
        return make_uint4(code_pair(e0, 0x003F003Fu), code_pair(e1, 0x003F003Fu), code_pair(e0 >> 8, 0x003F003Fu),
                          code_pair(e1 >> 8, 0x003F003Fu));
    }
    __device__ __forceinline__ static Scl scale(const RawQ &r, int)
    {
        const float d = h2f(r.d & 0xFFFFu);
        return {d * (float)(int8_t)((r.d >> 16) & 0xFFu), d * (float)(int8_t)(r.d >> 24), 0.0f};
    }
};

constexpr uint4 kZero4 = {0u, 0u, 0u, 0u};

// Activation part p of (token tile tt, sub-block s) for this lane: a wave-uniform base plus the
// lane's 32-bit byte offset, so each load is one scalar-base instruction with no per-lane
// 64-bit address arithmetic.
__device__ __forceinline__ uint4 ld_part(const uint8_t *xp, int tt, int nsb, int s, int p, uint32_t lane16)
{
    const uint8_t *base = xp + (((size_t)tt * nsb + s) * 3 + p) * 1024;
    return *(const uint4 *)(base + lane16);
}

// acc + sc * (C - off * sum x) - m * sum x as two fused steps: acc + sc*C - (sc*off + m) * sum x
// (cs = sc * off + m precomputed per row and sub-block).
__device__ __forceinline__ float accumulate1(float acc, float sc, float cs, float c, float sx)
{
    return __builtin_fmaf(sc, c, __builtin_fmaf(-cs, sx, acc));
}
// Two 16-element halves with their own scales (Q6_K): acc + sc*(Ca - off*sa) + sc2*(Cb - off*sb).
__device__ __forceinline__ float accumulate2(float acc, float sc, float sc2, float ca, float cb, float sa, float sb,
                                             float off)
{
    acc = __builtin_fmaf(-(sc * off), sa, acc);
    acc = __builtin_fmaf(-(sc2 * off), sb, acc);
    acc = __builtin_fmaf(sc, ca, acc);
    return __builtin_fmaf(sc2, cb, acc);
}
constexpr uint32_t kOnes = 0x3F803F80u;   // bf16 1.0 pair

// Inputs of the EPI_QKV epilogue for one (token, row) value, loaded by the caller ahead of the
// epilogue: the token's position, the RoPE factors of the row's pair (when it is rotated) and
// the token's K or V cache base (for K / V rows).
struct QkvPre {
    uint32_t pos;   // never negative: widening it is a zero extension, which waits for no load
    float c, sn;
    float *cache;
};

// Epilogue of one output value per (token, weight row); all lanes of the wave must call it
// (adjacent weight rows are exchanged with DPP for the paired SwiGLU / RoPE epilogues).
// Returns the new residual value for EPI_RESID with a.np set and the activation for EPI_GELU /
// EPI_SILU with a.yp set (0 for rows / tokens outside the output and up rows), else 0.  With pre, EPI_RESID takes the residual and the next norm's gamma from
// pres / pg, and EPI_QKV its position, RoPE factors and cache base from qp (all loaded by the
// caller before the epilogue) instead of loading them here, so the epilogue's stores do not
// wait for loads: vector-memory waits count stores as well, so a load between two stores
// would also wait for the first store.
__device__ __forceinline__ float qgemm_epilogue(const QgemmArgs &a, float v, uint32_t row, int tok, bool live,
                                                bool pre = false, float pres = 0.0f, float pg = 0.0f,
                                                QkvPre qp = QkvPre{0, 0.0f, 0.0f, nullptr})
{
    const uint32_t N = (uint32_t)a.w.rows;
    if (a.bias && row < N) v = v + a.bias[row];
    // value of the neighbouring weight row (lane li ^ 1 holds row ^ 1)
    const float nb = __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0xB1, 0xF, 0xF, false));
    if (!live || row >= N || tok >= a.M) return 0.0f;
    float *yr = a.y + (int64_t)tok * a.y_stride;
    switch (a.epi) {
    case EPI_STORE: yr[row] = v; break;
    case EPI_RESID: {
        const float xn = (pre ? pres : yr[row]) + v;
        yr[row] = xn;
        if (a.np) {   // the next GEMM's parts of gamma (.) x (RMSNormOps.cs:137-139 up to the factor r)
            xp_store(a.np, (int)(N >> 5), tok, (int)row, (pre ? pg : a.ngamma[row]) * xn);
            return xn;
        }
        break;
    }
    case EPI_GELU:
        if (a.yp) {
            const float y = gelu_pade(v);
            xp_store(a.yp, (int)(N >> 5), tok, (int)row, y);
            return y;
        }
        yr[row] = gelu_pade(v);
        break;
    case EPI_SILU:
        // rows interleave gate / up: out[i] = silu(gate_i) * up_i
        if (!(row & 1)) {
            const float y = silu_mul(v, nb);
            if (a.yp) {
                xp_store(a.yp, (int)(N >> 6), tok, (int)(row >> 1), y);
                return y;
            }
            yr[row >> 1] = y;
        }
        break;
    case EPI_QKV: {
        if (row & 1) break;
        const int d = a.d_model, kv = a.kv_dim, hd = a.head_dim, r = (int)row;
        const uint32_t pos = pre ? qp.pos : (uint32_t)a.tok_pos[tok];
        float v0 = v, v1 = nb;
        if (a.use_rope && r < d + kv) {
            const int pair = ((r < d ? r : r - d) % hd) / 2, half = hd / 2;
            const float c = pre ? qp.c : a.rope_cos[(int64_t)pos * half + pair];
            const float sn = pre ? qp.sn : a.rope_sin[(int64_t)pos * half + pair];
            const float t0 = v0 * c, t1 = v1 * sn, t2 = v0 * sn, t3 = v1 * c;   // RotaryEmbedding.cs:115-116
            v0 = t0 - t1;
            v1 = t2 + t3;
        }
        if (r < d) {
            yr[r] = v0;
            yr[r + 1] = v1;
        } else if (r < d + kv) {
            float *dst = (pre ? qp.cache : a.kc_tok[tok]) + a.layer_off + (int64_t)(r - d) * a.ctx_stride + pos;
            dst[0] = v0;
            dst[a.ctx_stride] = v1;
        } else {
            const int vr = r - d - kv;
            float *dst = (pre ? qp.cache : a.vc_tok[tok]) + a.layer_off + ((int64_t)(vr / hd) * a.ctx_stride + pos) * hd + (vr % hd);
            dst[0] = v0;
            dst[1] = v1;
        }
        break;
    }
    default: break;
    }
    return 0.0f;
}

// 16 bytes per lane from global address g into LDS at l + 16 * lane (l wave-uniform; M0 holds
// it, with the one wait state between the M0 write and the load)
__device__ __forceinline__ void lds_dma16(const void *g, void *l)
{
    const uint32_t la = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) void *)l;
    asm volatile("s_nop 0\n\tglobal_load_lds_dwordx4 %0, off" ::"v"(g), "{m0}"(la) : "memory");
}

// s_waitcnt vmcnt(n) lgkmcnt(0) (gfx9 encoding: vmcnt in bits 3:0 and 15:14, expcnt 6:4 left
// alone, lgkmcnt 11:8): the wave's vector-memory loads older than its last n have landed and
// its own LDS reads have completed
template <int N> __device__ __forceinline__ void wait_vm_lds()
{
    static_assert(N >= 0 && N < 64, "vmcnt is 6 bits");
    __builtin_amdgcn_s_waitcnt((N & 15) | ((N >> 4) << 14) | (7 << 4));
}

}  // namespace

}  // namespace smx

// k_quant.hip -- block-format kernels: GGUF dequantization, encoders, weight repacking.
//
// GGUF-layout dequantization restates GgufModelLoader.Convert*Tensor (GgufModelLoader.cs:
// 419-917) element for element; Q8_0/Q4_0 encoders restate Q8Tensor.Quantize /
// Q4Tensor.Quantize (Q8Tensor.cs:72-128, Q4Tensor.cs:75-134) at block 32 with an fp16 scale;
// the K-quant encoders (the reference has none) write the layout that the reference decodes.
#include <type_traits>

#include "smx_formats.h"

namespace smx {

namespace {

constexpr int kThreads = 256;

__device__ __forceinline__ float rd_half_exact(const uint8_t *p) { return h2f_exact(ld_u16(p)); }

// The codecs are bound by memory: 4 bytes per element on one side, and a block's bytes on the other.
// A thread takes 4 elements (8 of an 8-bit encoder), so that a wave reads or writes 1 KB of floats at once and the bytes of its
// blocks (one K-quant block, eight of the 32-element ones) together; headers are read by all lanes of a
// block from the same line, and an encoder's maxima are reduced over the lanes of its block.  Of 11.5 M
// elements of Q4_K (53 MB each way, 10.6 us at the 5.0 TB/s of a large copy), one thread per block or
// 32 elements, each with its own lines: encode 90 us, decode 125 us; now 28 and 21.

// Bytes at any alignment (the hardware's unaligned access).
template <typename T>
__device__ __forceinline__ T ld_any(const uint8_t *p)
{
    T v;
    __builtin_memcpy(&v, p, sizeof v);
    return v;
}
template <typename T>
__device__ __forceinline__ void st_any(uint8_t *p, T v) { __builtin_memcpy(p, &v, sizeof v); }

template <int T>
struct Type {
    static constexpr bool k = T == SMX_TYPE_Q4_K || T == SMX_TYPE_Q5_K || T == SMX_TYPE_Q6_K;
    static constexpr bool plain = T == SMX_TYPE_F32 || T == SMX_TYPE_F16;
    static constexpr int elems = k ? 256 : plain ? 4 : 32;
    static constexpr int bytes = T == SMX_TYPE_F32 ? 16 : T == SMX_TYPE_F16 ? 8 : T == SMX_TYPE_Q8_0 ? 34
                               : T == SMX_TYPE_Q4_0 ? 18 : T == SMX_TYPE_Q4_K ? 144 : T == SMX_TYPE_Q5_K ? 176
                               : T == SMX_TYPE_Q6_K ? 210 : T == SMX_TYPE_SMQ_Q8 ? 36 : 20;
    // elements per thread of the encoder (8-bit codes: 8, half as many stores, which lie at odd addresses; 51 M
    // elements of Q8_0, one thread per block / 4 / 8 elements per thread: 38 / 44 / 35 us)
    static constexpr int enc = T == SMX_TYPE_Q8_0 || T == SMX_TYPE_SMQ_Q8 ? 8 : 4;
};

// ---- GGUF dequantization --------------------------------------------------------------------
__device__ __forceinline__ int nib(uint32_t n) { return n < 8u ? (int)n : (int)n - 16; }

// 6-bit scale j of the packed scales at s (the minimums at s + 6)
__device__ __forceinline__ uint32_t k_scale(const uint8_t *s, int j)
{
    const int k = (6 * j) >> 3, sh = (6 * j) & 7;
    return (ld_any<uint16_t>(s + k) >> sh) & 63u;   // the byte after the last is masked away
}

// Element v (of 256, 32 or 4) of block b.
template <int T>
__device__ __forceinline__ float decode_one(const uint8_t *b, int v)
{
    if constexpr (T == SMX_TYPE_F32) {
        return __uint_as_float(ld_any<uint32_t>(b + 4 * v));
    } else if constexpr (T == SMX_TYPE_F16) {
        return rd_half_exact(b + 2 * v);
    } else if constexpr (T == SMX_TYPE_SMQ_Q8) {
        // Q8Tensor.Dequantize / Q4Tensor.Dequantize (Q8Tensor.cs:131-157, Q4Tensor.cs:150-178):
        // code * scale, one fp32 multiply; 32-element blocks of [fp32 scale | codes]
        return (float)(int8_t)b[4 + v] * __uint_as_float(ld_any<uint32_t>(b));
    } else if constexpr (T == SMX_TYPE_SMQ_Q4) {   // Q4Tensor.DecodeNibble (Q4Tensor.cs:140-143)
        return (float)nib((b[4 + v / 2] >> (4 * (v & 1))) & 15u) * __uint_as_float(ld_any<uint32_t>(b));
    } else if constexpr (T == SMX_TYPE_Q8_0) {   // GgufModelLoader.cs:464-492
        return (float)(int8_t)b[2 + v] * rd_half_exact(b);
    } else if constexpr (T == SMX_TYPE_Q4_0) {   // GgufModelLoader.cs:494-534
        return (float)nib((b[2 + v / 2] >> (4 * (v & 1))) & 15u) * rd_half_exact(b);
    } else if constexpr (T == SMX_TYPE_Q6_K) {   // GgufModelLoader.cs:849-917, 16-element sub-blocks
        const float sc = rd_half_exact(b + 208) * (float)(int8_t)b[192 + v / 16];
        const uint32_t low4 = (b[v / 2] >> (4 * (v & 1))) & 15u;
        const uint32_t high2 = (b[128 + v / 4] >> ((v % 4) * 2)) & 3u;
        return sc * (float)((int)(low4 | (high2 << 4)) - 32);
    } else {
        const int j = v / 32;
        const float sc = rd_half_exact(b) * (float)k_scale(b + 4, j);
        const float m = rd_half_exact(b + 2) * (float)k_scale(b + 10, j);
        if constexpr (T == SMX_TYPE_Q4_K) {   // GgufModelLoader.cs:657-741
            const float t = sc * (float)((b[16 + v / 2] >> (4 * (v & 1))) & 15u);
            return t - m;
        } else {   // Q5_K, GgufModelLoader.cs:748-840
            const uint32_t hb = ((b[16 + v / 8] >> (v % 8)) & 1u) << 4;
            const uint32_t low4 = (b[48 + v / 2] >> (4 * (v & 1))) & 15u;
            const float t = sc * (float)((int)(hb | low4) - 16);
            return t - m;
        }
    }
}

template <int T>
__global__ void k_dequant_gguf(const uint8_t *__restrict__ src, int64_t n, float *__restrict__ out)
{
    const int64_t e0 = 4 * ((int64_t)blockIdx.x * blockDim.x + threadIdx.x);
    if (e0 >= n) return;
    const uint8_t *b = src + e0 / Type<T>::elems * Type<T>::bytes;
    const int v = (int)(e0 % Type<T>::elems);
    if (e0 + 4 <= n && ((uintptr_t)out & 15) == 0) {
        *(float4 *)(out + e0) = make_float4(decode_one<T>(b, v), decode_one<T>(b, v + 1), decode_one<T>(b, v + 2),
                                            decode_one<T>(b, v + 3));
        return;
    }
    for (int i = 0; i < 4 && e0 + i < n; i++) {
        // the reference's Q4_K loop runs over whole pairs, so an odd last element stays zero
        const bool half = T == SMX_TYPE_Q4_K && (i & 1) == 0 && e0 + i + 1 == n;
        out[e0 + i] = half ? 0.0f : decode_one<T>(b, v + i);
    }
}

// ---- encoders -------------------------------------------------------------------------------
__device__ __forceinline__ float clampf(float v, float lo, float hi) { return v < lo ? lo : (v > hi ? hi : v); }

// Maximum over groups of G lanes of values that are not NaN.
template <int G>
__device__ __forceinline__ float group_max(float m)
{
#pragma unroll
    for (int o = 1; o < G; o <<= 1) m = fmaxf(m, __shfl_xor(m, o, 64));
    return m;
}

// Largest magnitude of the group's elements (E per lane), NaN left out
template <int G, int E = 4>
__device__ __forceinline__ float group_maxabs(const float *x)
{
    float m = 0.0f;
#pragma unroll
    for (int i = 0; i < E; i++) { const float a = fabsf(x[i]); if (a > m) m = a; }
    return group_max<G>(m);
}

// the OR over the eight groups of 8 lanes of a wave
__device__ __forceinline__ uint64_t or_groups(uint64_t v)
{
#pragma unroll
    for (int o = 8; o < 64; o <<= 1) v |= __shfl_xor((unsigned long long)v, o, 64);
    return v;
}

// Q8_0 / Q4_0 and Q8Tensor.Quantize / Q4Tensor.Quantize (Q8Tensor.cs:72-128, Q4Tensor.cs:75-134) as
// written, fp32 scale kept, at 32-element blocks (the SMQ upload layout: fp32 scale, then the codes).
template <int T>
__device__ __forceinline__ void encode32(const float *x, int v, uint8_t *b)
{
    constexpr bool q8 = T == SMX_TYPE_Q8_0 || T == SMX_TYPE_SMQ_Q8, smq = T == SMX_TYPE_SMQ_Q8 || T == SMX_TYPE_SMQ_Q4;
    constexpr int head = smq ? 4 : 2, E = Type<T>::enc;
    const float maxAbs = group_maxabs<32 / E, E>(x);
    const float scale = maxAbs > 0.0f ? maxAbs / (q8 ? 127.0f : 7.0f) : 1.0f;
    const float inv = 1.0f / scale;
    if (v == 0) {
        if (smq) st_any<uint32_t>(b, __float_as_uint(scale));
        else st_any<uint16_t>(b, (uint16_t)f2h_rne(scale));
    }
    int c[E];
#pragma unroll
    for (int i = 0; i < E; i++) {
        const float t = x[i] * inv;
        c[i] = (int)rintf(clampf(t, q8 ? -127.0f : -8.0f, q8 ? 127.0f : 7.0f));
    }
    if constexpr (q8) {
        struct { uint32_t w[E / 4]; } o;
#pragma unroll
        for (int i = 0; i < E; i += 4)
            o.w[i / 4] = (uint32_t)(c[i] & 255) | (uint32_t)(c[i + 1] & 255) << 8 | (uint32_t)(c[i + 2] & 255) << 16 |
                         (uint32_t)(c[i + 3] & 255) << 24;
        __builtin_memcpy(b + head + v, &o, E);
    } else {
        st_any<uint16_t>(b + head + v / 2, (uint16_t)((c[0] & 15) | (c[1] & 15) << 4 | (c[2] & 15) << 8 | (c[3] & 15) << 12));
    }
}

// d, dmin and the packed scales of a K-quant block, by the lane of its first element
__device__ __forceinline__ void put_k_header(uint8_t *b, int v, uint32_t d16, uint32_t m16, int ls, int lm)
{
    const int j = v / 32;
    const uint64_t s = or_groups((uint64_t)(ls & 63) << (6 * j)), m = or_groups((uint64_t)(lm & 63) << (6 * j));
    if (v == 0) {
        st_any<uint32_t>(b, d16 | m16 << 16);
        st_any<uint32_t>(b + 4, (uint32_t)s);
        st_any<uint32_t>(b + 8, (uint32_t)(s >> 32) | (uint32_t)m << 16);
        st_any<uint32_t>(b + 12, (uint32_t)(m >> 16));
    }
}

__device__ __forceinline__ void encode_q4_k(const float *x, int v, uint8_t *b)
{
    // lowest of the sub-block and 0, and highest, which is NaN if the first element is
    float lo = 0.0f, hi = -INFINITY;
#pragma unroll
    for (int i = 0; i < 4; i++) { if (x[i] < lo) lo = x[i]; if (x[i] > hi) hi = x[i]; }
    lo = -group_max<8>(-lo);
    hi = group_max<8>(hi);
    const float first = __shfl(x[0], (int)(threadIdx.x & 56), 64);
    if (first != first) hi = first;
    const float scl = (hi - lo) / 15.0f, mnv = -lo;
    float maxs = 0.0f, maxm = 0.0f;
    if (scl > maxs) maxs = scl;
    if (mnv > maxm) maxm = mnv;
    maxs = group_max<64>(maxs);
    maxm = group_max<64>(maxm);
    const uint32_t d16 = f2h_rne(maxs / 63.0f), m16 = f2h_rne(maxm / 63.0f);
    const float df = h2f_exact(d16), mf = h2f_exact(m16);
    const int ls = df > 0.0f ? (int)clampf(rintf(scl / df), 0.0f, 63.0f) : 0;
    const int lm = mf > 0.0f ? (int)clampf(rintf(mnv / mf), 0.0f, 63.0f) : 0;
    put_k_header(b, v, d16, m16, ls, lm);
    const float sc = df * (float)ls, m = mf * (float)lm;
    uint32_t q = 0;
#pragma unroll
    for (int i = 0; i < 4; i++) {
        const float t = x[i] + m;
        q |= (uint32_t)(sc > 0.0f ? (int)clampf(rintf(t / sc), 0.0f, 15.0f) : 0) << (4 * i);
    }
    st_any<uint16_t>(b + 16 + v / 2, (uint16_t)q);
}

__device__ __forceinline__ void encode_q5_k(const float *x, int v, uint8_t *b)
{
    const float scl = group_maxabs<8>(x) / 15.0f;
    float maxs = 0.0f;
    if (scl > maxs) maxs = scl;
    maxs = group_max<64>(maxs);
    const uint32_t d16 = f2h_rne(maxs / 63.0f);
    const float df = h2f_exact(d16);
    const int ls = df > 0.0f ? (int)clampf(rintf(scl / df), 0.0f, 63.0f) : 0;
    put_k_header(b, v, d16, 0u, ls, 0);
    const float sc = df * (float)ls;
    uint32_t lo = 0, hi = 0;
#pragma unroll
    for (int i = 0; i < 4; i++) {
        const int q = sc > 0.0f ? (int)clampf(rintf(x[i] / sc), -16.0f, 15.0f) + 16 : 16;
        lo |= (uint32_t)(q & 15) << (4 * i);
        hi |= (uint32_t)(q >> 4 & 1) << i;
    }
    st_any<uint16_t>(b + 48 + v / 2, (uint16_t)lo);
    hi |= __shfl_xor(hi, 1, 64) << 4;
    if ((v & 4) == 0) b[16 + v / 8] = (uint8_t)hi;
}

__device__ __forceinline__ void encode_q6_k(const float *x, int v, uint8_t *b)
{
    const float scl = group_maxabs<4>(x) / 31.0f;
    float maxs = 0.0f;
    if (scl > maxs) maxs = scl;
    maxs = group_max<64>(maxs);
    const uint32_t d16 = f2h_rne(maxs / 127.0f);
    const float df = h2f_exact(d16);
    const int ls = df > 0.0f ? (int)clampf(rintf(scl / df), -128.0f, 127.0f) : 0;
    const float sc = df * (float)ls;
    uint32_t lo = 0, hi = 0;
#pragma unroll
    for (int i = 0; i < 4; i++) {
        const int q = sc > 0.0f ? (int)clampf(rintf(x[i] / sc), -32.0f, 31.0f) + 32 : 32;
        lo |= (uint32_t)(q & 15) << (4 * i);
        hi |= (uint32_t)(q >> 4 & 3) << (2 * i);
    }
    st_any<uint16_t>(b + v / 2, (uint16_t)lo);
    b[128 + v / 4] = (uint8_t)hi;
    if ((v & 15) == 0) b[192 + v / 16] = (uint8_t)(int8_t)ls;
    if (v == 0) st_any<uint16_t>(b + 208, (uint16_t)d16);
}

// n is a multiple of the block size; F16 has blocks of one element.
template <int T>
__global__ void k_quantize(const float *__restrict__ x, int64_t n, uint8_t *__restrict__ out)
{
    constexpr int E = Type<T>::enc;
    const int64_t e0 = E * ((int64_t)blockIdx.x * blockDim.x + threadIdx.x);
    if (e0 >= n) return;   // whole groups of lanes: blocks are multiples of 32 elements
    uint8_t *b = out + e0 / Type<T>::elems * Type<T>::bytes;
    const int v = (int)(e0 % Type<T>::elems);
    float f[E];
    if (e0 + E <= n && ((uintptr_t)x & 15) == 0) {
#pragma unroll
        for (int i = 0; i < E; i += 4) {
            const float4 q = *(const float4 *)(x + e0 + i);
            f[i] = q.x, f[i + 1] = q.y, f[i + 2] = q.z, f[i + 3] = q.w;
        }
    } else {
#pragma unroll
        for (int i = 0; i < E; i++) f[i] = e0 + i < n ? x[e0 + i] : 0.0f;
    }
    if constexpr (T == SMX_TYPE_Q4_K) {
        encode_q4_k(f, v, b);
    } else if constexpr (T == SMX_TYPE_Q5_K) {
        encode_q5_k(f, v, b);
    } else if constexpr (T == SMX_TYPE_Q6_K) {
        encode_q6_k(f, v, b);
    } else if constexpr (T == SMX_TYPE_F16) {
        if (e0 + 4 <= n) {
            st_any<uint64_t>(b, (uint64_t)(f2h_rne(f[0]) | f2h_rne(f[1]) << 16) |
                                    (uint64_t)(f2h_rne(f[2]) | f2h_rne(f[3]) << 16) << 32);
        } else {
            for (int i = 0; e0 + i < n; i++) st_any<uint16_t>(b + 2 * i, (uint16_t)f2h_rne(f[i]));
        }
    } else {
        encode32<T>(f, v, b);
    }
}

__device__ __forceinline__ uint64_t splitmix64(uint64_t z)
{
    z += 0x9E3779B97F4A7C15ull;
    z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
    z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
    return z ^ (z >> 31);
}

__global__ void k_fill_normal(uint64_t seed, int64_t n, float std, float *__restrict__ out)
{
    const int64_t p = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;   // pair index
    if (2 * p >= n) return;
    uint64_t r = splitmix64(seed * 0xD1B54A32D192ED03ull + (uint64_t)p);
    float u1 = (float)((r >> 40) + 1) * 5.9604644775390625e-08f;
    float u2 = (float)(r & 0xFFFFFFu) * 5.9604644775390625e-08f;
    float rad = sqrtf(-2.0f * logf(u1));
    float th = 6.283185307179586f * u2;
    out[2 * p] = std * (rad * cosf(th));
    if (2 * p + 1 < n) out[2 * p + 1] = std * (rad * sinf(th));
}

// ---- GGUF -> backend layout ------------------------------------------------------------------
__global__ void k_repack(int fmt, const uint8_t *__restrict__ src, int64_t rows, int nb,
                         uint8_t *__restrict__ dq, uint16_t *__restrict__ dd, int64_t row_off,
                         int64_t row_step)
{
    const int64_t idx = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (idx >= rows * nb) return;
    const int64_t r = idx / nb;
    const int b = (int)(idx % nb);
    const int64_t dr = row_off + r * row_step;
    const int gb = fmt_gguf_bytes(fmt), mb = fmt_main_bytes(fmt);
    const uint8_t *s = src + idx * gb;
    uint8_t *o = dq + (dr * nb + b) * mb;
    if (fmt == FMT_F16 || fmt == FMT_F32) {
        for (int i = 0; i < mb; i++) o[i] = s[i];
    } else if (fmt == FMT_SQ8 || fmt == FMT_SQ4) {
        ((uint32_t *)dd)[dr * nb + b] = (uint32_t)s[0] | ((uint32_t)s[1] << 8) | ((uint32_t)s[2] << 16) |
                                        ((uint32_t)s[3] << 24);
        for (int i = 0; i < mb; i++) o[i] = s[4 + i];
    } else if (fmt == FMT_Q4_0 || fmt == FMT_Q8_0) {
        dd[dr * nb + b] = (uint16_t)ld_u16(s);
        for (int i = 0; i < mb; i++) o[i] = s[2 + i];
    } else if (fmt == FMT_Q4_K) {
        for (int i = 0; i < 144; i++) o[i] = s[i];
    } else if (fmt == FMT_Q5_K) {
        for (int i = 0; i < 16; i++) o[i] = s[i];
        for (int i = 0; i < 128; i++) o[48 + i] = s[48 + i];
        const uint8_t *qh = s + 16;
        for (int j = 0; j < 8; j++)
            for (int k = 0; k < 4; k++) {
                uint32_t byte = 0;
                for (int g = 0; g < 4; g++)
                    for (int p = 0; p < 2; p++) {
                        int v = 32 * j + 8 * g + 2 * k + p;
                        byte |= ((qh[v >> 3] >> (v & 7)) & 1u) << (2 * g + p);
                    }
                o[16 + 4 * j + k] = (uint8_t)byte;
            }
    } else {   // Q6_K
        for (int i = 0; i < 128; i++) o[i] = s[i];
        for (int i = 0; i < 16; i++) o[192 + i] = s[192 + i];
        dd[dr * nb + b] = (uint16_t)ld_u16(s + 208);
        const uint8_t *qh = s + 128;
        for (int c = 0; c < 8; c++)
            for (int p = 0; p < 2; p++)
                for (int k = 0; k < 4; k++) {
                    uint32_t byte = 0;
                    for (int g = 0; g < 4; g++) {
                        int v = 32 * c + 8 * g + 2 * k + p;
                        byte |= ((qh[v >> 2] >> (2 * (v & 3))) & 3u) << (2 * g);
                    }
                    o[128 + 8 * c + 4 * p + k] = (uint8_t)byte;
                }
    }
}

template <int F>
__global__ void k_dequant_smx(WView w, int64_t row0, int64_t nrows, float *__restrict__ out)
{
    const int nch = (int)(w.cols / 32);
    const int64_t idx = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (idx >= nrows * nch) return;
    const int64_t r = idx / nch;
    const int c = (int)(idx % nch);
    float y[32];
    decode_chunk_exact<F>(w, row0 + r, c, y);
    float *o = out + r * w.cols + (int64_t)c * 32;
#pragma unroll
    for (int i = 0; i < 32; i += 4) *(float4 *)(o + i) = make_float4(y[i], y[i + 1], y[i + 2], y[i + 3]);
}

unsigned grid_for(int64_t n) { return (unsigned)((n + kThreads - 1) / kThreads); }

template <typename F>
hipError_t by_type(int type, F f)
{
    switch (type) {
    case SMX_TYPE_F32: f(std::integral_constant<int, SMX_TYPE_F32>{}); break;
    case SMX_TYPE_F16: f(std::integral_constant<int, SMX_TYPE_F16>{}); break;
    case SMX_TYPE_Q4_0: f(std::integral_constant<int, SMX_TYPE_Q4_0>{}); break;
    case SMX_TYPE_Q8_0: f(std::integral_constant<int, SMX_TYPE_Q8_0>{}); break;
    case SMX_TYPE_Q4_K: f(std::integral_constant<int, SMX_TYPE_Q4_K>{}); break;
    case SMX_TYPE_Q5_K: f(std::integral_constant<int, SMX_TYPE_Q5_K>{}); break;
    case SMX_TYPE_Q6_K: f(std::integral_constant<int, SMX_TYPE_Q6_K>{}); break;
    case SMX_TYPE_SMQ_Q8: f(std::integral_constant<int, SMX_TYPE_SMQ_Q8>{}); break;
    case SMX_TYPE_SMQ_Q4: f(std::integral_constant<int, SMX_TYPE_SMQ_Q4>{}); break;
    default: return hipErrorInvalidValue;
    }
    return hipGetLastError();
}

}  // namespace

int fmt_from_type(int type)
{
    switch (type) {
    case SMX_TYPE_Q4_0: return FMT_Q4_0;
    case SMX_TYPE_Q8_0: return FMT_Q8_0;
    case SMX_TYPE_Q4_K: return FMT_Q4_K;
    case SMX_TYPE_Q5_K: return FMT_Q5_K;
    case SMX_TYPE_Q6_K: return FMT_Q6_K;
    case SMX_TYPE_F16: return FMT_F16;
    case SMX_TYPE_F32: return FMT_F32;
    case SMX_TYPE_SMQ_Q8: return FMT_SQ8;
    case SMX_TYPE_SMQ_Q4: return FMT_SQ4;
    default: return -1;
    }
}

// Elements per launch of a codec: at four per thread, half of the 2^32 threads above which a launch does
// not run them all.
constexpr int64_t kLaunchElems = (int64_t)1 << 33;

hipError_t launch_dequant_gguf(int type, const void *blocks, int64_t n, float *out, hipStream_t s)
{
    if (n == 0) return hipSuccess;
    return by_type(type, [&](auto t) {
        constexpr int T = decltype(t)::value;
        for (int64_t e = 0; e < n; e += kLaunchElems) {
            const int64_t m = n - e < kLaunchElems ? n - e : kLaunchElems;
            hipLaunchKernelGGL((k_dequant_gguf<T>), dim3(grid_for((m + 3) / 4)), dim3(kThreads), 0, s,
                               (const uint8_t *)blocks + e / Type<T>::elems * Type<T>::bytes, m, out + e);
        }
    });
}

hipError_t launch_quantize_gguf(int type, const float *x, int64_t n, void *blocks, hipStream_t s)
{
    if (n == 0) return hipSuccess;
    return by_type(type, [&](auto t) {
        constexpr int T = decltype(t)::value;
        if constexpr (T != SMX_TYPE_F32)
            for (int64_t e = 0; e < n; e += kLaunchElems) {
                const int64_t m = n - e < kLaunchElems ? n - e : kLaunchElems;
                hipLaunchKernelGGL((k_quantize<T>), dim3(grid_for((m + Type<T>::enc - 1) / Type<T>::enc)), dim3(kThreads), 0, s, x + e, m,
                                   (uint8_t *)blocks + e / Type<T>::elems * Type<T>::bytes);
            }
    });
}

hipError_t launch_fill_normal(uint64_t seed, int64_t n, float std, float *out, hipStream_t s)
{
    const int64_t pairs = (n + 1) / 2;
    if (pairs == 0) return hipSuccess;
    hipLaunchKernelGGL(k_fill_normal, dim3(grid_for(pairs)), dim3(kThreads), 0, s, seed, n, std, out);
    return hipGetLastError();
}

hipError_t launch_repack(int fmt, const uint8_t *gguf, int64_t rows, int64_t cols, uint8_t *dst_q,
                         uint16_t *dst_d, int64_t dst_rows, int64_t row_off, int64_t row_step,
                         hipStream_t s)
{
    (void)dst_rows;
    const int nb = (int)(cols / fmt_block_elems(fmt));
    const int64_t total = rows * nb;
    if (total == 0) return hipSuccess;
    hipLaunchKernelGGL(k_repack, dim3(grid_for(total)), dim3(kThreads), 0, s, fmt, gguf, rows, nb,
                       dst_q, dst_d, row_off, row_step);
    return hipGetLastError();
}

hipError_t launch_dequant_smx(const WView &w, int64_t row0, int64_t nrows, float *out, hipStream_t s)
{
    const int f = w.fmt;
    const int64_t total = nrows * (w.cols / 32);
    if (total == 0) return hipSuccess;
    const dim3 g(grid_for(total)), b(kThreads);
    switch (f) {
    case FMT_Q4_0: hipLaunchKernelGGL(k_dequant_smx<FMT_Q4_0>, g, b, 0, s, w, row0, nrows, out); break;
    case FMT_Q8_0: hipLaunchKernelGGL(k_dequant_smx<FMT_Q8_0>, g, b, 0, s, w, row0, nrows, out); break;
    case FMT_Q4_K: hipLaunchKernelGGL(k_dequant_smx<FMT_Q4_K>, g, b, 0, s, w, row0, nrows, out); break;
    case FMT_Q5_K: hipLaunchKernelGGL(k_dequant_smx<FMT_Q5_K>, g, b, 0, s, w, row0, nrows, out); break;
    case FMT_Q6_K: hipLaunchKernelGGL(k_dequant_smx<FMT_Q6_K>, g, b, 0, s, w, row0, nrows, out); break;
    case FMT_F16: hipLaunchKernelGGL(k_dequant_smx<FMT_F16>, g, b, 0, s, w, row0, nrows, out); break;
    case FMT_F32: hipLaunchKernelGGL(k_dequant_smx<FMT_F32>, g, b, 0, s, w, row0, nrows, out); break;
    case FMT_SQ8: hipLaunchKernelGGL(k_dequant_smx<FMT_SQ8>, g, b, 0, s, w, row0, nrows, out); break;
    case FMT_SQ4: hipLaunchKernelGGL(k_dequant_smx<FMT_SQ4>, g, b, 0, s, w, row0, nrows, out); break;
    default: return hipErrorInvalidValue;
    }
    return hipGetLastError();
}

}  // namespace smx

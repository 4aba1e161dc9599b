// k_sample.hip -- next-token sampling on the device, in the reference's pipeline order
// (InferenceSession.SampleNextToken, InferenceSession.cs:565-606):
//   1. repetition / presence / frequency penalties over the recent context (:765-843)
//   2. temperature: logits * (1 / T) (:741-763)
//   3. top-k: keep logits >= the k-th largest (:628-664)
//   4. softmax: exp(l - max) / sum over the finite logits (:666-706)
//   5. top-p: keep the largest probabilities whose running sum first reaches p, renormalise
//      by 1 / sum (:845-912, NormalizeProbabilities :969-1010)
//   6. min-p: zero probabilities below max * min_p, renormalise (:914-936)
//   7. sample: the first index whose running (double) sum of probabilities reaches u (:708-724)
// Selections are exact: the k-th largest logit and the top-p threshold are found by binary
// search over the float bit patterns.  Where the reference sorts, ties at the cutoff are all
// kept here (the reference's unstable Array.Sort keeps an arbitrary subset of them), and sums
// run in the order of a tree or scan rather than in sorted or index order.
//
// One workgroup of 1024 threads.  What bounds it is the chain of passes over the vocabulary: 63
// passes with a block reduction each, over global memory, took 380 us for 32000 tokens, whose 256 KB
// one compute unit moves in about 3.  So the values stay in LDS (above 32768 also in registers, above
// 65536 in the probs array), and the searches run over a short list of candidates in one wave, without
// a barrier: everything at or above the k-th largest of the 1024 per-thread maxima, which is never above
// the k-th largest value.  Top-k up to 192 searches the list of the logits, top-p the list of the 192
// largest probabilities (whose sum says whether the threshold is among them); what does not fit the
// list (ties, a flat distribution, fewer than k finite logits, infinities) is searched over all
// values.  Calls with penalties, top-k 40 and top-p 0.9, before -> now, us: 32000 tokens 375 -> 40 (the
// kernel 21), 50257 552 -> 50, 70000 693 -> 85.  Top-p 0.9 alone, not in the list: 32000 200 -> 88,
// 70000 361 -> 158; top-k 400: 221 -> 77, 403 -> 139.
#include <type_traits>
#include <utility>

#include "smx_device.h"
#include "smx_internal.h"

namespace smx {

namespace {

constexpr int kT = 1024;
constexpr int kW = kT / 64;
constexpr int kList = 256;          // candidates: four per lane of one wave
constexpr int kListK = 192;         // rank aimed at: the bound lets in about k^2 / 2048 more, and ties
constexpr int kCtx = 2048;          // penalty window kept in LDS
constexpr int kRows = 32;           // values per thread in LDS, and as many in registers
constexpr int kNear = 2 * kRows * kT;   // largest vocabulary held so
constexpr int kSeg = 16;            // draw: segments per wave

// Order-preserving unsigned image of a float (larger float -> larger key).
__device__ __forceinline__ uint32_t fkey(float f)
{
    const uint32_t u = __float_as_uint(f);
    return (u & 0x80000000u) ? ~u : (u | 0x80000000u);
}

__device__ __forceinline__ float kfloat(uint32_t k)
{
    return __uint_as_float((k & 0x80000000u) ? (k & 0x7FFFFFFFu) : ~k);
}

constexpr uint32_t kAboveNegInf = 0x00800000u;   // fkey(-inf) + 1
constexpr uint32_t kPosZero = 0x80000000u;       // fkey(+0); -0 is one below and equal to it as a float

static_assert(kRows * kT / 32 == kT, "one word of penalty bits per thread");

struct SampleShared {
    uint32_t bits[kRows * kT / 32];   // penalised tokens whose values are in registers
    int32_t ctx[kCtx];
    uint32_t top[kT];                    // per-thread maxima
    int idx[kList];                      // candidates as found
    float val[kList];
    uint32_t rank[kList];
    float sval[kList];                   // candidates by value
    int spos[kList], sidx[kList];        // their places by index; candidates by index
    double cum[kW * kSeg];
    float redf[2][kW];
    uint32_t redu[2][kW];
    uint32_t count, bound, key;
    int tok, ok;
};

// The n values; f gets the row (1024 j, uniform) of value row + tid, and the value.  Each thread keeps
// its own: the first 32 rows in LDS (loops over them are short code, where 32 registers per thread made
// 150 KB of it), R more in registers; all in mem for R < 0.
template <int R>
struct Vals {
    float v[R > 0 ? R : 1];
    float *lds, *mem;
    int n;

    template <typename F>
    __device__ __forceinline__ void each(F f)   // x = f(row, x)
    {
        const int tid = threadIdx.x, m = R < 0 ? n : min(n, kRows * kT);
        float *__restrict__ p = R < 0 ? mem : lds;
#pragma unroll 4
        for (int r = 0; r + tid < m; r += kT) (p + r)[tid] = f(r, (p + r)[tid]);
        if constexpr (R > 0) rows([&](int row, float &x) { x = f(row, x); }, std::make_integer_sequence<int, R>{});
    }

    template <typename F>
    __device__ __forceinline__ void scan(F f)
    {
        const int tid = threadIdx.x, m = R < 0 ? n : min(n, kRows * kT);
        const float *p = R < 0 ? mem : lds;
#pragma unroll 4
        for (int r = 0; r + tid < m; r += kT) f(r, (p + r)[tid]);
        if constexpr (R > 0) rows([&](int row, float &x) { f(row, x); }, std::make_integer_sequence<int, R>{});
    }

    // The first pass, x = src * scale: 16 loads in flight per thread.
    __device__ __forceinline__ void load(const float *__restrict__ src, float scale)
    {
        const int tid = threadIdx.x, m = R < 0 ? n : min(n, kRows * kT);
        float *__restrict__ p = R < 0 ? mem : lds;
        for (int r = 0; r < m; r += 16 * kT) {
            float t[16];
#pragma unroll
            for (int j = 0; j < 16; j++) t[j] = src[min(r + j * kT + tid, n - 1)];
#pragma unroll
            for (int j = 0; j < 16; j++)
                if (r + j * kT + tid < m) (p + r + j * kT)[tid] = t[j] * scale;
        }
        if constexpr (R > 0)
            rows([&](int row, float &x) { x = (src + row)[tid] * scale; }, std::make_integer_sequence<int, R>{});
    }

    template <typename F, int... J>
    __device__ __forceinline__ void rows(F f, std::integer_sequence<int, J...>)
    {
        int tid = threadIdx.x;
        asm volatile("" : "+v"(tid));   // else the rows' masks are kept from one call to the next
        (one(f, (kRows + J) * kT, tid, v[J]), ...);
    }

private:
    // Nothing is shared between rows or calls: masks, keys and addresses kept for later, or rows
    // interleaved, take more registers than there are.
    template <typename F>
    __device__ __forceinline__ void one(F f, int row, int tid, float &x)
    {
        asm volatile("" : "+v"(x));
        if (tid < n - row) f(row, x);
        __builtin_amdgcn_sched_barrier(0);
    }
};

// Sums over the workgroup of a float per thread and a count per wave: one barrier per call, two
// buffers in turn.
struct BlockSum {
    SampleShared &S;
    int turn = 0;
    float f;
    uint32_t c;

    __device__ __forceinline__ explicit BlockSum(SampleShared &s) : S(s) {}

    __device__ __forceinline__ void operator()(float v, uint32_t wave_count = 0)
    {
        const float w = wave_sum_uniform(v);
        if ((threadIdx.x & 63) == 0) {
            S.redf[turn][threadIdx.x >> 6] = w;
            S.redu[turn][threadIdx.x >> 6] = wave_count;
        }
        __syncthreads();
        f = 0.0f;
        c = 0;
#pragma unroll
        for (int i = 0; i < kW; i++) {
            f += S.redf[turn][i];
            c += S.redu[turn][i];
        }
        turn ^= 1;
    }
};

template <typename T>
__device__ __forceinline__ T wave_scan(T v, int lane)   // inclusive
{
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
        const T t = __shfl_up(v, o, 64);
        if (lane >= o) v += t;
    }
    return v;
}

// Penalties: each distinct token of the window w once, by the first thread that holds it.  The new
// value, times scale, goes to where the old one is held; for one in registers it goes to mem[t], marked by a bit.
// (logits[t] is read before anything is stored for token t, so mem may be the logits' own buffer.)
template <int R>
__device__ __forceinline__ void penalise(SampleShared &S, Vals<R> &x, const float *__restrict__ logits,
                                         const int32_t *w, int nw, const smx_sampling &sp, float scale)
{
    for (int j = threadIdx.x; j < nw; j += kT) {
        const int t = w[j];
        if (t < 0 || t >= x.n) continue;
        float l = logits[t];
        int count = 0, before = 0;
        // independent reads, 256 at a time; a wave whose tokens have all been seen earlier goes no further
        // (2000 tokens of a vocabulary of 33: 163 -> 52 us)
        for (int q0 = 0; q0 < nw && !__all(before); q0 += 256) {
#pragma unroll 8
            for (int q = q0; q < min(nw, q0 + 256); q++) {
                const int eq = w[q] == t;
                count += eq;
                before += q < j ? eq : 0;
            }
        }
        if (before) continue;
        if (sp.repetition_penalty != 1.0f) l = l > 0.0f ? l / sp.repetition_penalty : l * sp.repetition_penalty;
        if (sp.presence_penalty != 0.0f) l = l - sp.presence_penalty;
        if (sp.frequency_penalty != 0.0f) l = l - (float)count * sp.frequency_penalty;
        l = l * scale;
        if (R < 0) {
            x.mem[t] = l;
        } else if (R == 0 || t < kRows * kT) {
            x.lds[t] = l;
        } else {
            x.mem[t] = l;
            atomicOr(&S.bits[(t - kRows * kT) >> 5], 1u << (t & 31));
        }
    }
}

// S.idx / S.val: the values (in no order) whose key is at least S.bound, a key that at least k values
// reach if that many are finite; S.count of them, of which the first kList are stored.  -0 comes in
// where +0 does, and -infinity never.
template <int R>
__device__ __forceinline__ void make_list(SampleShared &S, Vals<R> &x, int k)
{
    const int tid = threadIdx.x;
    uint32_t top = 0;
    x.scan([&](int, float f) { top = max(top, fkey(f)); });
    S.top[tid] = top;
    if (tid == 0) S.count = 0;
    __syncthreads();
    if (tid < 64) {
        uint32_t m[kT / 64], key = 0;
#pragma unroll
        for (int q = 0; q < kT / 64; q++) m[q] = S.top[tid + 64 * q];
        // the upper half of the key: a bound need not be a value
        if (k <= 64) {   // 256 groups are enough: about k^2 / 512 more than k get in
#pragma unroll
            for (int q = 0; q < 4; q++) m[q] = max(max(m[q], m[q + 4]), max(m[q + 8], m[q + 12]));
            for (int b = 31; b >= 16; b--) {
                const uint32_t cand = key | (1u << b);
                int c = 0;
#pragma unroll
                for (int q = 0; q < 4; q++) c += __popcll(__ballot(m[q] >= cand));
                if (c >= k) key = cand;
            }
        } else {
            for (int b = 31; b >= 16; b--) {
                const uint32_t cand = key | (1u << b);
                int c = 0;
#pragma unroll
                for (int q = 0; q < kT / 64; q++) c += __popcll(__ballot(m[q] >= cand));
                if (c >= k) key = cand;
            }
        }
        if (key == kPosZero) key--;
        if (tid == 0) S.bound = max(key, kAboveNegInf);
    }
    __syncthreads();
    const uint32_t bound = S.bound;
    x.scan([&](int row, float f) {
        if (fkey(f) >= bound) {
            const uint32_t at = atomicAdd(&S.count, 1u);
            if (at < kList) {
                S.idx[at] = row + tid;
                S.val[at] = f;
            }
        }
    });
    __syncthreads();
}

// Sorts the list: by value from the largest (S.sval; S.spos is the place by index), and by index
// (S.sidx).  By counting, four threads to a candidate.
__device__ __forceinline__ void sort_list(SampleShared &S, int C)
{
    const int at = threadIdx.x & (kList - 1);
    if (threadIdx.x < kList) S.rank[at] = 0;
    __syncthreads();
    int i = 0;
    float f = 0.0f;
    if (at < C) {
        i = S.idx[at];
        f = S.val[at];
        const uint32_t key = fkey(f);
        uint32_t r = 0;   // rank by value, and by index in the upper half
#pragma unroll 4
        for (int o = threadIdx.x / kList; o < C; o += kT / kList) {
            const uint32_t other = fkey(S.val[o]);
            const int oi = S.idx[o];
            r += (other > key || (other == key && oi < i) ? 1u : 0u) + (oi < i ? 0x10000u : 0u);
        }
        atomicAdd(&S.rank[at], r);
    }
    __syncthreads();
    if (at < C && threadIdx.x < kList) {
        const uint32_t r = S.rank[at];
        S.sval[r & 0xFFFFu] = f;
        S.spos[r & 0xFFFFu] = (int)(r >> 16);
        S.sidx[r >> 16] = i;
    }
    __syncthreads();
}

// The stages from top-k (LOGITS) or top-p on over the sorted list, by the first wave, one to four
// candidates per lane from the largest on.  False (and nothing written) if the list does not settle
// the result.  The probabilities of the candidates go to probs, the token to S.tok.
template <bool LOGITS>
__device__ __forceinline__ bool finish_list(SampleShared &S, int C, int n, const smx_sampling &sp, double u,
                                            float *__restrict__ probs)
{
    const int lane = threadIdx.x, nq = (C + 63) >> 6;
    float p[4];
#pragma unroll
    for (int q = 0; q < 4; q++) p[q] = lane + 64 * q < C ? S.sval[lane + 64 * q] : 0.0f;
    if (LOGITS) {
        const float kth = S.sval[sp.top_k - 1];
        bool on[4];
        float mx = -INFINITY;
#pragma unroll
        for (int q = 0; q < 4; q++) {
            on[q] = lane + 64 * q < C && p[q] >= kth;
            if (on[q]) mx = fmaxf(mx, p[q]);
        }
        mx = wave_max(mx);
        float s = 0.0f;
#pragma unroll
        for (int q = 0; q < 4; q++) {
            p[q] = on[q] ? expf(p[q] - mx) : 0.0f;
            s += p[q];
        }
        s = wave_sum_uniform(s);
        if (!(s > 0.0f)) return false;   // infinities, NaN
#pragma unroll
        for (int q = 0; q < 4; q++) p[q] = p[q] / s;
    }
    const auto renorm = [&]() {
        const float s = wave_sum_uniform((p[0] + p[1]) + (p[2] + p[3]));
        if (s > 0.0f) {
            const float inv = 1.0f / s;
#pragma unroll
            for (int q = 0; q < 4; q++) p[q] = p[q] * inv;
        }
    };
    if (sp.top_p < 1.0) {
        // the first place at which the running sum reaches top_p
        float run = 0.0f, t = 0.0f;
        bool found = false;
#pragma unroll
        for (int q = 0; q < 4; q++) {
            if (q < nq && !found) {
                const float c = run + wave_scan(p[q], lane);
                const uint64_t hit = __ballot((double)c >= sp.top_p && c > 0.0f);   // float sum against the double TopP
                if (hit) {
                    t = __shfl(p[q], __ffsll((unsigned long long)hit) - 1, 64);
                    found = true;
                }
                run = __shfl(c, 63, 64);
            }
        }
        if (!LOGITS) {
            // the threshold has to lie above everything that the list leaves out: above its smallest
            // probability by more than expf and the division can be out of order
            if (!(t > S.sval[C - 1] * 1.00001f)) return false;
        }
#pragma unroll
        for (int q = 0; q < 4; q++) p[q] = p[q] >= t ? p[q] : 0.0f;
        renorm();
    }
    if (sp.min_p > 0.0f) {
        const float thr = wave_max(fmaxf(fmaxf(p[0], p[1]), fmaxf(p[2], p[3]))) * sp.min_p;
#pragma unroll
        for (int q = 0; q < 4; q++) p[q] = p[q] < thr ? 0.0f : p[q];
        renorm();
    }
    // from the order of values to that of indices
#pragma unroll
    for (int q = 0; q < 4; q++)
        if (lane + 64 * q < C) S.val[S.spos[lane + 64 * q]] = p[q];
    __threadfence_block();
    __builtin_amdgcn_wave_barrier();
    double run = 0.0;
    int tok = u <= 0.0 ? 0 : n - 1;   // the running sum at index 0 is at least 0
    bool found = u <= 0.0;
#pragma unroll
    for (int q = 0; q < 4; q++) {
        const int at = lane + 64 * q;
        if (q < nq) {
            const float v = at < C ? S.val[at] : 0.0f;
            const int i = at < C ? S.sidx[at] : 0;
            if (at < C) probs[i] = v;
            if (!found) {
                const double c = run + wave_scan((double)v, lane);
                const uint64_t hit = __ballot(v > 0.0f && c >= u);   // lanes' sums are rounded apart
                if (hit) {
                    tok = __shfl(i, __ffsll((unsigned long long)hit) - 1, 64);
                    found = true;
                }
                run = __shfl(c, 63, 64);
            }
        }
    }
    if (lane == 0) S.tok = tok;
    return true;
}

// Tries the list of the k largest values: true if it gave the result (probs and S.tok are written).
template <bool LOGITS, int R>
__device__ __forceinline__ bool by_list(SampleShared &S, Vals<R> &x, int k, const smx_sampling &sp, double u)
{
    make_list<R>(S, x, k);
    // fewer than k finite logits: the k-th largest is not in the list
    if (S.count > kList || S.count == 0 || (LOGITS && (int)S.count < k)) return false;
    const int C = (int)S.count;
    const uint32_t bound = S.bound;
    sort_list(S, C);
    const auto others = [&](int row, float f) {
        if (fkey(f) < bound) (x.mem + row)[threadIdx.x] = 0.0f;
    };
    if (threadIdx.x < 64) {
        const bool ok = finish_list<LOGITS>(S, C, x.n, sp, u, x.mem);
        if (threadIdx.x == 0) S.ok = ok;
    } else if (R >= 0) {
        x.scan(others);   // beside the first wave's search: mem is not read again if that fails
    }
    __syncthreads();
    if (!S.ok) return false;
    if (R < 0) {
        // candidates now hold probabilities in mem: mark them by index instead of by value
        for (int i = threadIdx.x; i < x.n; i += kT) {
            int at = 0, end = C;
            while (at < end) {
                const int mid = (at + end) >> 1;
                if (S.sidx[mid] < i) at = mid + 1;
                else end = mid;
            }
            if (at >= C || S.sidx[at] != i) x.mem[i] = 0.0f;
        }
    } else if (threadIdx.x < 64) {
        x.scan(others);
    }
    return true;
}

// p * (1 / sum) when sum > 0 (NormalizeProbabilities, InferenceSession.cs:969-1010)
template <int R>
__device__ __forceinline__ void renorm(Vals<R> &x, float sum)
{
    if (sum > 0.0f) {
        const float inv = 1.0f / sum;
        x.each([&](int, float p) { return p * inv; });
    }
}

// The pipeline; every thread of the workgroup calls it, and thread 0 receives the token.
template <int R>
__device__ __forceinline__ int sample_pipeline(const float *__restrict__ logits, int n, const int32_t *__restrict__ ctx, int n_ctx,
                               const smx_sampling &sp, double u, float *__restrict__ probs)
{
    __shared__ SampleShared S;
    extern __shared__ float values[];
    const int tid = threadIdx.x;
    Vals<R> x;
    x.lds = values;
    x.mem = probs;
    x.n = n;
    // 2. temperature, applied to each value as it is first held (x 1 is exact).  Where the values are held in
    // the logits' own buffer (probs == logits), the penalties still need the unscaled ones: scaled after them
    const bool penalties = sp.repetition_penalty != 1.0f || sp.presence_penalty != 0.0f || sp.frequency_penalty != 0.0f;
    const bool late = R < 0 && penalties && logits == probs;
    const float temp = sp.temperature != 1.0f ? 1.0f / sp.temperature : 1.0f, scale = late ? 1.0f : temp;
    x.load(logits, scale);

    // 1. penalties
    if (penalties) {
        const int win = sp.repetition_window > 0 ? sp.repetition_window : min(n_ctx, 256);
        const int start = max(0, n_ctx - win), nw = n_ctx - start;
        if (R > 0) S.bits[tid] = 0;
        if (nw <= kCtx)
            for (int j = tid; j < nw; j += kT) S.ctx[j] = ctx[start + j];
        __syncthreads();
        if (nw <= kCtx) penalise(S, x, logits, S.ctx, nw, sp, scale);
        else penalise(S, x, logits, ctx + start, nw, sp, scale);
        __threadfence_block();
        __syncthreads();
        if constexpr (R > 0)
            x.rows([&](int row, float &f) {
                if ((S.bits[((row - kRows * kT) >> 5) + (tid >> 5)] >> (tid & 31)) & 1u) f = (probs + row)[tid];
            }, std::make_integer_sequence<int, R>{});
        if (late) x.each([&](int, float l) { return l * temp; });
    }
    BlockSum sum(S);
    // 3. top-k
    if (sp.top_k > 0 && sp.top_k < n) {
        if (sp.top_k <= kListK && by_list<true, R>(S, x, sp.top_k, sp, u)) return S.tok;
        // the largest key with >= k at or above, bit by bit; with exactly k there, the smallest of these
        x.each([&](int, float f) { return __uint_as_float(fkey(f)); });
        uint32_t key = 0;
        for (int b = 31; b >= 0; b--) {
            const uint32_t cand = key | (1u << b);
            uint32_t c = 0;
            x.scan([&](int, float f) { c += __float_as_uint(f) >= cand; });
#pragma unroll
            for (int o = 32; o > 0; o >>= 1) c += __shfl_xor(c, o, 64);
            sum(0.0f, c);
            if (sum.c >= (uint32_t)sp.top_k) key = cand;
            if (sum.c == (uint32_t)sp.top_k) break;
        }
        uint32_t low = 0xFFFFFFFFu;
        x.scan([&](int, float f) {
            if (__float_as_uint(f) >= key) low = min(low, __float_as_uint(f));
        });
#pragma unroll
        for (int o = 32; o > 0; o >>= 1) low = min(low, __shfl_xor(low, o, 64));
        __syncthreads();
        if ((tid & 63) == 0) S.redu[0][tid >> 6] = low;
        __syncthreads();
#pragma unroll
        for (int i = 0; i < kW; i++) low = min(low, S.redu[0][i]);
        __syncthreads();
        const float kth = kfloat(low);
        x.each([&](int, float f) {
            const float l = kfloat(__float_as_uint(f));
            return l >= kth ? l : -INFINITY;
        });
    }
    // 4. softmax over the finite logits
    float mx = -INFINITY;
    x.scan([&](int, float l) {
        if (l != -INFINITY) mx = fmaxf(mx, l);
    });
    mx = block_max<kW>(mx, S.redf[0]);
    __syncthreads();
    float s = 0.0f;
    x.each([&](int, float l) {
        const float e = l != -INFINITY ? expf(l - mx) : 0.0f;
        s += e;
        return e;
    });
    sum(s);
    const float total = sum.f;
    if (total > 0.0f) x.each([&](int, float e) { return e / total; });
    // 5. top-p: threshold t = the largest probability with sum(p >= t) >= top_p
    if (sp.top_p < 1.0) {
        if (total > 0.0f && by_list<false, R>(S, x, kListK, sp, u)) return S.tok;
        // probabilities are >= 0: their bit patterns order like the values.  Between lo (reached) and
        // hi (not reached) until the list holds what lies between.
        uint32_t key = 0, c_lo = (uint32_t)n, c_hi = 0;
        float hi = INFINITY, f_hi = 0.0f;
        for (int b = 30; b >= 0; b--) {
            const uint32_t cand = key | (1u << b);
            const float t = __uint_as_float(cand);
            float c = 0.0f;
            uint32_t m = 0;
            x.scan([&](int, float p) {
                c += p >= t ? p : 0.0f;
                m += p >= t;
            });
#pragma unroll
            for (int o = 32; o > 0; o >>= 1) m += __shfl_xor(m, o, 64);
            sum(c, m);
            if ((double)sum.f >= sp.top_p && sum.f > 0.0f) {   // float sum against the double TopP
                key = cand;
                c_lo = sum.c;
            } else {
                hi = t;
                f_hi = sum.f;
                c_hi = sum.c;
            }
            if (c_lo - c_hi <= (uint32_t)kList && b > 0) {
                const float lo = __uint_as_float(key);
                __syncthreads();
                if (tid == 0) S.count = 0;
                __syncthreads();
                x.scan([&](int, float p) {
                    if (p >= lo && !(p >= hi)) S.val[atomicAdd(&S.count, 1u)] = p;
                });
                __syncthreads();
                if (tid < 64) {
                    float p[4];
#pragma unroll
                    for (int q = 0; q < 4; q++) p[q] = tid + 64 * q < (int)S.count ? S.val[tid + 64 * q] : 0.0f;
                    while (--b >= 0) {
                        const uint32_t cd = key | (1u << b);
                        const float tt = __uint_as_float(cd);
                        float cc = 0.0f;
#pragma unroll
                        for (int q = 0; q < 4; q++) cc += p[q] >= tt ? p[q] : 0.0f;
                        const float f = f_hi + wave_sum_uniform(cc);
                        if ((double)f >= sp.top_p && f > 0.0f) key = cd;
                    }
                    if (tid == 0) S.key = key;
                }
                __syncthreads();
                key = S.key;
                break;
            }
        }
        const float t = __uint_as_float(key);
        s = 0.0f;
        x.each([&](int, float p) {
            p = p >= t ? p : 0.0f;
            s += p;
            return p;
        });
        sum(s);
        renorm(x, sum.f);
    }
    // 6. min-p
    if (sp.min_p > 0.0f) {
        float pm = 0.0f;
        x.scan([&](int, float p) { pm = fmaxf(pm, p); });
        __syncthreads();
        pm = block_max<kW>(pm, S.redf[0]);
        __syncthreads();
        const float thr = pm * sp.min_p;
        s = 0.0f;
        x.each([&](int, float p) {
            p = p < thr ? 0.0f : p;
            s += p;
            return p;
        });
        sum(s);
        renorm(x, sum.f);
    }
    if (R >= 0) x.scan([&](int row, float p) { (probs + row)[tid] = p; });
    __threadfence_block();
    __syncthreads();
    // 7. inverse-CDF draw: sums of contiguous segments, then the segment in which u is reached
    // (a segment is a chain of a load and a reduction, so each wave takes no more of them than 64 values
    // each make: the kernel with 1000 values 15.2 -> 6.4 us)
    const int lane = tid & 63, w = tid >> 6;
    const int rows = (n + 63) / 64, segs = min(kSeg, (rows + kW - 1) / kW);
    const int seg = (rows + kW * segs - 1) / (kW * segs) * 64;
    if (tid >= kW * segs && tid < kW * kSeg) S.cum[tid] = 0.0;
#pragma unroll 4
    for (int k = 0; k < segs; k++) {
        const int64_t a = (int64_t)(w * segs + k) * seg, e = min((int64_t)n, a + seg);
        double c = 0.0;
        for (int64_t i = a + lane; i < e; i += 64) c += (double)probs[i];
#pragma unroll
        for (int o = 32; o > 0; o >>= 1) c += __shfl_xor(c, o, 64);
        if (lane == 0) S.cum[w * segs + k] = c;
    }
    __syncthreads();
    if (tid < 64) {
        double c[4], own = 0.0;
#pragma unroll
        for (int q = 0; q < 4; q++) {
            own += S.cum[4 * lane + q];
            c[q] = own;
        }
        const double before = wave_scan(own, lane) - own;
        int first = 4;
#pragma unroll
        for (int q = 3; q >= 0; q--)
            if (before + c[q] >= u) first = q;
        const uint64_t hit = __ballot(first < 4);
        int tok = n - 1;   // SampleFromProbs' fallback
        if (hit) {
            const int l = __ffsll((unsigned long long)hit) - 1;
            const int sg = 4 * l + __shfl(first, l, 64);
            double r = 0.0;
            for (int q = 0; q < sg; q++) r += S.cum[q];
            // past the end of the segment only where rounding left its sum short of u
            for (int64_t a = (int64_t)sg * seg; a < n; a += 64) {
                const float p = a + lane < n ? probs[a + lane] : 0.0f;
                const double v = r + wave_scan((double)p, lane);
                const uint64_t h = __ballot(v >= u && (p > 0.0f || (u <= 0.0 && a + lane == 0)));
                if (h) {
                    tok = (int)a + __ffsll((unsigned long long)h) - 1;
                    break;
                }
                r = __shfl(v, 63, 64);
            }
        }
        return tok;
    }
    return 0;
}

template <int R>
__global__ __launch_bounds__(kT) void k_sample(const float *__restrict__ logits, int n,
                                               const int32_t *__restrict__ ctx, int n_ctx, smx_sampling sp,
                                               double u, float *__restrict__ probs, int32_t *__restrict__ out)
{
    const int tok = sample_pipeline<R>(logits, n, ctx, n_ctx, sp, u, probs);
    if (threadIdx.x == 0) *out = tok;
}

// End of a sampled decode step: the context is tokens[0..pos] (prompt and generated so far),
// u = the st->counter-th draw of the stream seeded by st->seed; the token is appended at
// tokens[pos + 1], the position advanced and the draw counter incremented.
template <int R>
__global__ __launch_bounds__(kT) void k_sample_step(const float *__restrict__ logits, int n,
                                                    int32_t *__restrict__ tokens, int32_t *__restrict__ pos,
                                                    SampleState *__restrict__ st, float *__restrict__ probs)
{
    const int p = *pos;
    const smx_sampling sp = st->params;
    const double u = uniform_draw(st->seed, st->counter);
    const int tok = sample_pipeline<R>(logits, n, tokens, p + 1, sp, u, probs);
    if (threadIdx.x == 0) {
        tokens[p + 1] = tok;
        *pos = p + 1;
        st->counter = st->counter + 1;
    }
}

// Members of a lockstep step (one logits row each), after k_argmax_rows has appended each
// member's greedy token at tokens[pos] and advanced pos: a member with sampling on replaces
// that token (and the next step's input id) with the pipeline's draw over tokens[0..pos-1].
template <int R>
__global__ __launch_bounds__(kT) void k_sample_rows(const float *__restrict__ logits, int n, int64_t stride,
                                                    int32_t *const *__restrict__ tok_arr,
                                                    const int32_t *__restrict__ pos, int32_t *__restrict__ ids,
                                                    SampleState *__restrict__ st, const int32_t *__restrict__ on,
                                                    float *__restrict__ probs)
{
    const int r = blockIdx.x;
    if (!on[r]) return;   // the same for the whole workgroup
    const int p = pos[r];
    const smx_sampling sp = st[r].params;
    const double u = uniform_draw(st[r].seed, st[r].counter);
    const int tok = sample_pipeline<R>(logits + (size_t)r * stride, n, tok_arr[r], p, sp, u, probs + (size_t)r * n);
    if (threadIdx.x == 0) {
        tok_arr[r][p] = tok;
        ids[r] = tok;
        st[r].counter = st[r].counter + 1;
    }
}

// The values stay on the compute unit up to 65536 of them.
template <typename F>
hipError_t by_size(int n, F f)
{
    if (n <= kRows * kT) return f(std::integral_constant<int, 0>{});
    if (n <= kNear) return f(std::integral_constant<int, kRows>{});
    return f(std::integral_constant<int, -1>{});
}

template <int R, typename... P, typename... A>
hipError_t launch_pipeline(void (*kernel)(P...), int blocks, int n, hipStream_t s, A... args)
{
    const size_t lds = R < 0 ? 0 : sizeof(float) * (size_t)min(n, kRows * kT);
    if (R >= 0) {
        const hipError_t e = hipFuncSetAttribute((const void *)kernel, hipFuncAttributeMaxDynamicSharedMemorySize,
                                                 kRows * kT * (int)sizeof(float));
        if (e != hipSuccess) return e;
    }
    hipLaunchKernelGGL(kernel, dim3(blocks), dim3(kT), lds, s, args...);
    return hipGetLastError();
}

}  // namespace

hipError_t launch_sample_rows(const float *logits, int n, int64_t stride, int M, int32_t *const *tok_arr,
                              const int32_t *pos, int32_t *ids, SampleState *st, const int32_t *on, float *probs,
                              hipStream_t s)
{
    return by_size(n, [&](auto r) {
        constexpr int R = decltype(r)::value;
        return launch_pipeline<R>(k_sample_rows<R>, M, n, s, logits, n, stride, tok_arr, pos, ids, st, on, probs);
    });
}

hipError_t launch_sample(const float *logits, int n, const int32_t *ctx, int n_ctx, const smx_sampling &sp,
                         double u, float *probs, int32_t *out, hipStream_t s)
{
    return by_size(n, [&](auto r) {
        constexpr int R = decltype(r)::value;
        return launch_pipeline<R>(k_sample<R>, 1, n, s, logits, n, ctx, n_ctx, sp, u, probs, out);
    });
}

hipError_t launch_sample_step(const float *logits, int n, int32_t *tokens, int32_t *pos, SampleState *st,
                              float *probs, hipStream_t s)
{
    return by_size(n, [&](auto r) {
        constexpr int R = decltype(r)::value;
        return launch_pipeline<R>(k_sample_step<R>, 1, n, s, logits, n, tokens, pos, st, probs);
    });
}

}  // namespace smx

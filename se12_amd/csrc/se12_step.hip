// Decode-step kernels of a Gemma-2 style decoder (one new token per
// sequence), so that a step is a handful of launches around the fused
// products instead of ~80 small framework kernels per layer. They take the
// products' FP32 outputs (or BF16, for a BF16 baseline) and reproduce the
// rounding sequence of the eager step: every framework BF16 op rounds its
// FP32 result to BF16 (round to nearest even), so do these, op by op.
//
//   rmsnorm        norm(x) = x * rsqrt(mean(x^2) + eps) * (1 + w), FP32 math,
//                  BF16 result; mode 1 fuses t = bf16(y), x = bf16(x + norm(t, w1)),
//                  h = norm(x, w2) (post-norm, residual add, next pre-norm)
//   attention      two launches over (sequence, KV head, 64-position chunk):
//                  q/k/v to BF16, rotary embedding, K/V written to the caches
//                  at `pos`, scores against positions 0..pos (or the sliding
//                  window), scaling, tanh soft-capping; then softmax in FP32
//                  and the weighted sum of V, chunk partials added in order
//   gelu_mul       bf16(gelu_tanh(bf16(g)) * bf16(u))
//   logits_argmax  final soft-capping of the logits and the greedy token,
//                  blocks over vocabulary slices, the last one picks
//   advance        pos += 1, step += 1
//
// Every kernel is latency-bound at decode sizes (a few KB to a few MB per
// launch): each thread issues all its loads before using any of them, and
// the caches are read 16 bytes per lane.
//
// The caches: K transposed [batch, kv_heads, head_dim, max_len] (so that a
// framework batched product can read it as a contiguous right operand), V
// [batch, kv_heads, max_len, head_dim], both BF16.
//
// Cross-block results (attention partials, argmax partials) are written with
// device-scope stores and counted in per-row arrival counters; the last block
// reads them back with device-scope loads in a fixed order and resets its
// counter, so results are deterministic and no memset is needed between calls.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <algorithm>

#include "se12_step.h"
#include "se12_step_math.hpp"

namespace se12step {

// element i of an FP32 or BF16 tensor, rounded to BF16 (the framework's
// `.to(torch.bfloat16)` of a product output)
template <int DT>
__device__ __forceinline__ float load_as_bf16(const void* p, int64_t i) {
    if constexpr (DT == SE12_STEP_F32)
        return round_bf16(static_cast<const float*>(p)[i]);
    else
        return bf16_to_f(static_cast<const uint16_t*>(p)[i]);
}

__device__ __forceinline__ float load_as_bf16(const void* p, int dtype, int64_t i) {
    return dtype == SE12_STEP_F32 ? load_as_bf16<SE12_STEP_F32>(p, i) : load_as_bf16<SE12_STEP_BF16>(p, i);
}

// 8 BF16 values from 16 bytes
__device__ __forceinline__ void unpack8(const uint4 r, float* v) {
    const uint32_t w[4] = {r.x, r.y, r.z, r.w};
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        v[2 * i] = __uint_as_float(w[i] << 16);
        v[2 * i + 1] = __uint_as_float(w[i] & 0xFFFF0000u);
    }
}

// (value, index) with the larger value, the smaller index on a tie; NaN
// ranks above every number (torch.argmax's order), so a row of NaNs still
// gives an index in the vocabulary (its first NaN) and never the initial one
__device__ __forceinline__ void keep_first_max(float& bv, int& bi, float v, int i) {
    const bool vn = v != v, bn = bv != bv;
    if (vn ? (!bn || i < bi) : (!bn && (v > bv || (v == bv && i < bi)))) {
        bv = v;
        bi = i;
    }
}

// ---------------------------------------------------------------------------
// rmsnorm: one block per row, kNormPer elements per thread, all loads first
// ---------------------------------------------------------------------------

constexpr int kNormPer = 8;
constexpr int kNormMaxThreads = 1024;

struct NormArgs {
    const void* in;
    int64_t in_stride;
    const uint16_t* w1;
    const uint16_t* res_in;  // mode 1; residual itself, or another tensor
    uint16_t* residual;
    const uint16_t* w2;
    uint16_t* out;
    int hidden;
    float eps, in_scale;
};

template <int DT, int MODE>
__global__ __launch_bounds__(kNormMaxThreads) void rmsnorm_kernel(NormArgs a) {
    __shared__ float sh[17];
    const int r = blockIdx.x, t = threadIdx.x, nt = blockDim.x;
    const int64_t base = (int64_t)r * a.in_stride, rbase = (int64_t)r * a.hidden;
    float x[kNormPer], w1[kNormPer], res[kNormPer], w2[kNormPer];
#pragma unroll
    for (int k = 0; k < kNormPer; ++k) {
        const int i = t + k * nt;
        const int ic = i < a.hidden ? i : a.hidden - 1;  // clamped: every load is issued unconditionally
        x[k] = load_as_bf16<DT>(a.in, base + ic);
        w1[k] = bf16_to_f(a.w1[ic]);
        if constexpr (MODE == 1) {
            res[k] = bf16_to_f(a.res_in[rbase + ic]);
            w2[k] = bf16_to_f(a.w2[ic]);
        }
    }
    float ss = 0.0f;
#pragma unroll
    for (int k = 0; k < kNormPer; ++k) {
        if constexpr (MODE == 0)
            if (a.in_scale != 0.0f) x[k] = round_bf16(x[k] * a.in_scale);  // scaled embedding row
        if (t + k * nt < a.hidden) ss += x[k] * x[k];
    }
    const float inv = rms_inv(block_sum(ss, sh), a.hidden, a.eps);
    if constexpr (MODE == 0) {
#pragma unroll
        for (int k = 0; k < kNormPer; ++k) {
            const int i = t + k * nt;
            if (i < a.hidden) {
                if (a.residual) a.residual[rbase + i] = f_to_bf16(x[k]);
                a.out[rbase + i] = f_to_bf16(rms_scale(x[k], inv, w1[k]));
            }
        }
        return;
    }
    // mode 1: residual += norm(bf16(in), w1); out = norm(residual, w2)
    float ss2 = 0.0f;
#pragma unroll
    for (int k = 0; k < kNormPer; ++k) {
        const float n1 = round_bf16(rms_scale(x[k], inv, w1[k]));
        res[k] = round_bf16(res[k] + n1);
        if (t + k * nt < a.hidden) ss2 += res[k] * res[k];
    }
    const float inv2 = rms_inv(block_sum(ss2, sh), a.hidden, a.eps);
#pragma unroll
    for (int k = 0; k < kNormPer; ++k) {
        const int i = t + k * nt;
        if (i < a.hidden) {
            a.residual[rbase + i] = f_to_bf16(res[k]);
            a.out[rbase + i] = f_to_bf16(rms_scale(res[k], inv2, w2[k]));
        }
    }
}

// ---------------------------------------------------------------------------
// attention: the positions 0..pos are cut into chunks of 64; one block per
// (sequence, KV head, chunk) in each of two launches:
//   scores  rotary embedding of q (and of k, in the block holding pos, which
//           also writes the new K/V slot), the chunk's scores for the G query
//           heads of the KV head, the chunk's max m_c and sum l_c of
//           exp(s - m_c);
//   pv      one block per (sequence, KV head, 32 head-dim columns, span of
//           positions): the global max M = max m_c and sum S =
//           sum l_c exp(m_c - M), the probabilities p = bf16(exp(s - M) / S)
//           (softmax in FP32, rounded as the framework rounds it) and the
//           sum p . V of its columns over its span in FP32. A span covers
//           1024 positions (256 x G query heads of registers per thread),
//           so caches up to that need one span and write the output
//           directly; longer ones write partial sums that the last block of
//           a (sequence, KV head, columns) adds in span order. Splitting
//           the columns instead of the positions keeps a short cache's
//           blocks free of that cross-block reduction.
// ---------------------------------------------------------------------------

constexpr int kChunk = 64;
constexpr int kAttnThreads = 256;
constexpr int kMaxHeadDim = 256;

struct AttnArgs {
    const void* q;
    const void* k;
    const void* v;
    int dtype;
    int64_t q_stride, kv_stride;
    uint16_t* kt;            // [B, kvh, d, L]
    uint16_t* vc;            // [B, kvh, L, d]
    const float* inv_freq;   // [d / 2]
    const int64_t* pos;
    uint16_t* out;           // [B, heads * d]
    float* scores;           // [B, heads, chunks * 64]
    float* stats;            // [B, heads, chunks, 2]: m_c, l_c
    float* partial;          // [B, heads, spans <= chunks, d]
    int* counters;           // [B * kvh * column blocks], zero between launches
    int heads, kvh, d, max_len, chunks;
    float scaling, softcap;
    int window;
};

__device__ __forceinline__ int window_lo(int p, int window) {
    return window > 0 ? (p - window + 1 > 0 ? p - window + 1 : 0) : 0;
}

// a wave-uniform 64-bit value held in a vector register, as a scalar
__device__ __forceinline__ int64_t uniform_i64(int64_t v) {
    const uint32_t lo = (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)v);
    const uint32_t hi = (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)((uint64_t)v >> 32));
    return (int64_t)(((uint64_t)hi << 32) | lo);
}

// A block barrier for LDS data that leaves global loads in flight.
__device__ __forceinline__ void lds_barrier() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }

// Makes the wave wait for a loaded value here: issued before a branch on the
// position, loads would otherwise be sunk past it and wait for it.
__device__ __forceinline__ void pin(float v) { asm volatile("" ::"v"(v)); }
__device__ __forceinline__ void pin(const uint4& v) { asm volatile("" ::"v"(v.x), "v"(v.y), "v"(v.z), "v"(v.w)); }

// Rotary embedding, with the framework's roundings, of the G queries and
// the key whose element t thread t < d holds in x[0..G]; the rotated values
// land in y and in qk ([G + 1][d] in LDS). Every thread of the block calls
// it (two barriers).
template <int G>
__device__ __forceinline__ void rotate_qk(float* qk, const float (&x)[G + 1], float fr, int p, int d, int t,
                                          float (&y)[G + 1]) {
    const int half = d / 2;
    if (t < d) {
#pragma unroll
        for (int h = 0; h <= G; ++h) qk[h * d + t] = x[h];
    }
    __syncthreads();
    if (t < d) {
        const float freq = (float)p * fr;
        const float cs = round_bf16(cosf(freq)), sn = round_bf16(sinf(freq));
#pragma unroll
        for (int h = 0; h <= G; ++h) {
            const float* xv = qk + h * d;
            const float rot = t < half ? -xv[t + half] : xv[t - half];
            y[h] = round_bf16(round_bf16(xv[t] * cs) + round_bf16(rot * sn));
        }
    }
    __syncthreads();
    if (t < d) {
#pragma unroll
        for (int h = 0; h <= G; ++h) qk[h * d + t] = y[h];
    }
}

// One 64-position chunk of keys against the G rotated queries in qk, for a
// team of 4 waves (tt = thread in the team): lane group pg = tt % 8 takes 8
// consecutive positions jgl.. (one 16-byte load per head-dim element), the
// 32 slices es = tt / 8 every 32nd element. The key at position p comes from
// qk (its cache slot is written in the same launch). The wave's 8 slices
// are summed (lane bits 3..5) and lanes 0..7 write the wave's sums to red
// ([4 waves][G][64]).
template <int G>
__device__ __forceinline__ void chunk_key_dots(const uint4 (&raw)[kMaxHeadDim / 32], const float* qk, int d, int tt,
                                               int jgl, int p, float* red) {
    const int pg = tt & 7, es = tt >> 3, tw = tt >> 6;
    float acc[8][G];
#pragma unroll
    for (int m = 0; m < 8; ++m)
#pragma unroll
        for (int h = 0; h < G; ++h) acc[m][h] = 0.0f;
#pragma unroll
    for (int i = 0; i < kMaxHeadDim / 32; ++i) {
        const int e = es + 32 * i;
        if (e < d) {
            float kv[8];
            unpack8(raw[i], kv);
#pragma unroll
            for (int m = 0; m < 8; ++m)
                if (jgl + m == p) kv[m] = qk[G * d + e];
#pragma unroll
            for (int h = 0; h < G; ++h) {
                const float qv = qk[h * d + e];
#pragma unroll
                for (int m = 0; m < 8; ++m) acc[m][h] += qv * kv[m];
            }
        }
    }
#pragma unroll
    for (int m = 0; m < 8; ++m)
#pragma unroll
        for (int h = 0; h < G; ++h) {
            float v = acc[m][h];
            v += __shfl_xor(v, 8, 64);
            v += __shfl_xor(v, 16, 64);
            v += __shfl_xor(v, 32, 64);
            acc[m][h] = v;
        }
    if ((tt & 63) < 8) {
#pragma unroll
        for (int h = 0; h < G; ++h)
#pragma unroll
            for (int m = 0; m < 8; ++m) red[(tw * G + h) * kChunk + 8 * pg + m] = acc[m][h];
    }
}

// For thread t < 64 (one wave): the score of position j0 + t for each head
// (the 4 waves' dots in order, scaling, soft-capping, -inf outside
// [lo, p]) and the chunk's max m and sum l of exp(score - m).
template <int G, int STRIDE = kChunk>
__device__ __forceinline__ void chunk_scores(const float* red, const AttnArgs& a, int t, int j0, int p, int lo,
                                             float (&sc)[G], float (&m)[G], float (&l)[G]) {
    const int jq = j0 + t;
    const bool valid = jq <= p && jq >= lo;
#pragma unroll
    for (int h = 0; h < G; ++h) {
        const float dot = red[(0 * G + h) * STRIDE + t] + red[(1 * G + h) * STRIDE + t] +
                          red[(2 * G + h) * STRIDE + t] + red[(3 * G + h) * STRIDE + t];
        float v = round_bf16(round_bf16(dot) * a.scaling);
        if (a.softcap > 0.0f) v = round_bf16(round_bf16(tanhf(round_bf16(v / a.softcap))) * a.softcap);
        if (!valid) v = -INFINITY;
        sc[h] = v;
        m[h] = wave_max(v);                      // >= 1 valid position per chunk
        l[h] = wave_sum(valid ? expf(v - m[h]) : 0.0f);
    }
}

template <int G, int DT>
__global__ __launch_bounds__(kAttnThreads) void attn_scores_kernel(const int64_t* pos, const void* q, const void* k,
                                                                   uint16_t* kt, int32_t d_, int32_t L_, int32_t kvh,
                                                                   int32_t q_stride, int32_t kv_stride, AttnArgs ga) {
    // the leading arguments (preloaded into SGPRs by the dispatch) are the
    // ones the first loads need; the rest arrive by scalar loads meanwhile
    AttnArgs a = ga;
    a.pos = pos;
    a.q = q;
    a.k = k;
    a.kt = kt;
    a.d = d_;
    a.max_len = L_;
    a.kvh = kvh;
    a.q_stride = q_stride;
    a.kv_stride = kv_stride;
    __shared__ float qk[(G + 1) * kMaxHeadDim];   // rotated q of the G heads, then k
    __shared__ float red[4 * G * kChunk];         // per wave: G x 64 partial dot products
    const int t = threadIdx.x, lane = t & 63, w = t >> 6;
    const int kvb = blockIdx.x;                    // b * kvh + kh
    const int b = kvb / a.kvh, kh = kvb % a.kvh;
    const int c = blockIdx.y, j0 = c * kChunk;
    const int d = a.d, half = d / 2;
    const int L = a.max_len;

    // Every load whose address does not depend on the position goes out
    // together with the position's: q and k of the new token (to BF16) and
    // the chunk of the key cache, all from preloaded arguments; then v and
    // the rotary frequency, whose pointers are scalar loads. The position is
    // a vector load, so that waiting for those scalar loads does not wait for
    // it. Lane group pg = 8 consecutive positions read as one 16-byte load
    // per head-dim element; the 32 slices es take every 32nd element.
    const int64_t p64v = __hip_atomic_load(a.pos, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    float xq[G], xk = 0.0f, vv = 0.0f, fr = 0.0f;
    const int tc = t < d ? t : d - 1;
#pragma unroll
    for (int h = 0; h < G; ++h)
        xq[h] = load_as_bf16<DT>(a.q, (int64_t)b * a.q_stride + (int64_t)(kh * G + h) * d + tc);
    xk = load_as_bf16<DT>(a.k, (int64_t)b * a.kv_stride + (int64_t)kh * d + tc);
    const int pg = t & 7, es = t >> 3;
    const int jg = j0 + 8 * pg;
    const int jgl = jg + 8 <= L ? jg : L - 8;     // L % 8 == 0: a group is wholly in or out
    const uint16_t* kb = a.kt + (int64_t)kvb * d * L + jgl;
    uint4 raw[kMaxHeadDim / 32];
#pragma unroll
    for (int i = 0; i < kMaxHeadDim / 32; ++i) {
        const int e = es + 32 * i;
        raw[i] = *reinterpret_cast<const uint4*>(kb + (int64_t)(e < d ? e : d - 1) * L);
    }
    __builtin_amdgcn_sched_barrier(0);  // the loads above go out first
    vv = load_as_bf16<DT>(a.v, (int64_t)b * a.kv_stride + (int64_t)kh * d + tc);
    fr = a.inv_freq[tc % half];
#pragma unroll
    for (int h = 0; h < G; ++h) pin(xq[h]);
    pin(xk);
#pragma unroll
    for (int i = 0; i < kMaxHeadDim / 32; ++i) pin(raw[i]);
    const int64_t p64 = uniform_i64(p64v);

    if (p64 < 0 || p64 >= a.max_len) return;
    const int p = (int)p64, lo = window_lo(p, a.window);
    if (j0 > p || j0 + kChunk <= lo) return;
    const bool holds_p = p < j0 + kChunk;

    float x[G + 1], y[G + 1];
#pragma unroll
    for (int h = 0; h < G; ++h) x[h] = xq[h];
    x[G] = xk;
    rotate_qk<G>(qk, x, fr, p, d, t, y);
    if (t < d && holds_p) {
        a.kt[((int64_t)kvb * d + t) * L + p] = f_to_bf16(y[G]);
        a.vc[((int64_t)kvb * L + p) * d + t] = f_to_bf16(vv);
    }
    __syncthreads();
    chunk_key_dots<G>(raw, qk, d, t, jgl, p, red);
    __syncthreads();
    if (t < kChunk) {
        float sc[G], m[G], l[G];
        chunk_scores<G>(red, a, t, j0, p, lo, sc, m, l);
        const int64_t lp = (int64_t)a.chunks * kChunk;
#pragma unroll
        for (int h = 0; h < G; ++h) {
            const int64_t row = (int64_t)b * a.kvh * G + kh * G + h;
            a.scores[row * lp + j0 + t] = sc[h];
            if (t == 0) {
                a.stats[(row * a.chunks + c) * 2 + 0] = m[h];
                a.stats[(row * a.chunks + c) * 2 + 1] = l[h];
            }
        }
    }
}

// weighted V: positions per thread (all loads in flight at once) and the
// span of positions of one block
constexpr int kPvCols = 32;
template <int G>
constexpr int pv_per_thread() { return G <= 2 ? 16 : 32 / G; }
template <int G>
constexpr int pv_span() { return (kAttnThreads / (kPvCols / 8)) * pv_per_thread<G>(); }

template <int G>
__global__ __launch_bounds__(kAttnThreads) void attn_pv_kernel(const int64_t* pos, const float* stats, const float* scores,
                                                               const uint16_t* vc, int32_t d_, int32_t L_, int32_t kvh,
                                                               int32_t chunks, AttnArgs ga) {
    // the leading arguments (preloaded into SGPRs by the dispatch) are the
    // ones the first loads need; the rest arrive by scalar loads meanwhile
    AttnArgs a = ga;
    a.pos = pos;
    a.stats = const_cast<float*>(stats);
    a.scores = const_cast<float*>(scores);
    a.vc = const_cast<uint16_t*>(vc);
    a.d = d_;
    a.max_len = L_;
    a.kvh = kvh;
    a.chunks = chunks;
    constexpr int P = pv_per_thread<G>();
    constexpr int kSpan = pv_span<G>();
    __shared__ float ms[2 * G];
    __shared__ float red[4 * G * kPvCols];        // per wave: G x 32 column sums
    __shared__ int flag;
    const int t = threadIdx.x, lane = t & 63, w = t >> 6;
    const int kvb = blockIdx.x;
    const int b = kvb / a.kvh, kh = kvb % a.kvh;
    const int cb = blockIdx.y, sp = blockIdx.z;
    const int d = a.d, L = a.max_len;
    const int64_t obase = (int64_t)b * a.kvh * G * d + (int64_t)kh * G * d;
    const int64_t row0 = (int64_t)b * a.kvh * G + kh * G;
    const int64_t lp = (int64_t)a.chunks * kChunk;
    // thread: 8-column group cq of the block's 32 columns, position slice ps
    const int cq = t & 3, ps = t >> 2;
    const int e0 = cb * kPvCols + 8 * cq;
    const uint16_t* vb = a.vc + (int64_t)kvb * L * d + (e0 < d ? e0 : d - 8);
    const int jb = sp * kSpan;

    // Every load whose address does not depend on the position goes out
    // together with the position's: the statistics of the first 64 chunks of
    // the wave's heads (lane = chunk), and the span's V rows and scores.
    const int64_t p64v = __hip_atomic_load(a.pos, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);  // a vector load
    constexpr int kHeadsPerWave = (G + 3) / 4;
    float sm[kHeadsPerWave], sl[kHeadsPerWave];
    const int cl = lane < a.chunks ? lane : a.chunks - 1;
#pragma unroll
    for (int k = 0; k < kHeadsPerWave; ++k) {
        const int h = w + 4 * k < G ? w + 4 * k : G - 1;
        const float* st = a.stats + (row0 + h) * a.chunks * 2;
        sm[k] = st[cl * 2];
        sl[k] = st[cl * 2 + 1];
    }
    uint4 vr[P];
    float sc[P][G];
#pragma unroll
    for (int i = 0; i < P; ++i) {
        const int j = jb + ps + 64 * i;
        const int jc = j < L ? j : L - 1;
        vr[i] = *reinterpret_cast<const uint4*>(vb + (int64_t)jc * d);
#pragma unroll
        for (int h = 0; h < G; ++h) sc[i][h] = a.scores[(row0 + h) * lp + jc];
    }
#pragma unroll
    for (int k = 0; k < kHeadsPerWave; ++k) {
        pin(sm[k]);
        pin(sl[k]);
    }
#pragma unroll
    for (int i = 0; i < P; ++i) {
        pin(vr[i]);
#pragma unroll
        for (int h = 0; h < G; ++h) pin(sc[i][h]);
    }

    const int64_t p64 = uniform_i64(p64v);
    if (p64 < 0 || p64 >= L) {  // no cache slot: zeros, no cache or counter touched
        if (cb == 0 && sp == 0)
            for (int i = t; i < G * d; i += kAttnThreads) a.out[obase + i] = 0;
        return;
    }
    const int p = (int)p64, lo = window_lo(p, a.window);
    const int s_lo = lo / kSpan, s_hi = p / kSpan;
    if (sp < s_lo || sp > s_hi) return;
    const int c_lo = lo / kChunk, c_hi = p / kChunk;
    // global max and sum of each head over its chunks (one wave per head)
#pragma unroll
    for (int k = 0; k < kHeadsPerWave; ++k) {
        const int h = w + 4 * k;
        if (h >= G) break;
        const float* st = a.stats + (row0 + h) * a.chunks * 2;
        const bool mine = lane >= c_lo && lane <= c_hi;
        float m = mine ? sm[k] : -INFINITY;
        for (int cc = lane + 64; cc <= c_hi; cc += 64)
            if (cc >= c_lo) m = fmaxf(m, st[cc * 2]);
        m = wave_max(m);
        float s = mine ? sl[k] * expf(sm[k] - m) : 0.0f;
        for (int cc = lane + 64; cc <= c_hi; cc += 64)
            if (cc >= c_lo) s += st[cc * 2 + 1] * expf(st[cc * 2] - m);
        s = wave_sum(s);
        if (lane == 0) {
            ms[2 * h] = m;
            ms[2 * h + 1] = s;
        }
    }
    __syncthreads();
    float acc[8][G];
#pragma unroll
    for (int m = 0; m < 8; ++m)
#pragma unroll
        for (int h = 0; h < G; ++h) acc[m][h] = 0.0f;
#pragma unroll
    for (int i = 0; i < P; ++i) {
        const int j = jb + ps + 64 * i;
        if (j >= lo && j <= p) {   // V past pos may hold anything (0 x NaN)
            float v[8];
            unpack8(vr[i], v);
#pragma unroll
            for (int h = 0; h < G; ++h) {
                const float pr = round_bf16(expf(sc[i][h] - ms[2 * h]) / ms[2 * h + 1]);
#pragma unroll
                for (int m = 0; m < 8; ++m) acc[m][h] += pr * v[m];
            }
        }
    }
    // the 16 position slices of a wave (lane bits 2..5), then the 4 waves in order
#pragma unroll
    for (int m = 0; m < 8; ++m)
#pragma unroll
        for (int h = 0; h < G; ++h) {
            float v = acc[m][h];
            v += __shfl_xor(v, 4, 64);
            v += __shfl_xor(v, 8, 64);
            v += __shfl_xor(v, 16, 64);
            v += __shfl_xor(v, 32, 64);
            acc[m][h] = v;
        }
    if (lane < 4) {
#pragma unroll
        for (int h = 0; h < G; ++h)
#pragma unroll
            for (int m = 0; m < 8; ++m) red[(w * G + h) * kPvCols + 8 * cq + m] = acc[m][h];
    }
    __syncthreads();
    const int nspans = s_hi - s_lo + 1;
    const int h = t / kPvCols, e = cb * kPvCols + t % kPvCols;
    const bool owner = t < G * kPvCols && e < d;
    float o = 0.0f;
    if (owner)
        o = red[(0 * G + h) * kPvCols + t % kPvCols] + red[(1 * G + h) * kPvCols + t % kPvCols] +
            red[(2 * G + h) * kPvCols + t % kPvCols] + red[(3 * G + h) * kPvCols + t % kPvCols];
    if (nspans == 1) {
        if (owner) a.out[obase + h * d + e] = f_to_bf16(o);
        return;
    }
    // several spans: partial sums [row][span][d], the last block of the
    // (sequence, KV head, columns) adds them in span order
    float* part = a.partial + (row0 + h) * (int64_t)a.chunks * d;
    if (owner) __hip_atomic_store(&part[(int64_t)sp * d + e], o, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    int* counter = &a.counters[(int64_t)kvb * gridDim.y + cb];
    if (t == 0) {
        const int old = __hip_atomic_fetch_add(counter, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        flag = old == nspans - 1;
    }
    __syncthreads();
    if (!flag) return;
    if (owner) {
        float sum = 0.0f;
        for (int ss = s_lo; ss <= s_hi; ++ss)
            sum += __hip_atomic_load(&part[(int64_t)ss * d + e], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        a.out[obase + h * d + e] = f_to_bf16(sum);
    }
    if (t == 0) __hip_atomic_store(counter, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// ---------------------------------------------------------------------------
// attention over many positions: launches of kLongBlocks score blocks
// (sequences x KV heads x chunks) or more, e.g. a batch over a long cache. The
// blocks of the kernels above load their share of the cache before they know
// the position, one round trip less on a cache nearly all in use, but a launch
// of many blocks then reads the whole cache whatever part is in use, rotates q
// once per 64 positions, and computes each probability once per 8 columns.
// Here a block reads the position first (other blocks of the CU hide that),
// and the positions in use, not the cache's length, are cut among the grid's
// blocks:
//   scores  a run of units of 64 to 256 positions per block (by head_dim,
//           so that a unit is a few KB of keys per wave): q rotated once, the
//           next batch of keys in flight while one is used, a wave for each
//           of the unit's chunks at its end.
//   pv      a run of positions per block over all head-dim columns: whole
//           V rows per load, each probability computed once and shared
//           through LDS; the runs' FP32 sums meet as the spans above do.
// Bound by the cache's bytes in use. Two launches in a graph, cold cache, the
// short kernels above against these, in us at a full cache / position 3,000 or
// half / 300 / full with a window of an eighth:
//   8 seq x 8 KV heads x 256 x 1 query, 8,192 long  136/116/111/123 -> 126/57/18/30
//                            x 2                    152/123/114/129 -> 136/60/20/35
//                            x 8                    413/218/139/179 -> 273/122/38/72
//   32 x 8 x 128 x 2, 2,048 long                     86/ 75/ 68/ 72 ->  74/52/22/23
//   32 x 8 x  64 x 2, 4,096 long                    102/ 87/ 70/ 79 ->  73/58/19/22
//   1 x 1 x 256 x 8, 400,000 long                  1885/107/107/270 -> 490/41/36/168
// (136 us is 3.9 TB/s; the key rows are 16 KB apart, and a cache of 8,064
// takes 17 us less). Units of 128 / 256 at head_dim 256 took 60 / 62 us at
// position 3,000, 64 / 128 at head_dim 64 79 / 69; nontemporal loads 126 at a
// full cache but 40 and 97 on smaller ones.
// The grid is what the CUs hold at once: 1,024 blocks whatever the number of
// query heads took 298 us in the third line (2 blocks of 8 queries fit a CU)
// and 760 in the last, where each block of a wide grid also left a span of 64
// positions for one block to add up.
// The line between the two kernels: a short cache that is full is the case
// where reading the position first costs most. From kLongBlocks these kernels
// take at most 1.03 times the short ones there (2 queries 8 x 8 x 256 x 4,096:
// 81 -> 79 us, and 61 -> 20 at 300); on 1,152 blocks (9 x 8 x 256 x 1,024) 31
// -> 35 us at 2 queries and 68 -> 91 at 8. One query head per KV head leaves
// pv the least work per row, .91 to .98 of the short kernels' speed at 4,096
// blocks and 1.0 at kLongBlocks1; rows shorter than kLongDim leave most of a
// unit's lanes without elements (head_dim 8: .73 to .97).
// ---------------------------------------------------------------------------

constexpr int kLongBlocks = 4000, kLongBlocks1 = 5000;   // the second with one query head per KV head
constexpr int kLongDim = 32;
constexpr int kUnitLoads = 8;      // 16-byte loads of one batch per thread, two batches in flight
constexpr int kPvStep = 64;        // positions of one step of a pv block: 8 V rows per thread, two steps in flight

template <int G, int DT, int UNIT>
__global__ __launch_bounds__(kAttnThreads) void attn_scores_long_kernel(AttnArgs a) {
    __shared__ float qk[(G + 1) * kMaxHeadDim];
    __shared__ float red[4 * G * UNIT];
    const int t = threadIdx.x, lane = t & 63, w = __builtin_amdgcn_readfirstlane(t >> 6);
    const int kvb = blockIdx.x, b = kvb / a.kvh, kh = kvb % a.kvh;
    const int d = a.d, half = d / 2, L = a.max_len;
    const int64_t p64 = uniform_i64(__hip_atomic_load(a.pos, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT));
    if (p64 < 0 || p64 >= L) return;
    const int p = (int)p64, lo = window_lo(p, a.window);
    // units u0 .. u1 - 1 of the nu in use
    const int u_lo = lo / UNIT, nu = p / UNIT - u_lo + 1;
    const int Y = (int)gridDim.y, y = (int)blockIdx.y;
    const int u0 = u_lo + (int)((int64_t)y * nu / Y), u1 = u_lo + (int)((int64_t)(y + 1) * nu / Y);
    if (u0 >= u1) return;

    // lane group pg: 8 consecutive positions (UNIT contiguous positions of
    // one head-dim element's row per kLanes lanes); slice es: every
    // kSlices-th element, kUnitLoads of them in flight twice over
    constexpr int kLanes = UNIT / 8, kSlices = kAttnThreads / kLanes;
    const int pg = t % kLanes, es = t / kLanes;
    const int nb = (d + kSlices * kUnitLoads - 1) / (kSlices * kUnitLoads);   // load batches per unit
    auto load = [&](uint4 (&raw)[kUnitLoads], int u, int k) {
        const int jg = u * UNIT + 8 * pg;
        const uint16_t* kb = a.kt + (int64_t)kvb * d * L + (jg + 8 <= L ? jg : L - 8);
#pragma unroll
        for (int i = 0; i < kUnitLoads; ++i) {
            const int e = es + kSlices * (kUnitLoads * k + i);
            raw[i] = *reinterpret_cast<const uint4*>(kb + (int64_t)(e < d ? e : d - 1) * L);
        }
    };
    uint4 r0[kUnitLoads], r1[kUnitLoads];
    float x[G + 1], y0[G + 1];
    const int tc = t < d ? t : d - 1;
#pragma unroll
    for (int h = 0; h < G; ++h)
        x[h] = load_as_bf16<DT>(a.q, (int64_t)b * a.q_stride + (int64_t)(kh * G + h) * d + tc);
    x[G] = load_as_bf16<DT>(a.k, (int64_t)b * a.kv_stride + (int64_t)kh * d + tc);
    const float vv = load_as_bf16<DT>(a.v, (int64_t)b * a.kv_stride + (int64_t)kh * d + tc);
    const float fr = a.inv_freq[tc % half];
    load(r0, u0, 0);
    rotate_qk<G>(qk, x, fr, p, d, t, y0);
    if (t < d && u1 == u_lo + nu) {
        a.kt[((int64_t)kvb * d + t) * L + p] = f_to_bf16(y0[G]);
        a.vc[((int64_t)kvb * L + p) * d + t] = f_to_bf16(vv);
    }
    __syncthreads();
    float acc[8][G];
    auto clear = [&]() {
#pragma unroll
        for (int m = 0; m < 8; ++m)
#pragma unroll
            for (int h = 0; h < G; ++h) acc[m][h] = 0.0f;
    };
    auto dots = [&](const uint4 (&raw)[kUnitLoads], int u, int k) {
        const int jg = u * UNIT + 8 * pg, jgl = jg + 8 <= L ? jg : L - 8;
        const bool holds = p < (u + 1) * UNIT;   // block-uniform: the unit of the new token
#pragma unroll
        for (int i = 0; i < kUnitLoads; ++i) {
            const int e = es + kSlices * (kUnitLoads * k + i);
            if (e < d) {
                float kv[8];
                unpack8(raw[i], kv);
                if (holds) {
#pragma unroll
                    for (int m = 0; m < 8; ++m)
                        if (jgl + m == p) kv[m] = qk[G * d + e];
                }
#pragma unroll
                for (int h = 0; h < G; ++h) {
                    const float qv = qk[h * d + e];
#pragma unroll
                    for (int m = 0; m < 8; ++m) acc[m][h] += qv * kv[m];
                }
            }
        }
    };
    const int64_t lp = (int64_t)a.chunks * kChunk;
    const int64_t row0 = (int64_t)b * a.kvh * G + kh * G;
    // the unit's scores: the wave's two slices, then the four waves in order,
    // each wave taking one of the unit's chunks
    auto finish = [&](int u) {
#pragma unroll
        for (int h = 0; h < G; ++h)
#pragma unroll
            for (int m = 0; m < 8; ++m) {
                float v = acc[m][h];
#pragma unroll
                for (int o = kLanes; o < 64; o *= 2) v += __shfl_xor(v, o, 64);
                if (lane < kLanes) red[(w * G + h) * UNIT + 8 * pg + m] = v;
            }
        lds_barrier();
        const int c = u * (UNIT / kChunk) + w;
        if (w < UNIT / kChunk && c >= lo / kChunk && c <= p / kChunk) {
            float sc[G], m[G], l[G];
            chunk_scores<G, UNIT>(red + w * kChunk, a, lane, c * kChunk, p, lo, sc, m, l);
#pragma unroll
            for (int h = 0; h < G; ++h) {
                a.scores[(row0 + h) * lp + c * kChunk + lane] = sc[h];
                if (lane == 0) {
                    a.stats[((row0 + h) * a.chunks + c) * 2 + 0] = m[h];
                    a.stats[((row0 + h) * a.chunks + c) * 2 + 1] = l[h];
                }
            }
        }
        lds_barrier();
    };
    int u = u0, k = 0;
    auto step = [&](const uint4 (&cur)[kUnitLoads], uint4 (&next)[kUnitLoads]) {
        const bool last = k + 1 == nb;
        const int un = last ? u + 1 : u, kn = last ? 0 : k + 1;
        if (un < u1) load(next, un, kn);
        __builtin_amdgcn_sched_barrier(0);   // in flight while this batch is used
        if (k == 0) clear();
        dots(cur, u, k);
        if (last) finish(u);
        u = un;
        k = kn;
        return u < u1;
    };
    while (step(r0, r1) && step(r1, r0)) {
    }
}

template <int G>
__global__ __launch_bounds__(kAttnThreads) void attn_pv_long_kernel(AttnArgs a) {
    extern __shared__ __attribute__((aligned(16))) float lds[];  // [position slices][G][d] sums
    __shared__ float ms[2 * G];
    __shared__ float pr[2][G * kPvStep];
    __shared__ int flag;
    const int t = threadIdx.x, lane = t & 63, w = __builtin_amdgcn_readfirstlane(t >> 6);
    const int kvb = blockIdx.x, b = kvb / a.kvh, kh = kvb % a.kvh;
    const int d = a.d, L = a.max_len;
    const int Y = (int)gridDim.y, sp = (int)blockIdx.y;
    const int64_t obase = (int64_t)b * a.kvh * G * d + (int64_t)kh * G * d;
    const int64_t row0 = (int64_t)b * a.kvh * G + kh * G;
    const int64_t lp = (int64_t)a.chunks * kChunk;
    const int64_t p64 = uniform_i64(__hip_atomic_load(a.pos, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT));
    if (p64 < 0 || p64 >= L) {  // no cache slot: zeros, no cache or counter touched
        if (sp == 0)
            for (int i = t; i < G * d; i += kAttnThreads) a.out[obase + i] = 0;
        return;
    }
    const int p = (int)p64, lo = window_lo(p, a.window);
    // span sp of the positions in use: whole steps, the same for every block
    const int len = p - lo + 1;
    // (kPvStep at least, more on a wide grid: one block adds up the spans' sums)
    const int least = kPvStep * (Y > 128 ? Y / 128 : 1);
    const int even = ((len + Y - 1) / Y + kPvStep - 1) / kPvStep * kPvStep;
    const int span = even > least ? even : least;
    const int nspans = (len + span - 1) / span;
    if (sp >= nspans) return;
    const int j0 = lo + sp * span, j1 = j0 + span < p + 1 ? j0 + span : p + 1;

    // thread: columns 8 cq .. + 7 of position slice ps of rpp
    const int tpr = d / 8, rpp = kAttnThreads / tpr;
    const int cq = t % tpr, ps = t / tpr;
    const bool mine = ps < rpp;
    const uint16_t* vb = a.vc + (int64_t)kvb * L * d + 8 * cq;
    constexpr int kRows = kPvStep / 8;   // V rows per thread and step at head_dim 256 (fewer below)
    constexpr int kProbs = (G * kPvStep + kAttnThreads - 1) / kAttnThreads;
    const int rows = (kPvStep + rpp - 1) / rpp;
    auto load = [&](uint4 (&vr)[kRows], float (&sc)[kProbs], int j) {
#pragma unroll
        for (int i = 0; i < kProbs; ++i) {
            const int o = t + i * kAttnThreads, jj = j + o % kPvStep, h = o / kPvStep;
            sc[i] = a.scores[(row0 + (h < G ? h : G - 1)) * lp + (jj < j1 ? jj : j1 - 1)];
        }
#pragma unroll
        for (int i = 0; i < kRows; ++i)
            if (i < rows) {
                const int jj = j + ps + rpp * i;
                vr[i] = *reinterpret_cast<const uint4*>(vb + (int64_t)(jj < j1 ? jj : j1 - 1) * d);
            }
    };
    uint4 v0[kRows], v1[kRows];
    float s0[kProbs], s1[kProbs];
    load(v0, s0, j0);
    // global max and sum of each head over its chunks (one wave per head)
    const int c_lo = lo / kChunk, c_hi = p / kChunk;
    for (int h = w; h < G; h += 4) {
        const float* st = a.stats + (row0 + h) * a.chunks * 2;
        float m = -INFINITY;
        for (int cc = c_lo + lane; cc <= c_hi; cc += 64) m = fmaxf(m, st[cc * 2]);
        m = wave_max(m);
        float s = 0.0f;
        for (int cc = c_lo + lane; cc <= c_hi; cc += 64) s += st[cc * 2 + 1] * expf(st[cc * 2] - m);
        s = wave_sum(s);
        if (lane == 0) {
            ms[2 * h] = m;
            ms[2 * h + 1] = s;
        }
    }
    float acc[8][G];
#pragma unroll
    for (int m = 0; m < 8; ++m)
#pragma unroll
        for (int h = 0; h < G; ++h) acc[m][h] = 0.0f;
    lds_barrier();
    int j = j0, buf = 0;
    auto step = [&](const uint4 (&vr)[kRows], const float (&sc)[kProbs], uint4 (&vn)[kRows], float (&sn)[kProbs]) {
        // the step's probabilities, once each
#pragma unroll
        for (int i = 0; i < kProbs; ++i) {
            const int o = t + i * kAttnThreads, h = o / kPvStep;
            if (h < G)
                pr[buf][o] = j + o % kPvStep < j1 ? round_bf16(expf(sc[i] - ms[2 * h]) / ms[2 * h + 1]) : 0.0f;
        }
        if (j + kPvStep < j1) load(vn, sn, j + kPvStep);
        // (one barrier per step: a buffer is written again two steps later)
        lds_barrier();
        if (mine) {
#pragma unroll
            for (int i = 0; i < kRows; ++i) {
                const int o = ps + rpp * i;
                if (o < kPvStep && j + o < j1) {
                    float v[8];
                    unpack8(vr[i], v);
#pragma unroll
                    for (int h = 0; h < G; ++h) {
                        const float q = pr[buf][h * kPvStep + o];
#pragma unroll
                        for (int m = 0; m < 8; ++m) acc[m][h] += q * v[m];
                    }
                }
            }
        }
        buf ^= 1;
        j += kPvStep;
        return j < j1;
    };
    while (step(v0, s0, v1, s1) && step(v1, s1, v0, s0)) {
    }
    // the position slices in ascending order
    if (mine) {
#pragma unroll
        for (int h = 0; h < G; ++h)
#pragma unroll
            for (int m = 0; m < 8; ++m) lds[(ps * G + h) * d + 8 * cq + m] = acc[m][h];
    }
    __syncthreads();
    float* part = a.partial + row0 * (int64_t)a.chunks * d;   // [G][chunks][d]
    for (int i = t; i < G * d; i += kAttnThreads) {
        float o = 0.0f;
        for (int r = 0; r < rpp; ++r) o += lds[r * G * d + i];
        if (nspans == 1)
            a.out[obase + i] = f_to_bf16(o);
        else
            __hip_atomic_store(&part[((int64_t)(i / d) * a.chunks + sp) * d + i % d], o, __ATOMIC_RELAXED,
                               __HIP_MEMORY_SCOPE_AGENT);
    }
    if (nspans == 1) return;
    // several spans: the last block of the (sequence, KV head) adds them in order
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    int* counter = &a.counters[kvb];
    if (t == 0) flag = __hip_atomic_fetch_add(counter, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == nspans - 1;
    __syncthreads();
    if (!flag) return;
    for (int i = t; i < G * d; i += kAttnThreads) {
        const float* q = part + (int64_t)(i / d) * a.chunks * d + i % d;
        float sum = 0.0f;
        for (int s0 = 0; s0 < nspans; s0 += 8) {   // 8 loads in flight, added in span order
            float v[8];
#pragma unroll
            for (int k = 0; k < 8; ++k) {
                const int s = s0 + k < nspans ? s0 + k : nspans - 1;
                v[k] = __hip_atomic_load(&q[(int64_t)s * d], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            }
#pragma unroll
            for (int k = 0; k < 8; ++k)
                if (s0 + k < nspans) sum += v[k];
        }
        a.out[obase + i] = f_to_bf16(sum);
    }
    if (t == 0) __hip_atomic_store(counter, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// ---------------------------------------------------------------------------
// gelu(tanh) x up
// ---------------------------------------------------------------------------

template <int DT>
__global__ void gelu_mul_kernel(const void* gate, const void* up, int64_t stride, uint16_t* out, int rows, int cols) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= (int64_t)rows * cols) return;
    const int64_t r = i / cols, c = i - r * cols;
    out[i] = gelu_mul_bf16(load_as_bf16<DT>(gate, r * stride + c), load_as_bf16<DT>(up, r * stride + c));
}

// 8 consecutive values of an FP32 or BF16 tensor, rounded to BF16 (16-byte
// aligned)
template <int DT>
__device__ __forceinline__ void load8_as_bf16(const void* p, int64_t i, float* v) {
    if constexpr (DT == SE12_STEP_F32) {
        const float4 a = *reinterpret_cast<const float4*>(static_cast<const float*>(p) + i);
        const float4 b = *reinterpret_cast<const float4*>(static_cast<const float*>(p) + i + 4);
        v[0] = round_bf16(a.x); v[1] = round_bf16(a.y); v[2] = round_bf16(a.z); v[3] = round_bf16(a.w);
        v[4] = round_bf16(b.x); v[5] = round_bf16(b.y); v[6] = round_bf16(b.z); v[7] = round_bf16(b.w);
    } else {
        unpack8(*reinterpret_cast<const uint4*>(static_cast<const uint16_t*>(p) + i), v);
    }
}

// Rows of whole 8-column pieces (cols and stride multiples of 8, 16-byte
// aligned tensors) on a launch of kGelu8Min values and more: a piece per
// thread, the row from the grid. Bound by the bytes and the tanh: 1,024 x 9,216
// BF16 18.7 -> 11.4 us (5 TB/s) against an element per thread.
template <int DT>
__global__ __launch_bounds__(256) void gelu_mul8_kernel(const void* gate, const void* up, int64_t stride, uint16_t* out,
                                                        int cols) {
    const int64_t r = blockIdx.y;
    const int c = 8 * (int)(blockIdx.x * blockDim.x + threadIdx.x);
    if (c >= cols) return;
    float g[8], u[8];
    load8_as_bf16<DT>(gate, r * stride + c, g);
    load8_as_bf16<DT>(up, r * stride + c, u);
    uint32_t o[4];
#pragma unroll
    for (int k = 0; k < 4; ++k)
        o[k] = f_to_bf16x2(gelu_tanh_bf16(g[2 * k]) * u[2 * k], gelu_tanh_bf16(g[2 * k + 1]) * u[2 * k + 1]);
    *reinterpret_cast<uint4*>(out + r * cols + c) = make_uint4(o[0], o[1], o[2], o[3]);
}

// ---------------------------------------------------------------------------
// logits: blocks over vocabulary slices of kArgmaxPer x 256 logits per row
// ---------------------------------------------------------------------------

constexpr int kArgmaxThreads = 256;
constexpr int kArgmaxPer = 8;
constexpr int kArgmaxSlice = kArgmaxThreads * kArgmaxPer;

struct ArgmaxArgs {
    const void* logits;
    int64_t stride;
    int vocab;
    float softcap;
    uint16_t* logits_out;   // [rows, vocab] or NULL
    int64_t* ids;
    int64_t* tokens;
    int64_t token_stride;
    int64_t* step;          // read only unless pos is set
    int64_t* pos;           // NULL, or advance pos and step once every row's pick is stored
    float* part_v;          // [rows, blocks]
    int* part_i;            // [rows, blocks]
    int* counters;          // [rows + 1]: per-row block arrivals, then row arrivals; zero between launches
};

template <int DT>
__global__ __launch_bounds__(kArgmaxThreads) void logits_argmax_kernel(ArgmaxArgs a) {
    __shared__ float wv[kArgmaxThreads / 64];
    __shared__ int wi[kArgmaxThreads / 64];
    __shared__ int flag;
    const int r = blockIdx.y, blk = blockIdx.x, nblk = gridDim.x;
    const int t = threadIdx.x, lane = t & 63, w = t >> 6;
    const int s0 = blk * kArgmaxSlice;
    float z[kArgmaxPer];
#pragma unroll
    for (int k = 0; k < kArgmaxPer; ++k) {
        const int i = s0 + t + k * kArgmaxThreads;
        z[k] = load_as_bf16<DT>(a.logits, (int64_t)r * a.stride + (i < a.vocab ? i : a.vocab - 1));
    }
    float bv = -INFINITY;
    int bi = 0x7FFFFFFF;
#pragma unroll
    for (int k = 0; k < kArgmaxPer; ++k) {
        const int i = s0 + t + k * kArgmaxThreads;
        float v = z[k];
        if (a.softcap > 0.0f) v = round_bf16(round_bf16(tanhf(round_bf16(v / a.softcap))) * a.softcap);
        if (i < a.vocab) {
            if (a.logits_out) a.logits_out[(int64_t)r * a.vocab + i] = f_to_bf16(v);
            keep_first_max(bv, bi, v, i);
        }
    }
    for (int o = 32; o > 0; o >>= 1) keep_first_max(bv, bi, __shfl_xor(bv, o, 64), __shfl_xor(bi, o, 64));
    if (lane == 0) {
        wv[w] = bv;
        wi[w] = bi;
    }
    __syncthreads();
    if (t == 0) {
        for (int k = 1; k < kArgmaxThreads / 64; ++k) keep_first_max(bv, bi, wv[k], wi[k]);
        if (nblk > 1) {
            __hip_atomic_store(&a.part_v[(int64_t)r * nblk + blk], bv, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            __hip_atomic_store(&a.part_i[(int64_t)r * nblk + blk], bi, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
            const int old = __hip_atomic_fetch_add(&a.counters[r], 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            flag = old == nblk - 1;
        } else {
            flag = 1;
        }
    }
    __syncthreads();
    if (!flag) return;
    if (nblk > 1) {
        bv = -INFINITY;
        bi = 0x7FFFFFFF;
        for (int k = t; k < nblk; k += kArgmaxThreads)
            keep_first_max(bv, bi,
                           __hip_atomic_load(&a.part_v[(int64_t)r * nblk + k], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT),
                           __hip_atomic_load(&a.part_i[(int64_t)r * nblk + k], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT));
        for (int o = 32; o > 0; o >>= 1) keep_first_max(bv, bi, __shfl_xor(bv, o, 64), __shfl_xor(bi, o, 64));
        __syncthreads();
        if (lane == 0) {
            wv[w] = bv;
            wi[w] = bi;
        }
        __syncthreads();
        if (t == 0)
            for (int k = 1; k < kArgmaxThreads / 64; ++k) keep_first_max(bv, bi, wv[k], wi[k]);
    }
    if (t == 0) {
        a.ids[r] = bi;
        const int64_t st = *a.step;
        if (st >= 0 && st < a.token_stride) a.tokens[(int64_t)r * a.token_stride + st] = bi;
        if (nblk > 1) __hip_atomic_store(&a.counters[r], 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        if (a.pos) {
            // every row has read the step before the last row's block moves
            // it: a row arrives only once its step load has returned (the
            // wait is also a compiler barrier)
            bool last = true;
            const int rows = (int)gridDim.y;
            if (rows > 1) {
                asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
                last = __hip_atomic_fetch_add(&a.counters[rows], 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == rows - 1;
            }
            if (last) {
                if (rows > 1) __hip_atomic_store(&a.counters[rows], 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                *a.pos += 1;
                *a.step = st + 1;
            }
        }
    }
}

__global__ void advance_kernel(int64_t* pos, int64_t* step) {
    if (threadIdx.x == 0) {
        *pos += 1;
        *step += 1;
    }
}

}  // namespace se12step

namespace se12step {

static thread_local char g_step_err[256] = "";

int step_fail(const char* msg) {
    snprintf(g_step_err, sizeof g_step_err, "%s", msg);
    return SE12_STEP_E_INVALID;
}

int step_fail(const char* who, const char* msg) {
    snprintf(g_step_err, sizeof g_step_err, "%s: %s", who, msg);
    return SE12_STEP_E_INVALID;
}

int step_launched() {
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) {
        snprintf(g_step_err, sizeof g_step_err, "launch: %s", hipGetErrorString(e));
        return SE12_STEP_E_HIP;
    }
    return SE12_STEP_OK;
}

const char* step_error() { return g_step_err; }

}  // namespace se12step

using namespace se12step;

namespace {

bool dtype_ok(int32_t d) { return d == SE12_STEP_F32 || d == SE12_STEP_BF16; }

bool aligned16(const void* p) { return reinterpret_cast<uintptr_t>(p) % 16 == 0; }

// gelu_mul8_kernel's line: two waves per SIMD of 8 values per lane, so that one
// loads while the other computes (a value per thread gives 8 times the waves),
// in rows that fill a wave of pieces. FP32 / BF16, a value per thread -> 8:
// 114 x 9,216 3.55 / 3.63 -> 3.43 / 3.34 us, but 57 x 9,216 2.70 / 2.67 -> 2.97
// / 2.80; 3,000 x 512 4.62 / 4.50 -> 4.20 / 4.09, but 4,000 x 384 4.59 / 4.51
// -> 4.74 / 4.57.
constexpr int64_t kGelu8Min = 1048576;
constexpr int32_t kGelu8Cols = 512;

int64_t up256(int64_t x) { return (x + 255) & ~(int64_t)255; }

struct AttnLayout {
    int64_t chunks, counters, scores, stats, partial, total;  // byte offsets
};

AttnLayout attn_layout(int32_t batch, int32_t heads, int32_t kv_heads, int32_t head_dim, int32_t max_len) {
    AttnLayout l;
    l.chunks = (max_len + kChunk - 1) / kChunk;
    l.counters = 0;
    l.scores = up256((int64_t)batch * kv_heads * (kMaxHeadDim / kPvCols) * sizeof(int));
    l.stats = l.scores + up256((int64_t)batch * heads * l.chunks * kChunk * sizeof(float));
    l.partial = l.stats + up256((int64_t)batch * heads * l.chunks * 2 * sizeof(float));
    l.total = l.partial + up256((int64_t)batch * heads * l.chunks * head_dim * sizeof(float));
    return l;
}

bool attn_shape_ok(int32_t batch, int32_t heads, int32_t kv_heads, int32_t head_dim, int32_t max_len) {
    if (batch <= 0 || kv_heads <= 0 || heads <= 0 || heads % kv_heads != 0 || head_dim < 8 ||
        head_dim > kMaxHeadDim || head_dim % 8 || max_len < 8 || max_len % 8 || (max_len + kChunk - 1) / kChunk > 65535)
        return false;
    const int g = heads / kv_heads;
    return g == 1 || g == 2 || g == 4 || g == 8;
}

template <int G, int UNIT>
void launch_scores_long(const AttnArgs& a, dim3 grid, hipStream_t stream) {
    if (a.dtype == SE12_STEP_F32)
        hipLaunchKernelGGL((attn_scores_long_kernel<G, SE12_STEP_F32, UNIT>), grid, dim3(kAttnThreads), 0, stream, a);
    else
        hipLaunchKernelGGL((attn_scores_long_kernel<G, SE12_STEP_BF16, UNIT>), grid, dim3(kAttnThreads), 0, stream, a);
}

template <int G>
void launch_attention(const AttnArgs& a, int blocks_x, hipStream_t stream) {
    if (a.d >= kLongDim && (int64_t)blocks_x * a.chunks >= (G == 1 ? kLongBlocks1 : kLongBlocks)) {
        // whole units, the same number per block, on as many blocks as the CUs
        // hold at once
        constexpr int kResident = 256 * (G <= 2 ? 4 : G == 4 ? 3 : 2);
        const int64_t unit = a.d > 128 ? 64 : a.d > 64 ? 128 : 256, units = (a.max_len + unit - 1) / unit;
        const int64_t most = std::max(1, kResident / blocks_x), per_block = (units + most - 1) / most;
        const dim3 grid(blocks_x, (uint32_t)((units + per_block - 1) / per_block));
        // about 16 K key elements per unit
        if (a.d > 128)
            launch_scores_long<G, 64>(a, grid, stream);
        else if (a.d > 64)
            launch_scores_long<G, 128>(a, grid, stream);
        else
            launch_scores_long<G, 256>(a, grid, stream);
        const size_t sums = (size_t)(kAttnThreads / (a.d / 8)) * G * a.d * sizeof(float);
        hipLaunchKernelGGL(attn_pv_long_kernel<G>, grid, dim3(kAttnThreads), sums, stream, a);
        return;
    }
    const dim3 grid(blocks_x, a.chunks);
    const int32_t qs = (int32_t)a.q_stride, kvs = (int32_t)a.kv_stride;
    if (a.dtype == SE12_STEP_F32)
        hipLaunchKernelGGL((attn_scores_kernel<G, SE12_STEP_F32>), grid, dim3(kAttnThreads), 0, stream, a.pos, a.q, a.k, a.kt,
                           a.d, a.max_len, a.kvh, qs, kvs, a);
    else
        hipLaunchKernelGGL((attn_scores_kernel<G, SE12_STEP_BF16>), grid, dim3(kAttnThreads), 0, stream, a.pos, a.q, a.k,
                           a.kt, a.d, a.max_len, a.kvh, qs, kvs, a);
    const dim3 pv_grid(blocks_x, (a.d + kPvCols - 1) / kPvCols, (a.max_len + pv_span<G>() - 1) / pv_span<G>());
    hipLaunchKernelGGL(attn_pv_kernel<G>, pv_grid, dim3(kAttnThreads), 0, stream, a.pos, a.stats, a.scores, a.vc, a.d,
                       a.max_len, a.kvh, a.chunks, a);
}

struct ArgmaxLayout {
    int64_t blocks, counters, part_v, part_i, total;
};

ArgmaxLayout argmax_layout(int32_t rows, int32_t vocab) {
    ArgmaxLayout l;
    l.blocks = (vocab + kArgmaxSlice - 1) / kArgmaxSlice;
    l.counters = 0;
    l.part_v = up256((int64_t)(rows + 1) * sizeof(int));
    l.part_i = l.part_v + up256((int64_t)rows * l.blocks * sizeof(float));
    l.total = l.part_i + up256((int64_t)rows * l.blocks * sizeof(int));
    return l;
}

}  // namespace

namespace se12step {

int step_rmsnorm(const void* in, int32_t in_dtype, int64_t in_stride, const uint16_t* w1, const uint16_t* res_in,
                 uint16_t* res_out, const uint16_t* w2, uint16_t* out, int32_t rows, int32_t hidden, float eps,
                 float in_scale, int32_t mode, void* stream) {
    if (!in || !w1 || !out || rows <= 0 || hidden <= 0 || !dtype_ok(in_dtype) || in_stride < hidden)
        return step_fail("se12_step_rmsnorm: bad argument");
    if (mode == 1 && (!res_in || !res_out || !w2)) return step_fail("se12_step_rmsnorm: mode 1 needs residual and w2");
    if (mode != 0 && mode != 1) return step_fail("se12_step_rmsnorm: mode must be 0 or 1");
    if (hidden > kNormPer * kNormMaxThreads) return step_fail("se12_step_rmsnorm: hidden above 8192");
    NormArgs a{in, in_stride, w1, res_in, res_out, w2, out, hidden, eps, in_scale};
    const int threads = ((hidden + kNormPer - 1) / kNormPer + 63) / 64 * 64;
    const hipStream_t st = static_cast<hipStream_t>(stream);
    const bool f32 = in_dtype == SE12_STEP_F32;
    if (mode == 0) {
        if (f32)
            hipLaunchKernelGGL((rmsnorm_kernel<SE12_STEP_F32, 0>), dim3(rows), dim3(threads), 0, st, a);
        else
            hipLaunchKernelGGL((rmsnorm_kernel<SE12_STEP_BF16, 0>), dim3(rows), dim3(threads), 0, st, a);
    } else {
        if (f32)
            hipLaunchKernelGGL((rmsnorm_kernel<SE12_STEP_F32, 1>), dim3(rows), dim3(threads), 0, st, a);
        else
            hipLaunchKernelGGL((rmsnorm_kernel<SE12_STEP_BF16, 1>), dim3(rows), dim3(threads), 0, st, a);
    }
    return step_launched();
}

}  // namespace se12step

extern "C" {

const char* se12_step_last_error(void) { return step_error(); }

int se12_step_rmsnorm(const void* in, int32_t in_dtype, int64_t in_stride, const uint16_t* w1, uint16_t* residual,
                      const uint16_t* w2, uint16_t* out, int32_t rows, int32_t hidden, float eps, float in_scale,
                      int32_t mode, void* stream) {
    return step_rmsnorm(in, in_dtype, in_stride, w1, residual, residual, w2, out, rows, hidden, eps, in_scale, mode, stream);
}

int64_t se12_step_attention_workspace(int32_t batch, int32_t heads, int32_t kv_heads, int32_t head_dim,
                                      int32_t max_len) {
    if (!attn_shape_ok(batch, heads, kv_heads, head_dim, max_len)) {
        step_fail("se12_step_attention_workspace: bad shape");
        return SE12_STEP_E_INVALID;
    }
    return attn_layout(batch, heads, kv_heads, head_dim, max_len).total;
}

int se12_step_attention(const void* q, const void* k, const void* v, int32_t dtype, int64_t q_stride, int64_t kv_stride,
                        uint16_t* k_cache_t, uint16_t* v_cache, const float* inv_freq, const int64_t* pos, uint16_t* out,
                        int32_t batch, int32_t heads, int32_t kv_heads, int32_t head_dim, int32_t max_len, float scaling,
                        float softcap, int32_t window, void* workspace, int64_t workspace_bytes, void* stream) {
    if (!q || !k || !v || !k_cache_t || !v_cache || !inv_freq || !pos || !out || !workspace || !dtype_ok(dtype))
        return step_fail("se12_step_attention: NULL argument or bad dtype");
    if (!attn_shape_ok(batch, heads, kv_heads, head_dim, max_len) || q_stride < (int64_t)heads * head_dim ||
        kv_stride < (int64_t)kv_heads * head_dim || q_stride > INT32_MAX || kv_stride > INT32_MAX)
        return step_fail("se12_step_attention: bad shape");
    if (!aligned16(k_cache_t) || !aligned16(v_cache)) return step_fail("se12_step_attention: caches not 16-byte aligned");
    const AttnLayout l = attn_layout(batch, heads, kv_heads, head_dim, max_len);
    if (workspace_bytes < l.total) return step_fail("se12_step_attention: workspace too small");
    if (reinterpret_cast<uintptr_t>(workspace) % 256) return step_fail("se12_step_attention: workspace not 256-byte aligned");
    char* ws = static_cast<char*>(workspace);
    AttnArgs a;
    a.q = q;
    a.k = k;
    a.v = v;
    a.dtype = dtype;
    a.q_stride = q_stride;
    a.kv_stride = kv_stride;
    a.kt = k_cache_t;
    a.vc = v_cache;
    a.inv_freq = inv_freq;
    a.pos = pos;
    a.out = out;
    a.counters = reinterpret_cast<int*>(ws + l.counters);
    a.scores = reinterpret_cast<float*>(ws + l.scores);
    a.stats = reinterpret_cast<float*>(ws + l.stats);
    a.partial = reinterpret_cast<float*>(ws + l.partial);
    a.heads = heads;
    a.kvh = kv_heads;
    a.d = head_dim;
    a.max_len = max_len;
    a.chunks = (int)l.chunks;
    a.scaling = scaling;
    a.softcap = softcap;
    a.window = window;
    const hipStream_t st = static_cast<hipStream_t>(stream);
    switch (heads / kv_heads) {
        case 1: launch_attention<1>(a, batch * kv_heads, st); break;
        case 2: launch_attention<2>(a, batch * kv_heads, st); break;
        case 4: launch_attention<4>(a, batch * kv_heads, st); break;
        default: launch_attention<8>(a, batch * kv_heads, st); break;
    }
    return step_launched();
}

int se12_step_gelu_mul(const void* gate, const void* up, int32_t dtype, int64_t stride, uint16_t* out, int32_t rows,
                       int32_t cols, void* stream) {
    if (!gate || !up || !out || rows <= 0 || cols <= 0 || stride < cols || !dtype_ok(dtype))
        return step_fail("se12_step_gelu_mul: bad argument");
    const int64_t n = (int64_t)rows * cols;
    const dim3 grid((unsigned)((n + 255) / 256));
    const hipStream_t st = static_cast<hipStream_t>(stream);
    if (n >= kGelu8Min && cols >= kGelu8Cols && rows <= 65535 && cols % 8 == 0 && stride % 8 == 0 &&
        aligned16(gate) && aligned16(up) && aligned16(out)) {
        const dim3 grid8((unsigned)((cols / 8 + 255) / 256), rows);
        if (dtype == SE12_STEP_F32)
            hipLaunchKernelGGL(gelu_mul8_kernel<SE12_STEP_F32>, grid8, dim3(256), 0, st, gate, up, stride, out, cols);
        else
            hipLaunchKernelGGL(gelu_mul8_kernel<SE12_STEP_BF16>, grid8, dim3(256), 0, st, gate, up, stride, out, cols);
        return step_launched();
    }
    if (dtype == SE12_STEP_F32)
        hipLaunchKernelGGL(gelu_mul_kernel<SE12_STEP_F32>, grid, dim3(256), 0, st, gate, up, stride, out, rows, cols);
    else
        hipLaunchKernelGGL(gelu_mul_kernel<SE12_STEP_BF16>, grid, dim3(256), 0, st, gate, up, stride, out, rows, cols);
    return step_launched();
}

int64_t se12_step_logits_workspace(int32_t rows, int32_t vocab) {
    if (rows <= 0 || vocab <= 0 || rows > 65535) {
        step_fail("se12_step_logits_workspace: bad shape");
        return SE12_STEP_E_INVALID;
    }
    return argmax_layout(rows, vocab).total;
}

}  // extern "C"

namespace {

int launch_argmax(const char* who, const void* logits, int32_t dtype, int64_t stride, int32_t rows, int32_t vocab,
                  float softcap, uint16_t* logits_out, int64_t* ids, int64_t* tokens, int64_t token_stride,
                  int64_t* step, int64_t* pos, void* workspace, int64_t workspace_bytes, void* stream) {
    if (!logits || !ids || !tokens || !step || !workspace || rows <= 0 || rows > 65535 || vocab <= 0 || stride < vocab ||
        !dtype_ok(dtype))
        return step_fail(who, "bad argument");
    const ArgmaxLayout l = argmax_layout(rows, vocab);
    if (workspace_bytes < l.total) return step_fail(who, "workspace too small");
    if (reinterpret_cast<uintptr_t>(workspace) % 256) return step_fail(who, "workspace not 256-byte aligned");
    char* ws = static_cast<char*>(workspace);
    ArgmaxArgs a{logits, stride, vocab, softcap, logits_out, ids, tokens, token_stride, step, pos,
                 reinterpret_cast<float*>(ws + l.part_v), reinterpret_cast<int*>(ws + l.part_i),
                 reinterpret_cast<int*>(ws + l.counters)};
    const dim3 grid((unsigned)l.blocks, rows);
    const hipStream_t st = static_cast<hipStream_t>(stream);
    if (dtype == SE12_STEP_F32)
        hipLaunchKernelGGL(logits_argmax_kernel<SE12_STEP_F32>, grid, dim3(kArgmaxThreads), 0, st, a);
    else
        hipLaunchKernelGGL(logits_argmax_kernel<SE12_STEP_BF16>, grid, dim3(kArgmaxThreads), 0, st, a);
    return step_launched();
}

}  // namespace

extern "C" {

int se12_step_logits_argmax(const void* logits, int32_t dtype, int64_t stride, int32_t rows, int32_t vocab, float softcap,
                            uint16_t* logits_out, int64_t* ids, int64_t* tokens, int64_t token_stride,
                            const int64_t* step, void* workspace, int64_t workspace_bytes, void* stream) {
    // the kernel writes the step only when it is given pos
    return launch_argmax("se12_step_logits_argmax", logits, dtype, stride, rows, vocab, softcap, logits_out, ids, tokens,
                         token_stride, const_cast<int64_t*>(step), nullptr, workspace, workspace_bytes, stream);
}

int se12_step_logits_argmax_advance(const void* logits, int32_t dtype, int64_t stride, int32_t rows, int32_t vocab,
                                    float softcap, uint16_t* logits_out, int64_t* ids, int64_t* tokens,
                                    int64_t token_stride, int64_t* step, int64_t* pos, void* workspace,
                                    int64_t workspace_bytes, void* stream) {
    if (!pos) return step_fail("se12_step_logits_argmax_advance: NULL pos");
    return launch_argmax("se12_step_logits_argmax_advance", logits, dtype, stride, rows, vocab, softcap, logits_out, ids,
                         tokens, token_stride, step, pos, workspace, workspace_bytes, stream);
}

int se12_step_advance(int64_t* pos, int64_t* step, void* stream) {
    if (!pos || !step) return step_fail("se12_step_advance: NULL argument");
    hipLaunchKernelGGL(advance_kernel, dim3(1), dim3(64), 0, static_cast<hipStream_t>(stream), pos, step);
    return step_launched();
}

}  // extern "C"

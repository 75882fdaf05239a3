// Prompt-pass kernels of a Gemma-2 style decoder: what stands between the
// library matrix products of a layer, so that a prompt costs a handful of
// launches per layer instead of ~80 framework kernels that each pass over the
// activations (or the T x T scores) again.
//
//   rope       rotary embedding of q (in place) and k with the framework's
//              roundings, the K (transposed) and V cache slots, and K and V in
//              the order the attention's matrix instructions take them
//   attention  causal soft-capped attention on MFMA, scores kept in FP32
//              registers
//
// (The norms and the MLP gate are se12_step_rmsnorm and se12_step_gelu_mul.)
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <algorithm>
#include <cstdio>

#include "se12_step.h"
#include "se12_step_math.hpp"

namespace se12step {

typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef float floatx16_t __attribute__((ext_vector_type(16)));

// ---------------------------------------------------------------------------
// rope: one block per (64 positions, head of q, k or v, sequence)
// ---------------------------------------------------------------------------

constexpr int kRopeThreads = 256;
constexpr int kRopeTokens = 64;

struct RopeArgs {
    uint16_t* qkv;           // [B, T, stride]: q heads, k heads, v heads
    int64_t stride;
    const uint16_t* cos;     // [T, d] BF16
    const uint16_t* sin;
    uint16_t* kt;            // [B, kvh, d, L]
    uint16_t* vc;            // [B, kvh, L, d]
    uint16_t* ko;            // [B, kvh, Tp / 32][d / 16][64][8]: K operands of a key tile
    uint16_t* vo;            // [B, kvh, Tp / 32][d / 32][2][64][8]: V operands of a key tile
    int T, Tp, L, heads, kvh, d;
};

// the key (0..31) of row m of a tile's A operand (the attention kernel below)
__device__ __forceinline__ int key_of_row(int m) { return (m & 0x13) | ((m & 4) << 1) | ((m & 8) >> 1); }

__device__ __forceinline__ void unpack_bf16x8(const uint4 r, float* v) {
    const uint32_t w[4] = {r.x, r.y, r.z, r.w};
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        v[2 * i] = __uint_as_float(w[i] << 16);
        v[2 * i + 1] = __uint_as_float(w[i] & 0xFFFF0000u);
    }
}

__device__ __forceinline__ uint4 pack_bf16x8(const float* v) {
    return make_uint4(f_to_bf16x2(v[0], v[1]), f_to_bf16x2(v[2], v[3]), f_to_bf16x2(v[4], v[5]), f_to_bf16x2(v[6], v[7]));
}

// x cos + rotate_half(x) sin, each product and the sum rounded to BF16
__device__ __forceinline__ void rotate8(const float* x, const float* other, const float* cs, const float* sn, float sign,
                                        float* y) {
#pragma unroll
    for (int i = 0; i < 8; ++i) y[i] = round_bf16(x[i] * cs[i]) + round_bf16(sign * other[i] * sn[i]);
}

// Elements of a head go through in pairs of 16-byte pieces (columns c and c +
// d / 2, what the rotation mixes). k and v pass through LDS ([64][d], rows
// padded by 16 bytes) to be written in the other orders, 16 bytes per lane.
// Bound by the activations' bytes.
__global__ __launch_bounds__(kRopeThreads) void prefill_rope_kernel(RopeArgs a) {
    extern __shared__ __attribute__((aligned(16))) char tile[];
    const int t = threadIdx.x, head = blockIdx.y, b = blockIdx.z;
    const int t0 = blockIdx.x * kRopeTokens;
    const int n = min(kRopeTokens, a.T - t0);
    const int d = a.d, pairs = d / 16, row_bytes = 2 * d + 16;
    const bool is_q = head < a.heads, is_v = head >= a.heads + a.kvh;
    const int kh = is_v ? head - a.heads - a.kvh : head - a.heads;
    uint16_t* base = a.qkv + ((int64_t)b * a.T + t0) * a.stride + (int64_t)head * d;
    for (int i = t; i < n * pairs; i += kRopeThreads) {
        const int r = i / pairs, c = 8 * (i % pairs);
        uint4* lo = reinterpret_cast<uint4*>(base + r * a.stride + c);
        uint4* hi = reinterpret_cast<uint4*>(base + r * a.stride + c + d / 2);
        uint4 u = *lo, v = *hi;
        if (!is_v) {
            float x[8], y[8], cs[8], sn[8], lo_out[8], hi_out[8];
            const uint16_t* cp = a.cos + (int64_t)(t0 + r) * d + c;
            const uint16_t* sp = a.sin + (int64_t)(t0 + r) * d + c;
            unpack_bf16x8(u, x);
            unpack_bf16x8(v, y);
            // (both halves of a row of cos / sin are the same values)
            unpack_bf16x8(*reinterpret_cast<const uint4*>(cp), cs);
            unpack_bf16x8(*reinterpret_cast<const uint4*>(sp), sn);
            rotate8(x, y, cs, sn, -1.0f, lo_out);
            rotate8(y, x, cs, sn, 1.0f, hi_out);
            u = pack_bf16x8(lo_out);
            v = pack_bf16x8(hi_out);
            if (is_q) {
                *lo = u;
                *hi = v;
            }
        } else {
            uint16_t* slot = a.vc + (((int64_t)b * a.kvh + kh) * a.L + t0 + r) * d;
            *reinterpret_cast<uint4*>(slot + c) = u;
            *reinterpret_cast<uint4*>(slot + c + d / 2) = v;
        }
        if (!is_q) {
            *reinterpret_cast<uint4*>(tile + r * row_bytes + 2 * c) = u;
            *reinterpret_cast<uint4*>(tile + r * row_bytes + 2 * c + d) = v;
        }
    }
    if (is_q) return;
    // positions past the prompt are zeros
    for (int i = t + n * pairs; i < kRopeTokens * pairs; i += kRopeThreads) {
        const int r = i / pairs, c = 8 * (i % pairs);
        *reinterpret_cast<uint4*>(tile + r * row_bytes + 2 * c) = make_uint4(0u, 0u, 0u, 0u);
        *reinterpret_cast<uint4*>(tile + r * row_bytes + 2 * c + d) = make_uint4(0u, 0u, 0u, 0u);
    }
    __syncthreads();
    const uint16_t* lds = reinterpret_cast<const uint16_t*>(tile);
    const int row_elems = row_bytes / 2;
    const int64_t kv_head = (int64_t)b * a.kvh + kh;
    // 8 values of consecutive positions j .. of column e
    auto column8 = [&](int j, int e) {
        uint16_t v[8];
#pragma unroll
        for (int k = 0; k < 8; ++k) v[k] = lds[(j + k) * row_elems + e];
        return make_uint4(v[0] | ((uint32_t)v[1] << 16), v[2] | ((uint32_t)v[3] << 16), v[4] | ((uint32_t)v[5] << 16),
                          v[6] | ((uint32_t)v[7] << 16));
    };
    // the two key tiles' operands: 16-byte pieces, 4 d per tile
    uint16_t* op = (is_v ? a.vo : a.ko) + (kv_head * a.Tp + t0) * d;
    for (int i = t; i < 8 * d; i += kRopeThreads) {
        const int lane = i & 63, step = i >> 6, tile32 = step / (d / 16), st = step % (d / 16);
        uint4 u;
        if (is_v)   // row tile st / 2, inner step st % 2: 8 keys of one column
            u = column8(32 * tile32 + 16 * (st & 1) + 8 * (lane >> 5), 32 * (st >> 1) + (lane & 31));
        else        // inner step st: 8 columns of one key
            u = *reinterpret_cast<const uint4*>(tile + (32 * tile32 + key_of_row(lane & 31)) * row_bytes +
                                                2 * (16 * st + 8 * (lane >> 5)));
        *reinterpret_cast<uint4*>(op + (int64_t)8 * i) = u;
    }
    if (is_v) return;
    // the K cache, 8 positions per lane; past the prompt it keeps what it holds
    for (int i = t; i < d * (kRopeTokens / 8); i += kRopeThreads) {
        const int e = i / (kRopeTokens / 8), j = 8 * (i % (kRopeTokens / 8));
        uint16_t* p = a.kt + (kv_head * d + e) * a.L + t0 + j;
        if (j + 8 <= n)
            *reinterpret_cast<uint4*>(p) = column8(j, e);
        else
            for (int k = 0; k < 8 && j + k < n; ++k) p[k] = lds[(j + k) * row_elems + e];
    }
}

// ---------------------------------------------------------------------------
// attention: one block per (32 queries, head, sequence)
// ---------------------------------------------------------------------------

// S^T = K Q^T and O^T = V^T P^T with v_mfma_f32_32x32x16_bf16 (A: lane l holds
// row l % 32, 8 of the 16 inner positions 8 (l / 32) ..; B the same of column l
// % 32; D: column l % 32, rows (i % 4) + 8 (i / 4) + 4 (l / 32)). Each wave
// keeps its 32 queries (Q as the B operand) and 32 x D outputs in registers
// and takes every 4th tile of 32 keys; the four waves' sums meet once at the
// end, through LDS. The keys of a tile are loaded in the order that leaves
// the scores of a lane, as they come out of the first product, the B operand
// of the second (key of A row m: key_of_row), so probabilities never leave
// their lane.
// Scores, capping and sums are FP32; a probability is rounded to BF16 for the
// second product, and their sum is that of the rounded ones, so that the weights
// add up to one. A query's weights are 2^(s - m - shift): s its scores (base 2),
// m the largest of them seen, or up to kMaxSlack below it. m starts at the
// wave's first tile; a tile that passes it by more than kMaxSlack moves m and
// what is summed, and starts again. shift makes the weights add up to less than
// one, so the sums of any finite V stay finite, as with weights normalised
// first, and the largest weight stays above 2^-45: V down to 1e-24 keeps its
// bits. (e^s itself fits FP32 with |s| <= softcap, and summing it needs no m,
// but V above 6e16 then overflows at a softcap of 50: 1,024 / 4,096 positions, 8
// heads of 256, both launches, 32.8 / 147 us that way, 33.8 / 157 this, 40 where
// scores of a standard deviation of 16 make tiles start again.)
// K and V^T operands come straight from L2, 1 KB of consecutive bytes per
// instruction in the order prefill_rope_kernel left them; with K and V^T
// row-major, 32 bytes of each of 32 rows per instruction, the first-level cache
// kept missing: 1,024 positions, 8 heads of 256, 37.5 us against 19.2, both
// without the maximum, 20.3 with it (0.21 PFLOP/s of the causal half; a block per
// CU whose longest walks 32 tiles); the framework ops took ~120 us for the same.
constexpr int kPrefillThreads = 256;
constexpr int kPrefillRows = 32;
constexpr float kMaxSoftcap = 64.0f;
constexpr float kMaxSlack = 16.0f;      // base 2

struct PrefillAttnArgs {
    const uint16_t* qkv;     // [B, T, stride], rotated
    int64_t stride;
    const uint16_t* ko;      // K and V operands of the key tiles
    const uint16_t* vo;
    uint16_t* out;           // [B, T, heads * d]
    int T, Tp, heads, kvh, window;
    float c1;                // 2 scaling / softcap, base 2
    float c2;                // softcap, base 2
    float shift;             // log2 of the keys of a query (rounded up) + 1 + kMaxSlack
};

template <int D>
__global__ __launch_bounds__(kPrefillThreads) void prefill_attention_kernel(PrefillAttnArgs a) {
    constexpr int kSteps = D / 16;     // inner steps of the first product
    constexpr int kTiles = D / 32;     // row tiles of the second
    extern __shared__ __attribute__((aligned(16))) float sums[];   // [2][kTiles * 16 + 1][64]
    __shared__ float maxima[kPrefillThreads / 64][32];
    const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const int head = blockIdx.y, b = blockIdx.z, kh = head / (a.heads / a.kvh);
    // the blocks with the most keys first
    const int q0 = ((int)gridDim.x - 1 - (int)blockIdx.x) * kPrefillRows;
    const int col = lane & 31, half = lane >> 5;
    const int64_t seq = (int64_t)b * a.T;
    const int q = q0 + col;
    const uint16_t* qp = a.qkv + (seq + min(q, a.T - 1)) * a.stride + (int64_t)head * D + 8 * half;
    const int64_t kv_at = ((int64_t)b * a.kvh + kh) * a.Tp * D + 8 * lane;
    const uint16_t* kp = a.ko + kv_at;
    const uint16_t* vp = a.vo + kv_at;

    bf16x8_t qf[kSteps];
#pragma unroll
    for (int s = 0; s < kSteps; ++s) qf[s] = *reinterpret_cast<const bf16x8_t*>(qp + 16 * s);
    floatx16_t o[kTiles];
#pragma unroll
    for (int i = 0; i < kTiles; ++i)
#pragma unroll
        for (int e = 0; e < 16; ++e) o[i][e] = 0.0f;
    float l = 0.0f, m = -a.c2;     // no score is lower

    const int last = min(q0 + kPrefillRows, a.T) - 1;   // the block's last query sees keys up to itself
    const int lo = a.window > 0 ? max(0, q0 - a.window + 1) : 0;
    // K of the next tile is loaded once the scores are out of this one's
    // registers, V of the next once the outputs have used this one's: each has
    // most of a tile's work to arrive in (loads past the wave's last tile
    // repeat it)
    bf16x8_t kf[kSteps], vf[kTiles][2];
    const int t_last = last / 32;
    auto load_k = [&](int t) {
        const uint16_t* p = kp + (int64_t)min(t, t_last) * (32 * D);
#pragma unroll
        for (int s = 0; s < kSteps; ++s) {
            kf[s] = *reinterpret_cast<const bf16x8_t*>(p + 512 * s);
            __builtin_amdgcn_sched_barrier(0);
        }
    };
    auto load_v = [&](int t) {
        const uint16_t* p = vp + (int64_t)min(t, t_last) * (32 * D);
#pragma unroll
        for (int i = 0; i < kTiles; ++i)
#pragma unroll
            for (int s = 0; s < 2; ++s) {
                vf[i][s] = *reinterpret_cast<const bf16x8_t*>(p + 512 * (2 * i + s));
                __builtin_amdgcn_sched_barrier(0);
            }
    };
    constexpr int kWaves = kPrefillThreads / 64;
    const int kt0 = lo / 32 + w;
    int kt = kt0;
    float top = 0.0f;
    load_k(kt);
    __builtin_amdgcn_sched_barrier(0);   // the order of the loop's loads, and so its waits
    load_v(kt);
    while (true) {
        bool higher = false;
        for (; kt <= t_last; kt += kWaves) {
            const int k0 = 32 * kt;
            floatx16_t sc;
#pragma unroll
            for (int e = 0; e < 16; ++e) sc[e] = 0.0f;
#pragma unroll
            for (int s = 0; s < kSteps; ++s) sc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(kf[s], qf[s], sc, 0, 0, 0);
            __builtin_amdgcn_sched_barrier(0);
            load_k(kt + kWaves);
            __builtin_amdgcn_sched_barrier(0);
            // softcap tanh(x) = softcap (1 - 2 r), r = 1 / (1 + e^2x), base 2
            float r[16];
#pragma unroll
            for (int e = 0; e < 16; ++e)
                r[e] = __builtin_amdgcn_rcpf(1.0f + __builtin_amdgcn_exp2f(sc[e] * a.c1));
            const bool inside = k0 + 31 <= q0 && (a.window <= 0 || last - k0 < a.window);
            if (!inside) {
                const int reach = a.window > 0 ? a.window : INT32_MAX;
#pragma unroll
                for (int e = 0; e < 16; ++e) {
                    const int key = k0 + 16 * (e >> 3) + 8 * half + (e & 7);
                    r[e] = ((key > q) | (q - key >= reach)) ? INFINITY : r[e];
                }
            }
            float least[5];
#pragma unroll
            for (int e = 0; e < 5; ++e) least[e] = fminf(fminf(r[3 * e], r[3 * e + 1]), r[3 * e + 2]);
            top = a.c2 - 2.0f * a.c2 * fminf(fminf(fminf(least[0], least[1]), least[2]), fminf(fminf(least[3], least[4]), r[15]));
            // (the two lanes of a query keep one maximum)
            if (kt == kt0) m = fmaxf(m, fmaxf(top, __shfl_xor(top, 32, 64)));
            const float base = a.c2 - (m + a.shift);
            bf16x8_t pf[2];
            float tile_l = 0.0f;
#pragma unroll
            for (int s = 0; s < 2; ++s) {
                uint32_t u[4];
#pragma unroll
                for (int k = 0; k < 4; ++k) {
                    u[k] = f_to_bf16x2(__builtin_amdgcn_exp2f(base - 2.0f * a.c2 * r[8 * s + 2 * k]),
                                       __builtin_amdgcn_exp2f(base - 2.0f * a.c2 * r[8 * s + 2 * k + 1]));
                    tile_l += __uint_as_float(u[k] << 16) + __uint_as_float(u[k] & 0xFFFF0000u);
                }
                pf[s] = __builtin_bit_cast(bf16x8_t, make_uint4(u[0], u[1], u[2], u[3]));
            }
            higher = __builtin_amdgcn_ballot_w64(top > m + kMaxSlack) != 0;
            if (!higher) {
                l += tile_l;
#pragma unroll
                for (int i = 0; i < kTiles; ++i)
#pragma unroll
                    for (int s = 0; s < 2; ++s)
                        o[i] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(vf[i][s], pf[s], o[i], 0, 0, 0);
            }
            __builtin_amdgcn_sched_barrier(0);
            load_v(higher ? kt : kt + kWaves);   // on both paths, so that the waits stay exact
            if (higher) break;
        }
        if (!higher) break;
        // the tile passes the maximum: what is summed moves to the new one, and
        // the tile starts again (outside the loop over the tiles, so that the
        // sums stay in accumulation registers there)
        const float to = fmaxf(m, fmaxf(top, __shfl_xor(top, 32, 64)));
        const float scale = __builtin_amdgcn_exp2f(m - to);
        m = to;
        l *= scale;
#pragma unroll
        for (int i = 0; i < kTiles; ++i)
#pragma unroll
            for (int e = 0; e < 16; ++e) o[i][e] *= scale;
        load_k(kt);
        __builtin_amdgcn_s_waitcnt(0);   // rare: keeps the loop's waits exact
    }
    l += __shfl_xor(l, 32, 64);
    // the waves' sums on one maximum
    if (half == 0) maxima[w][col] = m;
    __syncthreads();
    float all = maxima[0][col];
#pragma unroll
    for (int k = 1; k < kWaves; ++k) all = fmaxf(all, maxima[k][col]);
    const float scale = __builtin_amdgcn_exp2f(m - all);

    // waves 2, 3 hand their sums to 0, 1, then 1 to 0: (w0 + w2) + (w1 + w3)
    constexpr int kValues = kTiles * 16 + 1;
    auto put = [&](int slot, float by) {
        float* to = sums + (size_t)slot * kValues * 64 + lane;
#pragma unroll
        for (int i = 0; i < kTiles; ++i)
#pragma unroll
            for (int e = 0; e < 16; ++e) to[(16 * i + e) * 64] = o[i][e] * by;
        to[(kValues - 1) * 64] = l * by;
    };
    auto add = [&](int slot, float by) {
        const float* from = sums + (size_t)slot * kValues * 64 + lane;
#pragma unroll
        for (int i = 0; i < kTiles; ++i)
#pragma unroll
            for (int e = 0; e < 16; ++e) o[i][e] = o[i][e] * by + from[(16 * i + e) * 64];
        l = l * by + from[(kValues - 1) * 64];
    };
    if (w >= 2) put(w - 2, scale);
    __syncthreads();
    if (w < 2) add(w, scale);
    __syncthreads();
    if (w == 1) put(0, 1.0f);
    __syncthreads();
    if (w > 0 || q >= a.T) {
        return;
    }
    add(0, 1.0f);
    const float inv = 1.0f / l;
    uint16_t* op = a.out + (seq + q) * (int64_t)a.heads * D + (int64_t)head * D + 4 * half;
#pragma unroll
    for (int i = 0; i < kTiles; ++i)
#pragma unroll
        for (int g = 0; g < 4; ++g) {
            const uint2 u = make_uint2(f_to_bf16x2(o[i][4 * g] * inv, o[i][4 * g + 1] * inv),
                                       f_to_bf16x2(o[i][4 * g + 2] * inv, o[i][4 * g + 3] * inv));
            *reinterpret_cast<uint2*>(op + 32 * i + 8 * g) = u;
        }
}

}  // namespace se12step

using namespace se12step;

namespace {

bool aligned(const void* p, size_t n) { return reinterpret_cast<uintptr_t>(p) % n == 0; }

bool prefill_shape_ok(int32_t batch, int32_t tokens, int32_t heads, int32_t kv_heads, int32_t head_dim, int64_t stride) {
    return batch > 0 && batch <= 65535 && tokens > 0 && heads > 0 && kv_heads > 0 && heads % kv_heads == 0 &&
           heads + 2 * kv_heads <= 65535 && (head_dim == 64 || head_dim == 128 || head_dim == 256) &&
           stride >= (int64_t)(heads + 2 * kv_heads) * head_dim && stride % 8 == 0;
}

int64_t padded_tokens(int32_t tokens) { return ((int64_t)tokens + kRopeTokens - 1) / kRopeTokens * kRopeTokens; }

template <int D>
void launch_prefill_attention(const PrefillAttnArgs& a, int batch, hipStream_t stream) {
    const dim3 grid((a.T + kPrefillRows - 1) / kPrefillRows, a.heads, batch);
    const size_t lds = (size_t)2 * (D / 32 * 16 + 1) * 64 * sizeof(float);
    hipLaunchKernelGGL(prefill_attention_kernel<D>, grid, dim3(kPrefillThreads), lds, stream, a);
}

}  // namespace

extern "C" {

int64_t se12_step_prefill_workspace(int32_t batch, int32_t tokens, int32_t heads, int32_t kv_heads, int32_t head_dim) {
    if (!prefill_shape_ok(batch, tokens, heads, kv_heads, head_dim, (int64_t)(heads + 2 * kv_heads) * head_dim))
        return step_fail("se12_step_prefill_workspace: bad shape");
    return 2 * (int64_t)batch * kv_heads * head_dim * padded_tokens(tokens) * (int64_t)sizeof(uint16_t);
}

int se12_step_prefill_attention(uint16_t* qkv, int64_t stride, const uint16_t* cos, const uint16_t* sin,
                                uint16_t* k_cache_t, uint16_t* v_cache, uint16_t* out, int32_t batch, int32_t tokens,
                                int32_t heads, int32_t kv_heads, int32_t head_dim, int32_t max_len, float scaling,
                                float softcap, int32_t window, void* workspace, int64_t workspace_bytes, void* stream) {
    const char* fn = "se12_step_prefill_attention";
    if (!qkv || !cos || !sin || !k_cache_t || !v_cache || !out || !workspace) return step_fail(fn, "NULL argument");
    if (!prefill_shape_ok(batch, tokens, heads, kv_heads, head_dim, stride) || max_len < tokens || max_len % 8)
        return step_fail(fn, "bad shape");
    if (!(softcap > 0.0f && softcap <= kMaxSoftcap)) return step_fail(fn, "softcap must be in (0, 64]");
    if (!aligned(qkv, 16) || !aligned(cos, 16) || !aligned(sin, 16) || !aligned(k_cache_t, 16) || !aligned(v_cache, 16) ||
        !aligned(out, 8) || !aligned(workspace, 16))
        return step_fail(fn, "misaligned tensor");
    if (workspace_bytes < se12_step_prefill_workspace(batch, tokens, heads, kv_heads, head_dim))
        return step_fail(fn, "workspace too small");
    const hipStream_t st = static_cast<hipStream_t>(stream);
    const int Tp = (int)padded_tokens(tokens);
    uint16_t* ko = static_cast<uint16_t*>(workspace);
    uint16_t* vo = ko + (int64_t)batch * kv_heads * head_dim * Tp;
    const RopeArgs r{qkv, stride, cos, sin, k_cache_t, v_cache, ko, vo, tokens, Tp, max_len, heads, kv_heads, head_dim};
    const dim3 rope_grid(Tp / kRopeTokens, heads + 2 * kv_heads, batch);
    const size_t rope_lds = (size_t)kRopeTokens * (2 * head_dim + 16);
    hipLaunchKernelGGL(prefill_rope_kernel, rope_grid, dim3(kRopeThreads), rope_lds, st, r);
    constexpr float kLog2E = 1.4426950408889634f;
    const int64_t keys = window > 0 ? std::min(window, tokens) : tokens;
    int keys_log2 = 0;
    while (((int64_t)1 << keys_log2) < keys) ++keys_log2;
    const PrefillAttnArgs a{qkv, stride, ko, vo, out, tokens, Tp, heads, kv_heads, window,
                            2.0f * scaling / softcap * kLog2E, softcap * kLog2E, (float)keys_log2 + 1.0f + kMaxSlack};
    if (head_dim == 64)
        launch_prefill_attention<64>(a, batch, st);
    else if (head_dim == 128)
        launch_prefill_attention<128>(a, batch, st);
    else
        launch_prefill_attention<256>(a, batch, st);
    return step_launched();
}

}  // extern "C"

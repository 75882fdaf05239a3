// Batched fused SE12 decode + matrix product for gfx950: Y[b, n] =
// sum_k W[n, k] X[b, k] for up to 32 batch rows (BF16, or FP32) in ONE pass over the
// weights (the dot2 kernel in se12_gemv.hip takes 4 rows per launch and so
// re-reads W once per 4 rows). Same semantics as the reference kernel
// lws/adapters/cuda/kernels/gemv_se12.cu:50-142 at batch B, which runs one
// warp per (row, batch) element and reads W B times.
//
// Grid: block = R x KG wave64s: R consecutive tile rows (R = ceil(batch / 8), 4 in place of 3,
// the fewest waves whose threads load an x slab in one go; FP32 x 4, or 8 above
// 16 rows) times KG K groups;
// wave w owns tile row R * row_block + w % R and, of the split's K tiles, the
// ones of K group w / R (every KG-th tile). blockIdx.y = K split s covering
// the K tiles [s*TC/S, (s+1)*TC/S). A grouped launch serves up to 4 matrices
// with the same K: blockIdx.z = matrix, blockIdx.x = row block (the grid's x
// spans the tallest matrix; blocks past a shorter one's rows leave at once).
//
// Per step each K group's waves share one copy of their x slab (batch rows x
// 256 columns, BF16) in LDS: every thread requests up to 4 pieces of 16
// bytes of a later step's slabs while its wave decodes tile i and writes
// them to LDS after its MFMAs. Double-buffered with a block barrier per step
// (slabs of step i + 1 written during step i), or, on launches of 12 or more
// steps where LDS holds it, a ring of 8 slabs written 4 steps ahead with a
// barrier every 4 steps. Each wave requests its tile streams two tiles ahead
// of the decode (the edge-handling and FP32 variants one).
//
// Each tile is loaded whole-line (a kilobyte of sm holding 4 tile
// rows per load instruction, as the resident-x kernel does) and moved into
// the block layout with DPP exchanges: lane l holds, in part p, the 16
// columns 16 (4 (l / 16) + p) .. + 15 of row l % 16, decoded through the
// pair table with listed escapes and raw tiles. Each part's first and second
// 8 columns are the A operands of two v_mfma_f32_16x16x32_bf16 (MFMA row =
// tile row); their K positions differ between lane groups, and the B
// operands (lane l: batch row 16 g + l % 16) read the same 8 columns of the
// x slab. The decoded tile never goes through memory;
// 8 MFMAs per tile and group of 16 batch rows, FP32 accumulate, in a fixed
// order. Rows of the LDS x slabs are padded to 528 bytes so that the 16-byte
// reads of 8 lanes per cycle hit distinct banks. Batch rows past the batch
// in a 16-row group read stale LDS: MFMA output column n depends on B column
// n only, and those columns are not stored.
//
// A wave adds its K tiles in ascending order; the K groups of a tile row are
// added in LDS in ascending group order by the group-0 wave, and for S > 1
// the last wave of a tile row to finish (device-scope arrival counter, reset
// by that wave) adds the S partials in ascending split order. The launch
// shape (W, S) fixes every sum: the raw-BF16 twin (same kernel, RAW) is
// bit-identical under one shape.
//
// How x is read (XMode): whole K tiles of 16-byte aligned BF16 rows; BF16 of
// any K and alignment (16-byte loads at any address, the columns past K cut
// where they are stored to LDS, weights past K zeroed: the SE12 streams
// themselves are whole, aligned tiles; loading the tiles whole-line and one
// ahead instead of element-wise x with each tile loaded and used in turn:
// 5003x2887 at 6 / 16 / 32 rows 21.5 / 25.0 / 28.2 -> 13.9 / 15.1 / 16.4 us,
// 14337x3585 at 8 / 24 56.6 / 72.1 -> 27.9 / 31.2); FP32 of any K (three BF16
// planes, below). The raw twin's W is guarded by its edges in the last two.
#include <algorithm>

#include "se12_device.hpp"
#include "se12_internal.hpp"

namespace se12 {

typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef float floatx4_t __attribute__((ext_vector_type(4)));

constexpr int kRowBytes = 528;                    // 512 B of BF16 + 16 B of padding

template <int BG>
constexpr int x_slab_bytes() {
    return 16 * BG * kRowBytes;
}

// How a launch reads x: kXFast, BF16 in whole K tiles and 16-byte aligned rows;
// kXEdge, BF16 of any K and alignment; kXF32, FP32 of any K.
enum XMode { kXFast, kXEdge, kXF32 };

// FP32 x goes to LDS as three BF16 planes, x = h + 2^-7 (m + 2^-8 l): each plane
// is the top 16 bits of what the ones before it leave (8 of the 24
// significand bits), m and l scaled up to at most x's own size, so that no bit
// of them falls below BF16's range where x is small (unscaled, x of 2^-116 kept
// 18 bits and x below 2^-133 none). The product is then three MFMAs per part
// whose BF16 products are exact, summed in FP32 per K tile and, h apart from m
// and l, over the tiles. The edge-handling dot2 kernel it replaces at 5 and more
// rows reads the weights once per 4 rows. Bound by the conversion and LDS traffic of the
// planes beside the weights' stream. Cold weights, before and after: 3584x14336
// at 8 / 16 / 32 rows 214 / 427 / 855 -> 28 / 33.7 / 52 us, 2304x9216 100 / 200 /
// 400 -> 17.5 / 21.8 / 37, 14336x3584 210 / 420 / 840 -> 28 / 33.7 / 45.5 (unscaled
// planes 27.7 / 33.4 / 52, 17.2 / 21.5 / 37, 27.7 / 32.6 / 45); error against 64
// bits 1.2e-7 from x of 2^-120 up (1.5e-7 to 2.8e-7 before).
constexpr int x_planes(XMode xm) { return xm == kXF32 ? 3 : 1; }
// a piece is 16 bytes of x: 8 BF16 or 4 FP32 columns of one batch row
constexpr int x_piece_cols(XMode xm) { return xm == kXF32 ? 4 : 8; }
constexpr int x_row_pieces(XMode xm) { return kTileCols / x_piece_cols(xm); }

// the pieces p = tid + k * threads (k < PC) of a step's slabs
template <int PC>
struct XPieces {
    uint4 v[PC];
};

// Every load here and below is issued unconditionally (indexes clamped into
// the matrix): a load skipped on some path leaves the compiler unable to
// count the loads in flight, and it then waits for all of them - the
// prefetched tiles included - before the next decode.
// The slabs of one step: K group g's slab is x at K tile kb + g + KG i
// (clamped into the split; a clamped slab is loaded but not used). Piece p
// of the step: group g = p / (batch * pieces per row), batch row and piece of
// the row from the remainder. Where a piece runs past the end of x (kXEdge and
// kXF32, the last row's end) the 16 bytes that end there are read instead;
// store_x_slab moves them down. The host sends x of fewer than one piece
// elsewhere.
struct XPiece {
    int g, row, c;  // K group, batch row, piece of the tile's 256 columns
    int kt;
};
template <XMode XM>
__device__ __forceinline__ XPiece x_piece(int batch, int kb, int n, int KG, int i, int p) {
    constexpr int kPer = x_row_pieces(XM);
    p = min(p, KG * batch * kPer - 1);
    XPiece r;
    r.g = p / (batch * kPer);
    const int q = p - r.g * (batch * kPer);
    r.row = q / kPer;
    r.c = q % kPer;
    const int t = r.g + KG * i;
    r.kt = kb + (t < n ? t : n - 1);
    return r;
}

template <XMode XM, int PC>
__device__ __forceinline__ XPieces<PC> load_x_slab(const GemvArgs& a, int batch, int kb, int n, int KG, int i, int tid,
                                                   int threads) {
    XPieces<PC> xr;
    constexpr int kCols = x_piece_cols(XM), kBytes = 16 / kCols;
#pragma unroll
    for (int k = 0; k < PC; ++k) {
        const XPiece r = x_piece<XM>(batch, kb, n, KG, i, tid + k * threads);
        int64_t at = (int64_t)r.row * a.K + (int64_t)r.kt * kTileCols + kCols * r.c;
        if constexpr (XM != kXFast) at = min(at, (int64_t)batch * a.K - kCols);
        const char* src = static_cast<const char*>(a.x) + at * kBytes;
        if constexpr (XM == kXFast)
            xr.v[k] = *reinterpret_cast<const uint4*>(src);
        else
            xr.v[k] = load16_unaligned(src);
    }
    return xr;
}

// v's elements from `shift` on, moved down to 0, those at or past `valid`
// zero: the columns past K of a piece at a row's end (16-bit elements, or
// 32-bit ones with WORDS)
template <bool WORDS>
__device__ __forceinline__ uint4 cut_piece(uint4 v, int shift, int valid) {
    uint32_t e[5] = {v.x, v.y, v.z, v.w, 0u};
    const int dw = WORDS ? shift : shift >> 1;
    uint32_t o[5];
#pragma unroll
    for (int i = 0; i < 5; ++i) {
        o[i] = 0u;
#pragma unroll
        for (int j = i; j < 4; ++j)
            if (j - i == dw) o[i] = e[j];
    }
    if constexpr (!WORDS) {
        if (shift & 1) {
#pragma unroll
            for (int i = 0; i < 4; ++i) o[i] = (o[i] >> 16) | (o[i + 1] << 16);
        }
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        if constexpr (WORDS)
            o[i] = i < valid ? o[i] : 0u;
        else
            o[i] = 2 * i + 1 < valid ? o[i] : 2 * i < valid ? (o[i] & 0xFFFFu) : 0u;
    }
    return make_uint4(o[0], o[1], o[2], o[3]);
}

// One FP32 value as three BF16 planes (bits in the high half): h + kPlaneM (m +
// kPlaneL l) == x for every finite x (to 2^-148: the last bit of a subnormal one
// may fall). An infinity goes to h alone; a NaN's m is a NaN, which no finite
// weight takes away.
constexpr float kPlaneM = 0x1p-7f, kPlaneL = 0x1p-8f;
__device__ __forceinline__ void split3(uint32_t u, uint32_t& h, uint32_t& m, uint32_t& l) {
    const float x = __uint_as_float(u);
    // (a subnormal x, which may be too small for BF16, keeps h from zero, so
    // that an infinite weight meets none; m takes the difference back)
    h = (u & 0xFFFF0000u) | (2u * u - 1u < 0x00FFFFFFu ? 0x10000u : 0u);
    const float r = __builtin_fabsf(x) == INFINITY ? 0.0f : (x - __uint_as_float(h)) * (1.0f / kPlaneM);
    m = __float_as_uint(r) & 0xFFFF0000u;
    l = __float_as_uint((r - __uint_as_float(m)) * (1.0f / kPlaneL));
}

// pieces past the step's slabs repeat the last piece: the same bytes to the
// same address as the thread that owns it. Group g's slab sits at xb + g *
// slab_bytes, its planes plane_bytes apart.
template <XMode XM, int PC>
__device__ __forceinline__ void store_x_slab(const GemvArgs& a, char* xb, int slab_bytes, int plane_bytes,
                                             const XPieces<PC>& xr, int batch, int kb, int n, int KG, int i, int tid,
                                             int threads) {
    constexpr int kCols = x_piece_cols(XM);
#pragma unroll
    for (int k = 0; k < PC; ++k) {
        const XPiece r = x_piece<XM>(batch, kb, n, KG, i, tid + k * threads);
        char* dst = xb + r.g * slab_bytes + r.row * kRowBytes + 2 * kCols * r.c;
        uint4 v = xr.v[k];
        if constexpr (XM != kXFast) {
            const int64_t col = (int64_t)r.kt * kTileCols + kCols * r.c;
            if (col + kCols > a.K) {
                const int64_t past = (int64_t)r.row * a.K + col + kCols - (int64_t)batch * a.K;
                const int64_t valid = a.K - col;
                v = cut_piece<XM == kXF32>(v, (int)min(max(past, (int64_t)0), (int64_t)kCols),
                                           (int)max(valid, (int64_t)0));
            }
        }
        if constexpr (XM == kXF32) {
            const uint32_t u[4] = {v.x, v.y, v.z, v.w};
            uint32_t h[4], m[4], l[4];
#pragma unroll
            for (int e = 0; e < 4; ++e) split3(u[e], h[e], m[e], l[e]);
            // the high halves of two values side by side
            *reinterpret_cast<uint2*>(dst) = make_uint2(perm(h[1], h[0], 0x07060302u), perm(h[3], h[2], 0x07060302u));
            *reinterpret_cast<uint2*>(dst + plane_bytes) =
                make_uint2(perm(m[1], m[0], 0x07060302u), perm(m[3], m[2], 0x07060302u));
            *reinterpret_cast<uint2*>(dst + 2 * plane_bytes) =
                make_uint2(perm(l[1], l[0], 0x07060302u), perm(l[3], l[2], 0x07060302u));
        } else {
            *reinterpret_cast<uint4*>(dst) = v;
        }
    }
}

// Raw-twin rows in the block layout, guarded by the matrix edges and of any
// alignment: the edge-handling form of load_raw_blocks.
__device__ __forceinline__ void load_raw_blocks_edge(uint4 r[4][2], const GemvArgs& a, int tr, int kt, uint32_t lane) {
    const int64_t row = (int64_t)tr * kTileRows + (lane & 15u);
    const uint16_t* p = a.wraw + min(row, a.N - 1) * a.K;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        const int64_t col = (int64_t)kt * kTileCols + block_layout_col(j, lane);
        if (row < a.N && col + 16 <= a.K) {
            r[j][0] = load16_unaligned(p + col);
            r[j][1] = load16_unaligned(p + col + 8);
        } else {
            uint32_t h[8];
#pragma unroll
            for (int q = 0; q < 8; ++q) {
                const int64_t c = col + 2 * q;
                const uint32_t lo = p[min(c, a.K - 1)];
                const uint32_t hi = p[min(c + 1, a.K - 1)];
                h[q] = row < a.N ? ((c < a.K ? lo : 0u) | (c + 1 < a.K ? hi << 16 : 0u)) : 0u;
            }
            r[j][0] = make_uint4(h[0], h[1], h[2], h[3]);
            r[j][1] = make_uint4(h[4], h[5], h[6], h[7]);
        }
    }
}

// weights at columns >= lim of the tile are zeroed (padding can decode to
// +inf when codebook[0] = 255)
__device__ __forceinline__ void zero_past_k(uint32_t w[8], int c0, int lim) {
#pragma unroll
    for (int q = 0; q < 8; ++q) {
        const int c = c0 + 2 * q;
        w[q] = (c >= lim) ? 0u : ((c + 1 >= lim) ? (w[q] & 0xFFFFu) : w[q]);
    }
}

// infinities and NaNs of a BF16 pair zeroed: the m and l planes of a finite x
// may be zero, and must add nothing to what the h plane gives
__device__ __forceinline__ uint32_t finite_pair(uint32_t w) {
    const uint32_t lo = (w & 0x7F80u) == 0x7F80u ? 0u : (w & 0xFFFFu);
    const uint32_t hi = (w & 0x7F800000u) == 0x7F800000u ? 0u : (w & 0xFFFF0000u);
    return lo | hi;
}
__device__ __forceinline__ bool pair_not_finite(uint32_t w) {
    return (w & 0x7F80u) == 0x7F80u || (w & 0x7F800000u) == 0x7F800000u;
}
__device__ __forceinline__ bool has_byte_ff(uint32_t w) { return ((~w - 0x01010101u) & w & 0x80808080u) != 0u; }

// The MFMAs of part p of a tile in the block layout (lane l holds row l % 16,
// columns 16 (4 (l / 16) + p) .. + 15 as 8 BF16 pairs):
// its first and second 8 columns are the A operands of two MFMAs whose B
// operands are the same 8 columns of the x slab (batch row 16 g + l % 16).
// The MFMA's K positions differ between lane groups; A and B agree on them.
template <int BG>
__device__ __forceinline__ void mfma_block_part(const uint32_t w[8], const char* xb, int p, uint32_t lane,
                                                floatx4_t acc[BG]) {
    const int off = (int)(lane & 15u) * kRowBytes + 128 * (int)(lane >> 4) + 32 * p;
#pragma unroll
    for (int h = 0; h < 2; ++h) {
        const bf16x8_t av = __builtin_bit_cast(bf16x8_t, make_uint4(w[4 * h], w[4 * h + 1], w[4 * h + 2], w[4 * h + 3]));
#pragma unroll
        for (int g = 0; g < BG; ++g) {
            const uint4 bv = *reinterpret_cast<const uint4*>(xb + g * 16 * kRowBytes + off + 16 * h);
            acc[g] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(av, __builtin_bit_cast(bf16x8_t, bv), acc[g], 0, 0, 0);
        }
    }
}

template <bool RAW>
struct GemmTile {
    TileSide side;
    TileLoads t;
    uint4 r[RAW ? 4 : 1][2];
};

template <int BG, bool RAW, XMode XM, int M, int PC = kGemmXPieces>
__global__ __launch_bounds__(kGemmMaxThreads) void gemm_kernel(GemvGroupArgs ga, int batch) {
    static_assert(M == 0 || (XM == kXFast && M >= 1), "the slab ring serves the FAST variants");
    SE12_DECLARE_LUT(lut);
    extern __shared__ __attribute__((aligned(16))) char gsm[];
    // the matrix comes from the grid; every argument the block needs goes out
    // in one batch of scalar loads (issued where first used, each would wait
    // behind the one before)
    const GemvArgs a = ga.m[blockIdx.z];
    const int threads = blockDim.x;
    const int R = ga.rows_per_block;
    asm volatile("" ::"s"(a.sm), "s"(a.ec), "s"(a.lut), "s"(a.side), "s"(a.wraw), "s"(a.x), "s"(a.y), "s"(a.K),
                 "s"(a.TR), "s"(a.TC), "s"(a.S), "s"(R), "s"(threads), "s"(batch));
    const int W = threads >> 6;
    const int KG = W / R;
    const int tid = threadIdx.x;
    const uint32_t lane = threadIdx.x & 63u;
    const int w = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const int kg = w / R;
    if ((int)blockIdx.x * R >= a.TR) return;  // past a shorter matrix of a grouped launch
    const int tr = (int)blockIdx.x * R + (w - kg * R);
    const bool active = tr < a.TR;
    const int trl = active ? tr : a.TR - 1;  // row the loads of an idle wave use
    const int S = a.S;
    const int s = blockIdx.y;
    const int kb = (int)(((uint32_t)s * (uint32_t)a.TC) / (uint32_t)S);
    const int ke = (int)(((uint32_t)(s + 1) * (uint32_t)a.TC) / (uint32_t)S);
    const int n = ke - kb;
    const int steps = (n + KG - 1) / KG;  // K group kg takes the split's tiles kg, kg + KG, ...
    const int64_t row_tiles = (int64_t)trl * a.TC;
    constexpr int plane_bytes = x_slab_bytes<BG>();
    constexpr int slab_bytes = x_planes(XM) * plane_bytes;
    // [NB buffers][KG slabs] of x: two with a block barrier per step, or a
    // ring of 2 M with a barrier every M steps
    constexpr int NB = M > 0 ? 2 * M : 2;
    char* xbuf = gsm;

    floatx4_t acc[BG];
#pragma unroll
    for (int g = 0; g < BG; ++g) acc[g] = floatx4_t{0.0f, 0.0f, 0.0f, 0.0f};
    floatx4_t low[XM == kXF32 ? BG : 1];  // the m and l planes' sums, times 1 / kPlaneM
    if constexpr (XM == kXF32) {
#pragma unroll
        for (int g = 0; g < BG; ++g) low[g] = floatx4_t{0.0f, 0.0f, 0.0f, 0.0f};
    }
    bool lut_special = false;  // the codebook holds exponent 255

    auto load_tile_i = [&](GemmTile<RAW>& t, int i) {
        const int j = kg + KG * i;
        const int kt = kb + (j < n ? j : n - 1);
        if constexpr (RAW && XM != kXFast) {
            load_raw_blocks_edge(t.r, a, trl, kt, lane);
        } else if constexpr (RAW) {
            load_raw_blocks(t.r, a.wraw, a.K, trl, kt, lane);
        } else {
            load_tile_block_order(t.t, t.side, a.sm, a.ec, a.side, row_tiles + kt, lane);
        }
    };
    auto use_tile = [&](GemmTile<RAW>& t, int i) {
        const int kt = kb + kg + KG * i;
        const char* xb = xbuf + ((i % NB) * KG + kg) * slab_bytes;
        // a decoded tile's (or raw tile's) 4 parts: edge columns zeroed, then
        // the MFMAs; `special` (wave-uniform): it may hold an infinity or NaN
        auto mfma_tile = [&](uint32_t (&wv)[4][8], bool special) {
            if constexpr (XM != kXFast) {
                const int64_t lim = a.K - (int64_t)kt * kTileCols;
                if (lim < kTileCols) {
#pragma unroll
                    for (int p = 0; p < 4; ++p) zero_past_k(wv[p], block_layout_col(p, lane), (int)lim);
                }
            }
            if constexpr (XM != kXF32) {
#pragma unroll
                for (int p = 0; p < 4; ++p) mfma_block_part<BG>(wv[p], xb, p, lane, acc);
            } else {
                floatx4_t tile[BG];
#pragma unroll
                for (int g = 0; g < BG; ++g) tile[g] = floatx4_t{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
                for (int p = 0; p < 4; ++p) mfma_block_part<BG>(wv[p], xb, p, lane, tile);
                if (special) {
#pragma unroll
                    for (int p = 0; p < 4; ++p)
#pragma unroll
                        for (int q = 0; q < 8; ++q) wv[p][q] = finite_pair(wv[p][q]);
                }
#pragma unroll
                for (int g = 0; g < BG; ++g) {
                    acc[g] += tile[g];
                    tile[g] = floatx4_t{0.0f, 0.0f, 0.0f, 0.0f};
                }
                if constexpr (BG > 1) __builtin_amdgcn_sched_barrier(0);   // no registers for both at once
#pragma unroll
                for (int p = 0; p < 4; ++p) mfma_block_part<BG>(wv[p], xb + 2 * plane_bytes, p, lane, tile);
#pragma unroll
                for (int p = 0; p < 4; ++p) mfma_block_part<BG>(wv[p], xb + plane_bytes, p, lane, low);
#pragma unroll
                for (int g = 0; g < BG; ++g) low[g] += tile[g] * kPlaneL;
            }
        };
        // raw words: looked at one by one (FP32 x only)
        auto raw_special = [&](const uint32_t (&wv)[4][8]) {
            bool any = false;
            if constexpr (XM == kXF32) {
#pragma unroll
                for (int p = 0; p < 4; ++p)
#pragma unroll
                    for (int q = 0; q < 8; ++q) any = any || pair_not_finite(wv[p][q]);
            }
            return wave_any(any);
        };
        if constexpr (RAW) {
            // block layout: each part's 16 columns are the A operands as loaded
            uint32_t wv[4][8];
#pragma unroll
            for (int p = 0; p < 4; ++p) {
                wv[p][0] = t.r[p][0].x; wv[p][1] = t.r[p][0].y; wv[p][2] = t.r[p][0].z; wv[p][3] = t.r[p][0].w;
                wv[p][4] = t.r[p][1].x; wv[p][5] = t.r[p][1].y; wv[p][6] = t.r[p][1].z; wv[p][7] = t.r[p][1].w;
            }
            mfma_tile(wv, raw_special(wv));
        } else {
            const uint32_t info = side_info(t.side, 0);
            if (info_is_fallback(info)) {
                const int16_t* raw = raw_tile_ptr(info, a.fb_raw, a.ovf_raw);
                uint32_t wv[4][8];
#pragma unroll
                for (int p = 0; p < 4; ++p) raw_block_part(raw, p, lane, wv[p]);
                wait_vector_loads();  // rare path: keeps the common path's waits exact
                mfma_tile(wv, raw_special(wv));
            } else {
                // whole-line loads (4 tile rows per instruction) into the block
                // layout, in place (the slot is reloaded next); each part's
                // patterns merged with its sm bytes as soon as looked up;
                // escapes only set exponent bits, which the merge takes from
                // the patterns, so they patch the merged words
                chunks_to_blocks(t.t);
                uint32_t wv[4][8];
#pragma unroll
                for (int p = 0; p < 4; ++p) {
                    uint32_t pat[8];
                    lookup_chunk(lut, t.t.ec[p], pat);
                    merge_chunk(pat, t.t.sm[p], wv[p]);
                }
                patch_tile_escapes<kBlockLayout>(wv, info, t.side, 0, lane);
                bool special = false;
                if constexpr (XM == kXF32) {
                    special = lut_special;
                    if (info_escapes(info) != 0u) {
                        const uint4 e = side_esc(t.side, 0);
                        special = special || has_byte_ff(e.x) || has_byte_ff(e.y) || has_byte_ff(e.z) || has_byte_ff(e.w);
                    }
                }
                mfma_tile(wv, special);
            }
        }
    };

    uint4 lutv;
    if constexpr (!RAW) lutv = reinterpret_cast<const uint4*>(a.lut)[lane];
    __builtin_amdgcn_sched_barrier(0);
    // rings of three: tile i's streams are requested two steps before its
    // decode, x slab i's pieces two steps before they are stored to LDS
    // Tile streams and x pieces are requested D - 1 steps ahead of their
    // use (D = 3): under a full-bandwidth stream
    // even the L2 hits of x take about a step to return. The loop body holds
    // D steps so that every step's loads are issued on every path that goes
    // on (loads past the last tile reload it): a load skipped on some path
    // would make the compiler wait for all loads in flight. Slab i + 1 is
    // stored to LDS at the end of step i.
    auto x_step = [&](int i) { return load_x_slab<XM, PC>(a, batch, kb, n, KG, i, tid, threads); };
    auto x_store = [&](char* to, const XPieces<PC>& xr, int i) {
        store_x_slab<XM, PC>(a, to, slab_bytes, plane_bytes, xr, batch, kb, n, KG, i, tid, threads);
    };
    // FP32 x: exponent 255 in the pair table (each lane's 4 entries)
    auto note_lut = [&]() {
        if constexpr (XM == kXF32 && !RAW)
            lut_special = wave_any(pair_not_finite(lutv.x) || pair_not_finite(lutv.y) || pair_not_finite(lutv.z) ||
                                   pair_not_finite(lutv.w));
    };
    auto has_tile = [&](int i) { return kg + KG * i < n; };
    if constexpr (M > 0) {
        // Slab ring: the slabs of step j sit in buffer j % NB (NB = 2 M);
        // every thread stores its pieces of the slabs of step j during step
        // j - M (pieces requested one step before; the prologue stores steps
        // 0 .. M - 1), and the block meets only before steps M, 2 M, ...
        // Slab j is read at step j after the meeting before the multiple of M
        // in (j - M, j], so after every wave's store of it; storing slab j
        // during step j - M overwrites slab j - 2 M, which every wave read
        // before the meeting before the multiple of M in (j - 2 M, j - M].
        // Fewer meetings let the waves' tile
        // arrivals even out (14336x3584 B = 32: 24.5 us against 26.0 with one
        // per step).
        constexpr int L = M;
        auto buf = [&](int j) { return xbuf + (j % NB) * KG * slab_bytes; };
        GemmTile<RAW> t0, t1, t2;
        load_tile_i(t0, 0);
        load_tile_i(t1, 1);
        XPieces<PC> xp[L];
#pragma unroll
        for (int j = 0; j < L; ++j) xp[j] = x_step(j);
        XPieces<PC> x0 = x_step(L), x1, x2;
        if constexpr (!RAW) store_block_lut(lut, lutv, lane);
#pragma unroll
        for (int j = 0; j < L; ++j) x_store(buf(j), xp[j], j);
        lds_barrier();  // the pair table and the slabs of steps 0 .. L - 1 are in LDS
        auto step = [&](GemmTile<RAW>& cur, GemmTile<RAW>& ahead, const XPieces<PC>& x_next, XPieces<PC>& x_ahead, int i) {
            x_ahead = x_step(i + L + 1);
            load_tile_i(ahead, i + 2);
            if (i > 0 && i % M == 0) lds_barrier();
            if (has_tile(i)) use_tile(cur, i);  // an idle wave decodes row trl; its sums are dropped
            x_store(buf(i + L), x_next, i + L);
        };
        int i = 0;
        while (true) {
            step(t0, t2, x0, x1, i);
            if (++i >= steps) break;
            step(t1, t0, x1, x2, i);
            if (++i >= steps) break;
            step(t2, t1, x2, x0, i);
            if (++i >= steps) break;
        }
    } else if constexpr (XM != kXFast) {
        // the edge-handling variants: tiles one step ahead (their x address
        // and cut arithmetic leaves no registers for a third tile)
        GemmTile<RAW> t0, t1;
        load_tile_i(t0, 0);
        XPieces<PC> x0 = x_step(0), x1 = x_step(1);
        if constexpr (!RAW) store_block_lut(lut, lutv, lane);
        note_lut();
        x_store(xbuf, x0, 0);
        lds_barrier();
        auto step = [&](GemmTile<RAW>& cur, GemmTile<RAW>& ahead, const XPieces<PC>& x_next, XPieces<PC>& x_ahead, int i) {
            load_tile_i(ahead, i + 1);
            x_ahead = x_step(i + 2);
            __builtin_amdgcn_sched_barrier(0);
            if (has_tile(i)) use_tile(cur, i);
            __builtin_amdgcn_sched_barrier(0);
            x_store(xbuf + ((i + 1) & 1) * KG * slab_bytes, x_next, i + 1);
            lds_barrier();
        };
        int i = 0;
        while (true) {
            step(t0, t1, x1, x0, i);
            if (++i >= steps) break;
            step(t1, t0, x0, x1, i);
            if (++i >= steps) break;
        }
    } else {
        GemmTile<RAW> t0, t1, t2;
        load_tile_i(t0, 0);
        XPieces<PC> x0 = x_step(0);
        load_tile_i(t1, 1);
        XPieces<PC> x1 = x_step(1);
        XPieces<PC> x2;
        if constexpr (!RAW) store_block_lut(lut, lutv, lane);
        x_store(xbuf, x0, 0);
        lds_barrier();
        auto step = [&](GemmTile<RAW>& cur, GemmTile<RAW>& ahead, const XPieces<PC>& x_next, XPieces<PC>& x_ahead,
                        int i) {
            x_ahead = x_step(i + 2);
            load_tile_i(ahead, i + 2);
            if (has_tile(i)) use_tile(cur, i);  // an idle wave decodes row trl; its sums are dropped
            x_store(xbuf + ((i + 1) & 1) * KG * slab_bytes, x_next, i + 1);
            lds_barrier();
        };
        // the loop leaves after the last step (not after a group of three):
        // past it nothing waits on the loads it issued
        int i = 0;
        while (true) {
            step(t0, t2, x1, x2, i);
            if (++i >= steps) break;
            step(t1, t0, x2, x0, i);
            if (++i >= steps) break;
            step(t2, t1, x0, x1, i);
            if (++i >= steps) break;
        }
    }
    if constexpr (XM == kXF32) {
#pragma unroll
        for (int g = 0; g < BG; ++g) acc[g] += low[g] * kPlaneM;
    }
    // the K groups of a tile row: groups 1..KG-1 hand their sums to group 0
    // through LDS (the x slabs are no longer read: every wave passed the
    // last step's barrier), which adds them in ascending group order
    if (KG > 1) {
        // [KG - 1][R][64 lanes][BG][4]: over the x slabs, which every wave
        // has passed the last barrier of, or past the slab ring, whose last
        // slabs other waves may still read
        float* red = reinterpret_cast<float*>(gsm + (M > 0 ? NB * KG * slab_bytes : 0));
        const int rw = w - kg * R;
        if (kg > 0) {
#pragma unroll
            for (int g = 0; g < BG; ++g)
                *reinterpret_cast<floatx4_t*>(red + ((((kg - 1) * R + rw) * 64 + (int)lane) * BG + g) * 4) = acc[g];
        }
        lds_barrier();
        if (kg > 0) return;
        for (int k = 1; k < KG; ++k)
#pragma unroll
            for (int g = 0; g < BG; ++g)
                acc[g] += *reinterpret_cast<const floatx4_t*>(red + ((((k - 1) * R + rw) * 64 + (int)lane) * BG + g) * 4);
    }
    if (!active) return;

    // accumulator layout: lane l holds D[4 * (l / 16) + e][l % 16] of each
    // batch group: tile row 4 * (l / 16) + e, batch row 16 * g + l % 16
    const int64_t n0 = (int64_t)tr * kTileRows + 4 * (int)(lane >> 4);
    // the row's sum of squares (GemvEpilogue::row_ss): lanes l, l + 16, l + 32
    // and l + 48 hold the quads of batch row 16 g + l; rows past N count 0
    float* const row_ss = ga.epi.row_ss;
    auto store_row_ss = [&](const float* sums, int g) {
        if (!row_ss) return;
        float v[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) v[e] = n0 + e < a.N ? sums[e] : 0.0f;
        float q = quad_sumsq(v);
        q += __shfl_xor(q, 16, 64);
        q += __shfl_xor(q, 32, 64);
        const int b = 16 * g + (int)lane;
        if (lane < 16u && b < batch) row_ss[(int64_t)b * a.TR + tr] = q;
    };
    if (S == 1) {
#pragma unroll
        for (int g = 0; g < BG; ++g) {
            const int b = 16 * g + (int)(lane & 15u);
            if (b < batch)
#pragma unroll
                for (int e = 0; e < 4; ++e)
                    if (n0 + e < a.N) a.y[(int64_t)b * a.N + n0 + e] = acc[g][e];
            const float sums[4] = {acc[g][0], acc[g][1], acc[g][2], acc[g][3]};
            store_row_ss(sums, g);
        }
        return;
    }
    // split-K: device-scope partial stores, then the wave's arrival on the
    // tile row's counter; the last of the S waves adds the partials in order
#pragma unroll
    for (int g = 0; g < BG; ++g) {
        const int b = 16 * g + (int)(lane & 15u);
        if (b < batch) {
            const float v[4] = {acc[g][0], acc[g][1], acc[g][2], acc[g][3]};
            store_partial4(&a.partial[((int64_t)s * batch + b) * a.Np + n0], v);
        }
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    int old = 0;
    if (lane == 0) old = __hip_atomic_fetch_add(&a.counters[tr], 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    old = __builtin_amdgcn_readfirstlane(old);
    if (old != S - 1) return;
#pragma unroll
    for (int g = 0; g < BG; ++g) {
        const int b = 16 * g + (int)(lane & 15u);
        float sum[4] = {0.0f, 0.0f, 0.0f, 0.0f};
        if (b < batch) {
            // every split's loads first (in groups of 8), then the adds in
            // ascending split order
            for (int s0 = 0; s0 < S; s0 += 8) {
                uint64_t lo[8], hi[8];
#pragma unroll
                for (int k = 0; k < 8; ++k) {
                    lo[k] = hi[k] = 0;
                    if (s0 + k < S) {
                        const float* pp = &a.partial[((int64_t)(s0 + k) * batch + b) * a.Np + n0];
                        lo[k] = load_partial2(pp);
                        hi[k] = load_partial2(pp + 2);
                    }
                }
#pragma unroll
                for (int k = 0; k < 8; ++k)
                    if (s0 + k < S) {
                        sum[0] += partial_lo(lo[k]);
                        sum[1] += partial_hi(lo[k]);
                        sum[2] += partial_lo(hi[k]);
                        sum[3] += partial_hi(hi[k]);
                    }
            }
#pragma unroll
            for (int e = 0; e < 4; ++e)
                if (n0 + e < a.N) a.y[(int64_t)b * a.N + n0 + e] = sum[e];
        }
        store_row_ss(sum, g);
    }
    if (lane == 0) __hip_atomic_store(&a.counters[tr], 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

namespace {

template <int BG, bool RAW>
hipError_t gemm_b(const GemvGroupArgs& a, int batch, const GemvPlan& p, hipStream_t stream) {
    const dim3 grid(group_grid_x(a), a.m[0].S, a.count), block(p.waves * 64);
    const int pieces = (batch * x_row_pieces(kXF32) + p.waves * 64 - 1) / (p.waves * 64);   // FP32 x: per thread and step
    if (p.xf32 && BG == 1 && pieces <= 1)
        hipLaunchKernelGGL((gemm_kernel<1, RAW, kXF32, 0, 1>), grid, block, p.lds, stream, a, batch);
    else if (p.xf32 && BG == 1 && pieces <= 2)
        hipLaunchKernelGGL((gemm_kernel<1, RAW, kXF32, 0, 2>), grid, block, p.lds, stream, a, batch);
    else if (p.xf32)
        hipLaunchKernelGGL((gemm_kernel<BG, RAW, kXF32, 0>), grid, block, p.lds, stream, a, batch);
    else if (p.generic)
        hipLaunchKernelGGL((gemm_kernel<BG, RAW, kXEdge, 0>), grid, block, p.lds, stream, a, batch);
    else if (p.slab_ring == kGemmSlabRing)
        hipLaunchKernelGGL((gemm_kernel<BG, RAW, kXFast, kGemmSlabRing>), grid, block, p.lds, stream, a, batch);
    else
        hipLaunchKernelGGL((gemm_kernel<BG, RAW, kXFast, 0>), grid, block, p.lds, stream, a, batch);
    return hipGetLastError();
}

}  // namespace

size_t gemm_lds_bytes(int waves, int batch, int slab_ring, bool xf32) {
    const int bg = batch > 16 ? 2 : 1, planes = x_planes(xf32 ? kXF32 : kXFast);
    const int rows = gemm_min_waves(batch, xf32), kgroups = std::max(1, waves / rows);
    const size_t sums = (size_t)(kgroups - 1) * rows * 64 * bg * 4 * sizeof(float);
    if (slab_ring > 0) return (size_t)2 * slab_ring * kgroups * 16 * bg * kRowBytes + sums;
    const size_t slabs = (size_t)2 * kgroups * planes * 16 * bg * kRowBytes;
    return std::max(slabs, sums);
}

hipError_t launch_gemm(const GemvGroupArgs& a, int batch, const GemvPlan& p, hipStream_t stream) {
    const int rows = gemm_min_waves(batch, p.xf32);
    if (batch < 1 || batch > 32 || p.waves % rows != 0 || a.rows_per_block != rows) return hipErrorInvalidValue;
    if (batch > 16) return p.raw ? gemm_b<2, true>(a, batch, p, stream) : gemm_b<2, false>(a, batch, p, stream);
    return p.raw ? gemm_b<1, true>(a, batch, p, stream) : gemm_b<1, false>(a, batch, p, stream);
}

}  // namespace se12

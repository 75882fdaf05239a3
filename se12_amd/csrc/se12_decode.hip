// Decode-only kernels: SE12 streams -> row-major BF16 bits, bit-exact with the
// reference decoder (lws/domain/se12/codec.py:144-186). A wave decodes a
// 16x256 tile with the same per-lane routine as the fused GEMV and writes its
// rows straight to the cropped [rows, cols] output (the whole-matrix decode
// streams several tiles per wave; the row decode takes one row of four K
// tiles per wave), replacing the reference's
// one-thread-per-tile kernel plus device untile/crop
// (lws/adapters/cuda/kernels/se12_decode.cu:12-43,
// lws/adapters/cuda/se12_decoder.py:147-185).
//
// Also here: bind's per-tile side records. A fallback tile's word holds the
// tile's rank among all fallback tiles (cumsum(bitmap bits) - 1, as in
// lws/adapters/cuda/gemv.py:47-53); any other tile's which of its four 4-row
// chunks hold escape codes, their count and positions (one wave per tile reads
// the tile's `ec` bytes). The kernels read the records instead of the bitmap.
#include "se12_device.hpp"
#include "se12_internal.hpp"
#include "se12_step_math.hpp"

#include <type_traits>

namespace se12 {

constexpr int kDecodeWaves = 4;

__device__ __forceinline__ void store16(uint16_t* out_row, int64_t col, int64_t K, bool vec_ok, const uint32_t w[8]) {
    if (vec_ok && col + 16 <= K) {
        reinterpret_cast<uint4*>(out_row + col)[0] = make_uint4(w[0], w[1], w[2], w[3]);
        reinterpret_cast<uint4*>(out_row + col)[1] = make_uint4(w[4], w[5], w[6], w[7]);
    } else {
#pragma unroll
        for (int i = 0; i < 16; ++i)
            if (col + i < K) out_row[col + i] = (uint16_t)(w[i >> 1] >> (16 * (i & 1)));
    }
}

// 8 decoded weights (4 BF16 pairs) to out_row[col .. col + 8) clipped at K:
// one 16-byte nontemporal store when the output allows it (streamed: the
// decoded matrix is written once and read later by another kernel).
__device__ __forceinline__ void store8(uint16_t* out_row, int64_t col, int64_t K, bool vec_ok, const uint32_t w[4]) {
    typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
    if (vec_ok && col + 8 <= K) {
        const u32x4 v = {w[0], w[1], w[2], w[3]};
        __builtin_nontemporal_store(v, reinterpret_cast<u32x4*>(out_row + col));
    } else {
#pragma unroll
        for (int i = 0; i < 8; ++i)
            if (col + i < K) out_row[col + i] = (uint16_t)(w[i >> 1] >> (16 * (i & 1)));
    }
}

// Patches the escapes of a tile in the half layout as its ec words show them:
// parts, then lanes, then weights are the row-major order in which escapes take
// the esc slots (past the 15th: the last, like the reference's clip). Scalar work
// per escape; a tile of N(0, 0.02) weights holds less than one. esc: lane k holds
// word k of the slots.
__device__ __forceinline__ void patch_found_escapes(uint32_t pat[4][8], const HalfTileLoads& t, uint32_t esc, uint32_t lane) {
    uint32_t found[8], any = 0;
#pragma unroll
    for (int p = 0; p < 8; ++p) any |= found[p] = escape_nibbles(t.ec[p]);
    if (!wave_any(any != 0u)) return;
    uint32_t r = 0;
#pragma unroll
    for (int p = 0; p < 8; ++p) {
        uint32_t* q = &pat[p >> 1][4 * (p & 1)];
        for (uint64_t lanes = __builtin_amdgcn_ballot_w64(found[p] != 0u); lanes != 0; lanes &= lanes - 1) {
            const int owner = __builtin_ctzll(lanes);
            uint32_t m = (uint32_t)__builtin_amdgcn_readlane((int)found[p], owner);
            for (; m != 0u; m &= m - 1u, ++r) {
                const uint32_t c = (uint32_t)__builtin_ctz(m) >> 2, slot = r < 15u ? r : 15u;
                const uint32_t e = ((uint32_t)__builtin_amdgcn_readlane((int)esc, (int)(slot >> 2)) >> (8u * (slot & 3u))) & 0xFFu;
                const uint32_t v = (int)lane == owner ? e << ((c & 1u) ? 23u : 7u) : 0u;
#pragma unroll
                for (uint32_t i = 0; i < 4; ++i) q[i] |= (c >> 1) == i ? v : 0u;
            }
        }
    }
}

// Whole-matrix decode: nw waves stream the tiles, wave g taking tiles g,
// g + nw, ... (the waves read a moving window of the tile-major streams),
// each with the next tile's loads in flight while it decodes and stores the
// current one. The last tile loads nothing after it (a wave cannot end
// before its loads land), and every load inside the loop is issued on every
// path, so the compiler's wait counts stay exact.
//
// Lane layout (the half layout): part p = 0..7 of a tile covers tile rows
// 2p and 2p + 1; lane l takes row 2p + l / 32, columns 8 (l % 32) .. + 7
// (8 bytes of sm, 4 of ec), so each part's store instruction writes two
// whole 512-byte row segments, 16 contiguous bytes per lane. (The fused
// kernels' chunk layout gives each lane 16 columns, whose two 16-byte stores
// each write alternate halves of 32-byte pieces: 2304x9216 took 19.0 us
// with it against 15.7 here, the stores nontemporal in both; 14336x3584
// 39.0 against 33.5.)
//
// Up to kMaxGroup matrices share a launch, each with blocks of its own (the pair
// table in LDS is a matrix's): the
// seven matrices of a Gemma-2-2B layer take 59.5 us in four launches against 70 in
// seven, mostly on q, k, v (9.0 us), whose own launches end before they fill HBM.
//
// DIRECT: from the format's streams alone, for a matrix that is decoded once and
// never bound: the fallback bit and the 16 esc bytes are read per tile, the
// escapes found in the ec words that the tile holds anyway. A fallback rank past
// raw_tiles gives zeros (the caller refuses such streams).
//
// One matrix has arguments of its own (DecodeOne): as a group of one, with the
// search for the block's matrix and its place in the arguments, 9216x2304 took
// 14.9 us a call against 14.5, all of it raw tiles 20.9 against 20.5.
struct DecodeOne {
    DecodeArgs m[1];
    int64_t nw[1];
};

template <bool DIRECT, typename Args>
__global__ __launch_bounds__(kDecodeWaves * kWave) void decode_stream_kernel(Args grp) {
    constexpr bool GROUP = std::is_same<Args, DecodeGroup>::value;
    SE12_DECLARE_LUT(lut);
    int mi = 0;
    if constexpr (GROUP)
        while (mi + 1 < grp.count && (int)blockIdx.x >= grp.block0[mi + 1]) ++mi;
    const DecodeArgs a = grp.m[mi];
    const int64_t nw = grp.nw[mi];
    const int tid = threadIdx.x;
    const uint32_t lane = tid & 63;
    const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
    // tile indices in 32 bits (the library refuses matrices of 2^31 tiles or
    // more), so the per-tile division is a 32-bit one
    const uint32_t T = (uint32_t)a.T, NW = (uint32_t)nw, TC = (uint32_t)a.TC;
    uint32_t block = blockIdx.x;
    if constexpr (GROUP) block -= (uint32_t)grp.block0[mi];
    const uint32_t g = block * kDecodeWaves + (uint32_t)w;
    const uint32_t n = g < NW && g < T ? (T - 1u - g) / NW + 1u : 0u;  // tiles of this wave
    struct Slot {
        TileSide side;        // DIRECT: lane k % 4 the k-th word of the esc slots
        HalfTileLoads t;
        uint32_t bits;        // DIRECT: the tile's byte of the bitmap
    };
    auto load = [&](Slot& sl, uint32_t i) {
        const uint32_t tile = min(g + i * NW, T - 1u);
        if constexpr (DIRECT) {
            sl.side.rec = reinterpret_cast<const uint32_t*>(a.esc + (int64_t)tile * kEscBudget)[lane & 3u];
            sl.bits = a.bitmap[tile >> 3];
        } else {
            load_side(sl.side, a.side, tile, lane);
        }
        load_tile_half(sl.t, a.sm, a.ec, tile, lane);
    };
    const bool vec_ok = a.out_vec_ok != 0;
    RankCursor ranked;   // DIRECT
    auto emit = [&](const Slot& sl, uint32_t i) {
        const uint32_t tile = g + i * NW;
        const int tr = (int)(tile / TC);
        const int kt = (int)(tile - (uint32_t)tr * TC);
        const int64_t col = (int64_t)kt * kTileCols + 8 * (lane & 31u);
        const int64_t row0 = (int64_t)tr * kTileRows + (lane >> 5);
        const bool direct_fallback =
            DIRECT && ((__builtin_amdgcn_readfirstlane((int)sl.bits) >> (7u - (tile & 7u))) & 1) != 0;
        const uint32_t info = DIRECT ? (direct_fallback ? kInfoFallback : 0u) : side_info(sl.side, 0);
        // wave-uniform: a tile inside the matrix whose rows take whole
        // 16-byte stores needs no per-lane guard
        const bool full = vec_ok && (int64_t)(tr + 1) * kTileRows <= a.N && (int64_t)(kt + 1) * kTileCols <= a.K;
        uint16_t* const out0 = a.out + row0 * a.K + col;
        auto put = [&](int p, const uint32_t wv[4]) {
            if (full) {
                typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
                const u32x4 v = {wv[0], wv[1], wv[2], wv[3]};
                __builtin_nontemporal_store(v, reinterpret_cast<u32x4*>(out0 + 2 * p * a.K));
            } else if (row0 + 2 * p < a.N) {
                store8(a.out + (row0 + 2 * p) * a.K, col, a.K, vec_ok, wv);
            }
        };
        if (info_is_fallback(info)) {
            // a tile read as raw BF16 (tile-local row-major, like sm)
            uint4 r[8];
            const int64_t rank = DIRECT ? fallback_rank(a.bitmap, tile, lane, ranked) : 0;
            if (!DIRECT || rank < a.raw_tiles) {
                const int16_t* raw = (DIRECT ? a.fb_raw + rank * kTile : raw_tile_ptr(info, a.fb_raw, a.ovf_raw)) + 8 * lane;
#pragma unroll
                for (int p = 0; p < 8; ++p) r[p] = stream_load(reinterpret_cast<const uint4*>(raw + 512 * p));
            } else {
#pragma unroll
                for (int p = 0; p < 8; ++p) r[p] = make_uint4(0u, 0u, 0u, 0u);
            }
            wait_vector_loads();  // rare path: keeps the common path's waits exact
#pragma unroll
            for (int p = 0; p < 8; ++p) {
                const uint32_t wv[4] = {r[p].x, r[p].y, r[p].z, r[p].w};
                put(p, wv);
            }
        } else {
            uint32_t pat[4][8];
            lookup_tile_half(lut, sl.t, pat);
            if constexpr (DIRECT)
                patch_found_escapes(pat, sl.t, sl.side.rec, lane);
            else
                patch_tile_escapes<kHalfLayout>(pat, info, sl.side, 0, lane);
#pragma unroll
            for (int p = 0; p < 8; ++p) {
                uint32_t wv[4];
                merge_part_half(pat, sl.t, p, wv);
                put(p, wv);
            }
        }
    };
    // the pair table, then the first tile (a wave past the grid's waves
    // re-loads tile g's clamp, so that the table's wait count is exact)
    static_assert(kDecodeWaves * kWave == 256, "a thread per entry of the pair table");
    uint4 lutv = make_uint4(0u, 0u, 0u, 0u);
    uint8_t code[2];
    if constexpr (DIRECT) {
        code[0] = a.codebook[min(tid & 15, kCodebook - 1)];
        code[1] = a.codebook[min(tid >> 4, kCodebook - 1)];
    } else {
        lutv = reinterpret_cast<const uint4*>(a.lut)[lane];
    }
    Slot s0, s1;
    load(s0, 0);
    if constexpr (DIRECT)
        lut[tid] = ((tid & 15) < kCodebook ? (uint32_t)code[0] << 7 : 0u) | ((tid >> 4) < kCodebook ? (uint32_t)code[1] << 23 : 0u);
    else
        store_block_lut(lut, lutv, lane);
    lds_barrier();
    if (n == 0) return;
    uint32_t i = 0;
    while (true) {
        if (i + 1 >= n) {
            emit(s0, i);
            break;
        }
        load(s1, i + 1);
        emit(s0, i);
        if (++i + 1 >= n) {
            emit(s1, i);
            break;
        }
        load(s0, i + 1);
        emit(s1, i);
        ++i;
    }
}

// Decodes single rows, in request order: one wave per (row, 4 K tiles). Lane
// 16 s + c takes 16 columns of the row in the wave's s-th tile, so the wave
// reads the row's own 256 bytes of sm and 128 of ec per tile (not the tile's
// 6 KB) and the four tiles' side records in one 256-byte load; the record's
// fields reach the 16 lanes of its tile by lane shuffles. Rows outside the
// matrix give zeros. SCALED: each weight times `scale` (a BF16 value), rounded
// to BF16. Bound by latency and the scattered 128..256-byte reads: 2,048 rows of
// 256000x2304 25.9 -> 6.3 us against a wave decoding the whole tile for one of
// its rows (and no separate multiply, 6.8 us, with a factor copied from the host).
constexpr int kRowTiles = 4;

template <bool SCALED>
__global__ __launch_bounds__(kDecodeWaves * kWave) void decode_rows_kernel(DecodeArgs a, float scale) {
    SE12_DECLARE_LUT(lut);
    const int tid = threadIdx.x;
    const uint32_t lane = tid & 63;
    const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
    const uint4 lutv = reinterpret_cast<const uint4*>(a.lut)[lane];
    const int64_t groups = (a.TC + kRowTiles - 1) / kRowTiles;
    const int64_t item = (int64_t)blockIdx.x * kDecodeWaves + w;
    const bool here = item < a.items;
    const int64_t ri = (here ? item : a.items - 1) / groups;
    const int64_t row = a.rows[ri];
    const int kt = (int)((here ? item : a.items - 1) - ri * groups) * kRowTiles + (int)(lane >> 4);
    const bool inside = row >= 0 && row < a.N;
    const int64_t tile = (inside ? row / kTileRows : 0) * a.TC + (kt < a.TC ? kt : a.TC - 1);
    const uint32_t lr = (uint32_t)row & (kTileRows - 1), c = lane & 15u;
    const uint32_t rec = a.side[tile * kSideWords + c];
    const uint4 sm = *reinterpret_cast<const uint4*>(a.sm + tile * kTile + lr * kTileCols + 16 * c);
    const uint2 ec = *reinterpret_cast<const uint2*>(a.ec + tile * (kTile / 2) + lr * (kTileCols / 2) + 8 * c);
    store_block_lut(lut, lutv, lane);
    lds_barrier();

    // word k of this lane's record, from the lane of its 16 that loaded it
    auto word = [&](int k) { return (uint32_t)__shfl((int)rec, (int)(lane & 48u) + k, 64); };
    const uint32_t info = word(0);
    uint32_t pat[8], v[8];
    lookup_chunk(lut, ec, pat);
    const uint32_t n = info_is_fallback(info) ? 0u : info_escapes(info);
    // the tile's listed escapes that fall on this lane's columns of this row
    for (uint32_t k = 0; wave_any(k < n); ++k) {
        const uint32_t p = (word(5 + (int)(k >> 1)) >> (16 * (k & 1u))) & 0xFFFFu;
        const uint32_t e = (word(1 + (int)(k >> 2)) >> (8 * (k & 3u))) & 0xFFu;
        if (k < n && (p >> 4) == ((lr << 4) | c)) patch_exponent(pat, p & 15u, e);
    }
    merge_chunk(pat, sm, v);
    if (info_is_fallback(info)) {
        const uint4* raw = reinterpret_cast<const uint4*>(raw_tile_ptr(info, a.fb_raw, a.ovf_raw) + lr * kTileCols + 16 * c);
        const uint4 r0 = raw[0], r1 = raw[1];
        v[0] = r0.x; v[1] = r0.y; v[2] = r0.z; v[3] = r0.w;
        v[4] = r1.x; v[5] = r1.y; v[6] = r1.z; v[7] = r1.w;
    }
    if (!here || kt >= a.TC) return;
    // (a NaN is the framework's, 0x7FC0 whatever the weight's sign and payload)
    auto scaled = [&](uint32_t w) {
        const float f = __uint_as_float(w) * scale;
        return f != f ? __uint_as_float(0x7FC00000u) : f;
    };
#pragma unroll
    for (int i = 0; i < 8; ++i) {
        if (!inside) v[i] = 0u;
        if constexpr (SCALED) v[i] = se12step::f_to_bf16x2(scaled(v[i] << 16), scaled(v[i] & 0xFFFF0000u));
    }
    store16(a.out + ri * a.K, (int64_t)kt * kTileCols + 16 * c, a.K, a.out_vec_ok != 0, v);
}

// waves of the whole-matrix decode per CU (MI355X, cold HBM, half layout:
// 2304x9216 15.65 us with 4, 16.6 with 6, 15.6 with 8, 15.55 with 12;
// 14336x3584 33.5 / 36.5 / 33.6 / 33.9)
constexpr int kDecodeStreamWavesPerCu = 4;

template <bool DIRECT>
static hipError_t launch_decode_one(const DecodeArgs& a, hipStream_t stream, int cu_count) {
    const DecodeOne one{{a}, {std::min<int64_t>(a.T, (int64_t)std::max(1, cu_count) * kDecodeStreamWavesPerCu)}};
    const dim3 grid((uint32_t)((one.nw[0] + kDecodeWaves - 1) / kDecodeWaves)), block(kDecodeWaves * kWave);
    hipLaunchKernelGGL((decode_stream_kernel<DIRECT, DecodeOne>), grid, block, 0, stream, one);
    return hipGetLastError();
}

// The waves are shared out by the matrices' tiles, in whole blocks.
hipError_t launch_decode(DecodeGroup& g, hipStream_t stream, int cu_count) {
    if (g.count == 1) return launch_decode_one<false>(g.m[0], stream, cu_count);
    const int64_t waves = (int64_t)std::max(1, cu_count) * kDecodeStreamWavesPerCu;
    int64_t tiles = 0;
    for (int i = 0; i < g.count; ++i) tiles += g.m[i].T;
    g.block0[0] = 0;
    for (int i = 0; i < g.count; ++i) {
        const int64_t share = std::max<int64_t>(kDecodeWaves, waves * g.m[i].T / tiles / kDecodeWaves * kDecodeWaves);
        g.nw[i] = std::min<int64_t>(g.m[i].T, share);
        g.block0[i + 1] = g.block0[i] + (int32_t)((g.nw[i] + kDecodeWaves - 1) / kDecodeWaves);
    }
    hipLaunchKernelGGL((decode_stream_kernel<false, DecodeGroup>), dim3((uint32_t)g.block0[g.count]), dim3(kDecodeWaves * kWave),
                       0, stream, g);
    return hipGetLastError();
}

hipError_t launch_decode_direct(const DecodeArgs& a, hipStream_t stream, int cu_count) {
    return launch_decode_one<true>(a, stream, cu_count);
}

// One block: the fallback tiles of the bitmap and the codebook, into memory that
// the host reads (system-scope stores). Ahead of a direct decode, so that the
// host has its answer while that still runs.
constexpr int kCheckThreads = 1024;

__global__ __launch_bounds__(kCheckThreads) void check_streams_kernel(const uint8_t* bitmap, int64_t T, const uint8_t* codebook,
                                                                       BindResult* out) {
    __shared__ unsigned long long sum[kCheckThreads / kWave];
    const int tid = threadIdx.x;
    const int64_t bytes = T >> 3;
    unsigned long long n = 0;
    for (int64_t b = 8 * (int64_t)tid; b < bytes; b += 8 * kCheckThreads) {
        if (b + 8 <= bytes) {
            uint64_t v;
            __builtin_memcpy(&v, bitmap + b, sizeof v);
            n += __popcll(v);
        } else {
            for (int64_t i = b; i < bytes; ++i) n += __popc((uint32_t)bitmap[i]);
        }
    }
    if (tid == 0 && (T & 7)) n += __popc((uint32_t)bitmap[bytes] >> (8 - (T & 7)));
    for (int o = 32; o > 0; o /= 2) n += __shfl_xor(n, o, 64);
    if ((tid & 63) == 0) sum[tid >> 6] = n;
    __syncthreads();
    if (tid < 16) {
        const uint8_t c = tid < kCodebook ? codebook[tid] : 0;
        __hip_atomic_store(&out->codebook[tid], c, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
    }
    if (tid == 0) {
        n = 0;
        for (int k = 0; k < kCheckThreads / kWave; ++k) n += sum[k];
        __hip_atomic_store(&out->fallback_tiles, n, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
    }
}

hipError_t launch_check_streams(const uint8_t* bitmap, int64_t T, const uint8_t* codebook, BindResult* out, hipStream_t stream) {
    hipLaunchKernelGGL(check_streams_kernel, dim3(1), dim3(kCheckThreads), 0, stream, bitmap, T, codebook, out);
    return hipGetLastError();
}

hipError_t launch_decode_rows(const DecodeArgs& args, float scale, hipStream_t stream) {
    DecodeArgs a = args;
    a.items = a.nrows * ((a.TC + kRowTiles - 1) / kRowTiles);
    if (a.items <= 0) return hipSuccess;
    const dim3 grid((uint32_t)((a.items + kDecodeWaves - 1) / kDecodeWaves)), block(kDecodeWaves * kWave);
    if (scale != 0.0f)
        hipLaunchKernelGGL(decode_rows_kernel<true>, grid, block, 0, stream, a, scale);
    else
        hipLaunchKernelGGL(decode_rows_kernel<false>, grid, block, 0, stream, a, scale);
    return hipGetLastError();
}

// ---------------------------------------------------------------------------
// bind: the per-tile side records, the pair table and the tile counts
// ---------------------------------------------------------------------------

// One wave per tile. Escapes are ranked in row-major order (chunk, then lane,
// then weight within the lane), the order in which they take the tile's esc
// slots; the first kListedEscapes positions go into the tile's record. A
// fallback tile's word holds its rank in the bitmap (counted by its wave),
// a tile with more escapes than listed the next free place
// of the raw buffer bind decodes those into (in no fixed order: the place is
// only looked up). One kernel for what were a one-block scan of the bitmap, the
// escape positions, a one-block scan of the counts and the record writes:
// 9216x2304 18 us in four launches -> 5.5.
constexpr int kBindThreads = 512;

__global__ __launch_bounds__(kBindThreads) void bind_tiles_kernel(const uint8_t* bitmap, const uint8_t* ec,
                                                                   const uint8_t* esc, const uint8_t* codebook, int64_t T,
                                                                   int64_t run_bytes, uint32_t* side, uint32_t* lut,
                                                                   BindResult* result) {
    constexpr int kWaves = kBindThreads / kWave;
    __shared__ uint32_t pos[kWaves][kListedEscapes / 2];
    __shared__ uint32_t over[kWaves], fall[kWaves], base;
    const int tid = threadIdx.x;
    const uint32_t lane = tid & 63u;
    const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
    if (blockIdx.x == 0) {
        if (tid < 256) lut[tid] = pair_lut_entry(codebook, (uint32_t)tid);
        if (tid < kCodebook) result->codebook[tid] = codebook[tid];
    }
    RankCursor ranked;
    const int64_t byte0 = (int64_t)blockIdx.x * run_bytes;
    for (int64_t byte = byte0; byte < byte0 + run_bytes && byte * kWaves < T; ++byte) {
        if (byte > byte0) __syncthreads();   // the last turn's counts are read
        const int64_t tile = byte * kWaves + w;
        const bool here = tile < T;
        const int64_t t = here ? tile : T - 1;   // a wave past the last tile works on it, and stores nothing
        const uint8_t* ect = ec + t * (kTile / 2) + 8u * lane;
        uint2 e[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) e[j] = *reinterpret_cast<const uint2*>(ect + 512 * j);
        const uint32_t slots = reinterpret_cast<const uint32_t*>(esc + t * kEscBudget)[(lane - 1u) & 3u];
        const bool fallback = here && ((bitmap[t >> 3] >> (7 - (t & 7))) & 1u) != 0u;
        if (lane < kListedEscapes / 2) pos[w][lane] = 0u;
        __builtin_amdgcn_wave_barrier();
        uint16_t* listed = reinterpret_cast<uint16_t*>(pos[w]);
        uint32_t mask = 0, run = 0;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            uint32_t t0 = escape_nibbles(e[j].x), t1 = escape_nibbles(e[j].y);
            const uint32_t cnt = __popc(t0) + __popc(t1);
            const uint32_t incl = wave_incl_scan(cnt);
            const uint32_t total = __builtin_amdgcn_readlane(incl, kWave - 1);
            if (total) mask |= 1u << j;
            uint32_t r = run + incl - cnt;
            const uint32_t first = (4u * j + (lane >> 4)) * kTileCols + 16u * (lane & 15u);
            while (t0 | t1) {
                uint32_t p;
                if (t0) {
                    p = (uint32_t)__builtin_ctz(t0) >> 2;
                    t0 &= t0 - 1u;
                } else {
                    p = 8u + ((uint32_t)__builtin_ctz(t1) >> 2);
                    t1 &= t1 - 1u;
                }
                if (r < kListedEscapes) listed[r] = (uint16_t)(first + p);
                ++r;
            }
            run += total;
        }
        const bool too_many = here && !fallback && run > kListedEscapes;
        if (lane == 0) {
            over[w] = too_many ? 1u : 0u;
            fall[w] = fallback ? 1u : 0u;
        }
        __syncthreads();
        if (tid == 0) {
            uint32_t n_over = 0, n_fall = 0;
#pragma unroll
            for (int k = 0; k < kWaves; ++k) {
                n_over += over[k];
                n_fall += fall[k];
            }
            base = n_over ? (uint32_t)__hip_atomic_fetch_add(&result->overflow_tiles, (unsigned long long)n_over,
                                                             __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)
                          : 0u;
            if (n_fall)
                __hip_atomic_fetch_add(&result->fallback_tiles, (unsigned long long)n_fall, __ATOMIC_RELAXED,
                                       __HIP_MEMORY_SCOPE_AGENT);
        }
        __syncthreads();
        uint32_t info = mask | ((run < kInfoCountMax ? run : kInfoCountMax) << kInfoCountShift);
        if (fallback) {
            info = kInfoFallback | (uint32_t)fallback_rank(bitmap, t, lane, ranked);
        } else if (too_many) {
            uint32_t rank = base;
            for (int k = 0; k < w; ++k) rank += over[k];
            info = kInfoFallback | kInfoOverflow | rank;
        }
        if (here && lane < kSideWords)
            side[tile * kSideWords + lane] = lane == 0   ? info
                                             : lane <= 4 ? slots
                                             : lane <= 8 ? pos[w][lane - 5]
                                                         : 0u;
    }
}

// Decodes every tile with more than the listed escapes into raw[rank]
// (tile-local order, the layout of the format's fallback tiles), ranking its
// escapes per chunk (lanes, then weights within a lane): one wave per tile.
constexpr int kInfoWaves = 4;

__global__ __launch_bounds__(kInfoWaves * kWave) void overflow_decode_kernel(DecodeArgs a, int16_t* raw) {
    SE12_DECLARE_LUT(lut);
    const uint32_t lane = threadIdx.x & 63u;
    store_block_lut(lut, reinterpret_cast<const uint4*>(a.lut)[lane], lane);
    lds_barrier();
    const int64_t tile = (int64_t)blockIdx.x * kInfoWaves + (threadIdx.x >> 6);
    if (tile >= a.T) return;
    const uint32_t info = a.side[tile * kSideWords];
    if (!info_is_overflow(info)) return;
    TileLoads t;
    load_tile(t, a.sm, a.ec, tile, lane);
    const uint4 esc = *reinterpret_cast<const uint4*>(a.esc + tile * kEscBudget);
    uint32_t pat[4][8];
    lookup_tile(lut, t, pat);
    resolve_tile_escapes(pat, t, 0xFu, esc);
    int16_t* out = raw + (int64_t)info_rank(info) * kTile;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        uint32_t w[8];
        merge_chunk(pat[j], t.sm[j], w);
        uint4* p = reinterpret_cast<uint4*>(out + 1024 * j + 16 * lane);
        p[0] = make_uint4(w[0], w[1], w[2], w[3]);
        p[1] = make_uint4(w[4], w[5], w[6], w[7]);
    }
}

hipError_t launch_overflow_decode(const DecodeArgs& a, int16_t* raw, hipStream_t stream) {
    const int64_t blocks = (a.T + kInfoWaves - 1) / kInfoWaves;
    hipLaunchKernelGGL(overflow_decode_kernel, dim3((uint32_t)blocks), dim3(kInfoWaves * kWave), 0, stream, a, raw);
    return hipGetLastError();
}

hipError_t launch_bind_tiles(const uint8_t* bitmap, const uint8_t* ec, const uint8_t* esc, const uint8_t* codebook, int64_t T,
                             uint32_t* side, uint32_t* lut, BindResult* result, hipStream_t stream) {
    static_assert(kBindThreads / kWave == 8, "a byte of the bitmap per block and turn");
    const int64_t bytes = (T + 7) / 8, run = rank_run(bytes);
    hipLaunchKernelGGL(bind_tiles_kernel, dim3((uint32_t)((bytes + run - 1) / run)), dim3(kBindThreads), 0, stream, bitmap, ec,
                       esc, codebook, T, run, side, lut, result);
    return hipGetLastError();
}

}  // namespace se12

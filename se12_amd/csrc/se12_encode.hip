// SE12 encoder on the GPU, byte-identical to the reference encoder
// lws/domain/se12/codec.py:111-141 (which runs numpy on the host at pack time,
// lws/application/codec/pack_model.py:113-120). Kernels:
//   histogram  - 256-bin exponent histogram over the real weights, one partial
//                histogram per block
//   select     - the histogram, and from it the codebook (codebook.py:41-59)
//                and the code of every exponent value, on the device, so that
//                the next kernel follows without a round trip to the host
//   tiles      - sm / ec / esc of every tile, one wave per tile with the same
//                lane mapping as the decoder: escapes (weights whose exponent
//                is not in the codebook; padding never escapes, codec.py:
//                119-125) take slots in tile-local row-major order (codec.py:
//                131,332-343); the fallback bitmap (more than 16 escapes,
//                MSB first, codec.py:132-133,351-353) and its count. Fallback
//                tiles have zero esc slots.
//   raw        - the fallback tiles' padded bits (codec.py:363-365), ranked by
//                the bitmap: launched only where there are any.
//
// Bound by the weights' bytes: read once for the histogram, once (from the
// last-level cache where they fit) for the streams.
// 9216x2304 as the packer's call issues it 253 -> 58 us (histogram 78 -> 10.2:
// it read 2 bytes per load, divided 64-bit indexes and queued on shared LDS
// counters; select 6.5; tiles 17.2 + 2 x 11 of counting + 9.4 of scanning ->
// 18.5; the result's way to the host 4.0; the rest is the call's one
// synchronisation, was 4, and its allocations, most of them made while the
// first two kernels run); 256000x2304 2,024 -> 621 us, 5.2 TB/s of weights read
// twice and streams.
#include <algorithm>

#include "se12_device.hpp"
#include "se12_internal.hpp"

namespace se12 {

constexpr int kTilesThreads = 512;                     // 8 waves: one bitmap byte per block
constexpr int kHistThreads = 1024;
constexpr int kHistCopies = 32;                        // per bin, by lane: no LDS bank conflicts
constexpr int kBins = 256;

// Adds the exponents of two BF16 weights: the bin's row of copies is at byte
// (exponent << 7), which is where the exponent sits in the low half.
__device__ __forceinline__ void count_pair(uint32_t v, char* mine) {
    __hip_atomic_fetch_add(reinterpret_cast<uint32_t*>(mine + (v & 0x7F80u)), 1u, __ATOMIC_RELAXED,
                           __HIP_MEMORY_SCOPE_WORKGROUP);
    __hip_atomic_fetch_add(reinterpret_cast<uint32_t*>(mine + ((v >> 16) & 0x7F80u)), 1u, __ATOMIC_RELAXED,
                           __HIP_MEMORY_SCOPE_WORKGROUP);
}

// Each lane counts in its own copy of the bins (lane % 32, the copies of a bin
// side by side): weights share a handful of exponents, so lanes adding to one
// counter would queue. 16 bytes per load; a matrix whose rows follow each
// other without gaps is read as one row, other rows by a group of lanes each
// (by a block each, narrow rows left most of its lanes idle: 1,000,000 x 256 in
// rows of 264 2,211 us for the histogram and the count of escapes, 227 now).
__global__ __launch_bounds__(kHistThreads) void encode_histogram_kernel(EncodeArgs a) {
    static_assert(kHistCopies * sizeof(uint32_t) == 128, "a bin's copies span 1 << 7 bytes");
    __shared__ __attribute__((aligned(16))) uint32_t hist[kBins * kHistCopies];
    const int tid = threadIdx.x;
    for (int i = tid; i < kBins * kHistCopies / 4; i += kHistThreads)
        reinterpret_cast<uint4*>(hist)[i] = make_uint4(0u, 0u, 0u, 0u);
    __syncthreads();
    char* mine = reinterpret_cast<char*>(hist) + 4 * (tid & (kHistCopies - 1));
    const bool flat = a.ld == a.K;
    const int64_t rows = flat ? 1 : a.N, cols = flat ? a.N * a.K : a.K;
    // a group of lanes per row: a wave, or fewer where a row has fewer loads
    // (8 lanes at least, which take a row's last columns); fewer rows than
    // groups are cut into segments, one per group
    int tpr = 8;
    while (tpr < kWave && 8 * tpr < cols) tpr *= 2;
    const int64_t groups = (int64_t)gridDim.x * kHistThreads / tpr;
    const int64_t item0 = ((int64_t)blockIdx.x * kHistThreads + tid) / tpr;
    const int64_t segs = rows < groups ? std::min<int64_t>(groups / rows, (cols + 8 * tpr - 1) / (8 * tpr)) : 1;
    const int64_t lanes = segs * tpr;
    for (int64_t item = item0; item < rows * segs; item += groups) {
        const int64_t r = segs > 1 ? (int64_t)((uint32_t)item / (uint32_t)segs) : item;   // (fewer than `groups` items then)
        const int64_t block = segs > 1 ? item - r * segs : 0;
        const int lane = tid & (tpr - 1);
        const uint16_t* p = a.w + r * a.ld;
        const int64_t whole = cols / 8;
        int64_t c = block * tpr + lane;
        // four loads in flight
        for (; c + 3 * lanes < whole; c += 4 * lanes) {
            uint4 v[4];
#pragma unroll
            for (int k = 0; k < 4; ++k) v[k] = load16_unaligned(p + 8 * (c + k * lanes));
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                count_pair(v[k].x, mine);
                count_pair(v[k].y, mine);
                count_pair(v[k].z, mine);
                count_pair(v[k].w, mine);
            }
        }
        for (; c < whole; c += lanes) {
            const uint4 v = load16_unaligned(p + 8 * c);
            count_pair(v.x, mine);
            count_pair(v.y, mine);
            count_pair(v.z, mine);
            count_pair(v.w, mine);
        }
        if (block == 0 && lane < cols - 8 * whole)
            __hip_atomic_fetch_add(reinterpret_cast<uint32_t*>(mine + (p[8 * whole + lane] & 0x7F80u)), 1u, __ATOMIC_RELAXED,
                                   __HIP_MEMORY_SCOPE_WORKGROUP);
    }
    __syncthreads();
    if (tid < kBins) {
        uint32_t n = 0;
#pragma unroll
        for (int k = 0; k < kHistCopies; ++k) n += hist[tid * kHistCopies + ((tid + k) & (kHistCopies - 1))];
        a.ws->partial[(int64_t)blockIdx.x * kBins + tid] = n;
    }
}

// One block: the partial histograms' sum, each exponent's rank (more weights
// first, the larger exponent on a tie: the order of se12_codebook_from_
// histogram), and from it the codebook and the codes (15 = escape).
__global__ __launch_bounds__(kHistThreads) void encode_select_kernel(EncodeWork* ws, int blocks, uint8_t* codebook_out) {
    __shared__ uint64_t part[kHistThreads];
    __shared__ __attribute__((aligned(16))) uint64_t key[kBins];   // count << 8 | exponent
    constexpr int kGroups = kBins / 4, kRuns = kHistThreads / kGroups, kFlight = 16;
    __shared__ uint64_t sums[kRuns * kBins];
    const int tid = threadIdx.x, e = tid & (kBins - 1), s = tid / kBins;
    constexpr int kSlices = kHistThreads / kBins;
    // one block waits for its loads alone, so 256 blocks' counts are all in
    // flight at once: four bins per load, 16 loads per thread (7.1 -> 6.5 us)
    uint64_t n4[4] = {0, 0, 0, 0};
    for (int b0 = tid / kGroups; b0 < blocks; b0 += kRuns * kFlight) {
        uint4 v[kFlight];
#pragma unroll
        for (int k = 0; k < kFlight; ++k) {
            const int b = b0 + k * kRuns;
            v[k] = reinterpret_cast<const uint4*>(ws->partial + (int64_t)(b < blocks ? b : b0) * kBins)[tid & (kGroups - 1)];
        }
#pragma unroll
        for (int k = 0; k < kFlight; ++k) {
            if (b0 + k * kRuns >= blocks) continue;
            n4[0] += v[k].x;
            n4[1] += v[k].y;
            n4[2] += v[k].z;
            n4[3] += v[k].w;
        }
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) sums[4 * tid + i] = n4[i];
    __syncthreads();
    if (tid < kBins) {
        uint64_t n = 0;
#pragma unroll
        for (int k = 0; k < kRuns; ++k) n += sums[k * kBins + tid];
        key[tid] = (n << 8) | (uint64_t)tid;
    }
    __syncthreads();
    // four threads per exponent, each against a quarter of the others
    int before = 0;
    const uint64_t mine = key[e];
    const ulonglong2* quarter = reinterpret_cast<const ulonglong2*>(key + s * (kBins / kSlices));
#pragma unroll
    for (int k = 0; k < kBins / kSlices / 2; ++k) {
        const ulonglong2 u = quarter[k];
        before += (u.x > mine ? 1 : 0) + (u.y > mine ? 1 : 0);
    }
    part[tid] = (uint64_t)before;
    __syncthreads();
    if (tid < kBins) {
        int rank = 0;
#pragma unroll
        for (int k = 0; k < kSlices; ++k) rank += (int)part[tid + k * kBins];
        ws->code_of[tid] = (uint8_t)(rank < kCodebook ? rank : 15);
        if (rank < kCodebook) {
            ws->codebook[rank] = (uint8_t)tid;
            if (codebook_out) codebook_out[rank] = (uint8_t)tid;
        }
    }
    if (tid == 0) {
        ws->codebook[kCodebook] = 0;
        ws->fallback_tiles = 0;
    }
}

// the codes of a codebook given by the caller
__global__ __launch_bounds__(kBins) void encode_codes_kernel(EncodeWork* ws, uint4 codebook) {
    const uint32_t cb[4] = {codebook.x, codebook.y, codebook.z, codebook.w};
    const int e = threadIdx.x;
    uint32_t c = 15;
    for (int i = kCodebook - 1; i >= 0; --i)
        if (((cb[i >> 2] >> (8 * (i & 3))) & 0xFFu) == (uint32_t)e) c = i;
    ws->code_of[e] = (uint8_t)c;
    if (e == 0) ws->fallback_tiles = 0;
}

// the lane's 16 weights of chunk j (zero outside the matrix = padding)
__device__ __forceinline__ void load_weights16(const EncodeArgs& a, int64_t row, int64_t col, uint32_t v[8]) {
    const uint16_t* p = a.w + row * a.ld + col;
    if (row < a.N && col + 16 <= a.K) {
        const uint4 u0 = load16_unaligned(p), u1 = load16_unaligned(p + 8);
        v[0] = u0.x; v[1] = u0.y; v[2] = u0.z; v[3] = u0.w;
        v[4] = u1.x; v[5] = u1.y; v[6] = u1.z; v[7] = u1.w;
    } else {
#pragma unroll
        for (int q = 0; q < 8; ++q) {
            uint32_t lo = (row < a.N && col + 2 * q < a.K) ? (uint32_t)p[2 * q] : 0u;
            uint32_t hi = (row < a.N && col + 2 * q + 1 < a.K) ? (uint32_t)p[2 * q + 1] : 0u;
            v[q] = lo | (hi << 16);
        }
    }
}

// codes of the chunk (padding -> 0) and the escape mask (bit i = weight i)
__device__ __forceinline__ void chunk_codes(const EncodeArgs& a, const uint8_t* code_of, int64_t row, int64_t col,
                                            const uint32_t v[8], uint32_t codes[16], uint32_t& escmask) {
    escmask = 0;
    if (row < a.N && col + 16 <= a.K) {
#pragma unroll
        for (int i = 0; i < 16; ++i) codes[i] = (uint32_t)code_of[((v[i >> 1] >> (16 * (i & 1))) >> 7) & 0xFFu];
    } else {
#pragma unroll
        for (int i = 0; i < 16; ++i) {
            const bool valid = row < a.N && col + i < a.K;
            codes[i] = valid ? (uint32_t)code_of[((v[i >> 1] >> (16 * (i & 1))) >> 7) & 0xFFu] : 0u;
        }
    }
#pragma unroll
    for (int i = 0; i < 16; ++i)
        if (codes[i] == 15u) escmask |= 1u << i;
}

// WRITE = false: the count of fallback tiles only
template <bool WRITE>
__global__ __launch_bounds__(kTilesThreads) __attribute__((amdgpu_waves_per_eu(4))) void encode_tiles_kernel(EncodeArgs a) {
    constexpr int kWaves = kTilesThreads / kWave;
    __shared__ __attribute__((aligned(4))) uint8_t code_of[kBins];
    __shared__ uint8_t esc_buf[kWaves][kEscBudget];
    __shared__ uint32_t fallback[kWaves];
    const int tid = threadIdx.x;
    const uint32_t lane = tid & 63;
    const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int64_t tile = (int64_t)blockIdx.x * kWaves + w;
    const bool here = tile < a.T;
    const int64_t t = here ? tile : a.T - 1;   // a wave past the last tile works on it, and stores nothing
    const int tr = (int)(t / a.TC);
    const int kt = (int)(t - (int64_t)tr * a.TC);
    const int64_t col = (int64_t)kt * kTileCols + 16 * (lane & 15u);
    uint32_t v[4][8];
#pragma unroll
    for (int j = 0; j < 4; ++j) load_weights16(a, (int64_t)tr * kTileRows + 4 * j + (lane >> 4), col, v[j]);
    if (tid < kBins / 4)
        reinterpret_cast<uint32_t*>(code_of)[tid] = reinterpret_cast<const uint32_t*>(a.ws->code_of)[tid];
    lds_barrier();

    uint32_t escm[4];
    uint32_t cnt[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        const int64_t row = (int64_t)tr * kTileRows + 4 * j + (lane >> 4);
        uint32_t codes[16];
        chunk_codes(a, code_of, row, col, v[j], codes, escm[j]);
        cnt[j] = __popc(escm[j]);
        if constexpr (WRITE) {
            // sm bytes: ((b >> 8) & 0x80) | (b & 0x7F) for each weight
            uint32_t smw[4];
#pragma unroll
            for (int d = 0; d < 4; ++d) {
                uint32_t word = 0;
#pragma unroll
                for (int k = 0; k < 2; ++k) {
                    const uint32_t u = v[j][2 * d + k];
                    const uint32_t both = ((u >> 8) & 0x00800080u) | (u & 0x007F007Fu);
                    word |= ((both & 0xFFu) | (both >> 8)) << (16 * k);
                }
                smw[d] = word;
            }
            uint32_t ecw[2] = {0u, 0u};
#pragma unroll
            for (int q = 0; q < 8; ++q) ecw[q >> 2] |= (codes[2 * q] | (codes[2 * q + 1] << 4)) << (8 * (q & 3));
            if (here) {
                *reinterpret_cast<uint4*>(a.sm + tile * kTile + 1024 * j + 16 * lane) =
                    make_uint4(smw[0], smw[1], smw[2], smw[3]);
                *reinterpret_cast<uint2*>(a.ec + tile * (kTile / 2) + 512 * j + 8 * lane) = make_uint2(ecw[0], ecw[1]);
            }
        }
    }

    // escape ranks: chunk j, then lane, then position (tile-local row-major)
    const uint32_t s01 = wave_incl_scan(cnt[0] | (cnt[1] << 16));
    const uint32_t s23 = wave_incl_scan(cnt[2] | (cnt[3] << 16));
    const uint32_t t01 = __builtin_amdgcn_readlane(s01, kWave - 1);
    const uint32_t t23 = __builtin_amdgcn_readlane(s23, kWave - 1);
    const uint32_t tot[4] = {t01 & 0xFFFFu, t01 >> 16, t23 & 0xFFFFu, t23 >> 16};
    const uint32_t incl[4] = {s01 & 0xFFFFu, s01 >> 16, s23 & 0xFFFFu, s23 >> 16};
    const uint32_t total = tot[0] + tot[1] + tot[2] + tot[3];
    const bool over = here && total > (uint32_t)kEscBudget;
    if constexpr (WRITE) {
        if (total <= (uint32_t)kEscBudget) {
            uint32_t run = 0;
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                uint32_t r = run + incl[j] - cnt[j];
                uint32_t m = escm[j];
                while (m) {
                    const int i = __builtin_ctz(m);
                    m &= m - 1u;
                    const uint32_t bits = (v[j][i >> 1] >> (16 * (i & 1))) & 0xFFFFu;
                    esc_buf[w][r] = (uint8_t)((bits >> 7) & 0xFFu);
                    ++r;
                }
                run += tot[j];
            }
            __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
            __builtin_amdgcn_wave_barrier();
            __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
        }
        if (here && lane < (uint32_t)kEscBudget)
            a.esc[tile * kEscBudget + lane] = lane < total && !over ? esc_buf[w][lane] : (uint8_t)0;
    }
    if (lane == 0) fallback[w] = over ? 1u : 0u;
    lds_barrier();
    if (tid == 0) {
        uint32_t byte = 0;
#pragma unroll
        for (int k = 0; k < kWaves; ++k) byte |= fallback[k] << (7 - k);
        if constexpr (WRITE) a.bitmap[blockIdx.x] = (uint8_t)byte;
        if (byte)
            __hip_atomic_fetch_add(&a.ws->fallback_tiles, (unsigned long long)__popc(byte), __ATOMIC_RELAXED,
                                   __HIP_MEMORY_SCOPE_AGENT);
    }
}

// One wave per tile and turn: a fallback tile's rank is the number of set
// bitmap bits before it, counted by the wave.
__global__ __launch_bounds__(kTilesThreads) void encode_raw_kernel(EncodeArgs a, int64_t run_bytes) {
    const uint32_t lane = threadIdx.x & 63;
    const int w = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    RankCursor ranked;
    const int64_t byte0 = (int64_t)blockIdx.x * run_bytes;
    for (int64_t byte = byte0; byte < byte0 + run_bytes; ++byte) {
        const int64_t tile = byte * 8 + w;
        if (tile >= a.T) return;
        if (!((a.bitmap[byte] >> (7 - w)) & 1u)) continue;
        const int64_t rank = fallback_rank(a.bitmap, tile, lane, ranked);
        if (rank >= a.raw_tiles) return;
        const int tr = (int)(tile / a.TC);
        const int kt = (int)(tile - (int64_t)tr * a.TC);
        const int64_t col = (int64_t)kt * kTileCols + 16 * (lane & 15u);
        int16_t* raw = a.raw + rank * kTile;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            uint32_t v[8];
            load_weights16(a, (int64_t)tr * kTileRows + 4 * j + (lane >> 4), col, v);
            uint4* p = reinterpret_cast<uint4*>(raw + 1024 * j + 16 * lane);
            p[0] = make_uint4(v[0], v[1], v[2], v[3]);
            p[1] = make_uint4(v[4], v[5], v[6], v[7]);
        }
    }
}

int encode_histogram_blocks(const EncodeArgs& a, int cu_count) {
    // one block per CU (its waves fill it), fewer where the weights are few
    const int64_t blocks = (a.N * a.K + 8 * kHistThreads - 1) / (8 * kHistThreads);
    return (int)std::max<int64_t>(1, std::min<int64_t>({blocks, (int64_t)cu_count, (int64_t)kEncodeHistBlocks}));
}

hipError_t launch_encode_histogram(const EncodeArgs& a, int cu_count, uint8_t* codebook_out, hipStream_t stream) {
    const int blocks = encode_histogram_blocks(a, cu_count);
    hipLaunchKernelGGL(encode_histogram_kernel, dim3((uint32_t)blocks), dim3(kHistThreads), 0, stream, a);
    hipLaunchKernelGGL(encode_select_kernel, dim3(1), dim3(kHistThreads), 0, stream, a.ws, blocks, codebook_out);
    return hipGetLastError();
}

hipError_t launch_encode_codes(const EncodeArgs& a, const uint8_t codebook[16], hipStream_t stream) {
    uint4 cb;
    __builtin_memcpy(&cb, codebook, sizeof cb);
    hipLaunchKernelGGL(encode_codes_kernel, dim3(1), dim3(kBins), 0, stream, a.ws, cb);
    return hipGetLastError();
}

hipError_t launch_encode_tiles(const EncodeArgs& a, bool write, hipStream_t stream) {
    const dim3 grid((uint32_t)((a.T + kTilesThreads / kWave - 1) / (kTilesThreads / kWave))), block(kTilesThreads);
    if (write)
        hipLaunchKernelGGL(encode_tiles_kernel<true>, grid, block, 0, stream, a);
    else
        hipLaunchKernelGGL(encode_tiles_kernel<false>, grid, block, 0, stream, a);
    return hipGetLastError();
}

// What the host reads of a call, into memory that it can: a copy of the
// runtime's takes 4.2 us on the device and as long again to issue.
// The count starts again at zero, for another pass over the tiles.
__global__ void encode_result_kernel(EncodeWork* ws, EncodeResult* host) {
    const int tid = threadIdx.x;
    if (tid < 16) __hip_atomic_store(&host->codebook[tid], ws->codebook[tid], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
    if (tid == 16) {
        __hip_atomic_store(&host->fallback_tiles, ws->fallback_tiles, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
        ws->fallback_tiles = 0;
    }
}

hipError_t launch_encode_result(const EncodeArgs& a, EncodeResult* host, hipStream_t stream) {
    hipLaunchKernelGGL(encode_result_kernel, dim3(1), dim3(kWave), 0, stream, a.ws, host);
    return hipGetLastError();
}

hipError_t launch_encode_raw(const EncodeArgs& a, hipStream_t stream) {
    static_assert(kTilesThreads / kWave == 8, "a byte of the bitmap per block and turn");
    const int64_t bytes = (a.T + 7) / 8, run = rank_run(bytes);
    hipLaunchKernelGGL(encode_raw_kernel, dim3((uint32_t)((bytes + run - 1) / run)), dim3(kTilesThreads), 0, stream, a, run);
    return hipGetLastError();
}

}  // namespace se12

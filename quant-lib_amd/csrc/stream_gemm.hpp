// stream_gemm.hpp -- GEMM of few token rows as a stream of the weight matrix:
// C[M,N] = A[M,K] W[N,K]^T, weights binary16 or FP8 codes (a Weights policy),
// fp32 accumulation, binary16 result.  Included by gemm_stream.hip and fp8.hip.
#pragma once

#include "ql_common.hpp"

namespace ql {

typedef _Float16 sg_half8 __attribute__((ext_vector_type(8)));
typedef float sg_floatx4 __attribute__((ext_vector_type(4)));

// none (binary16 weights); one per tensor or row (applied to the sums; the row
// stride groups_per_row is 0 or 1); per group of a multiple of 128, or of 64, codes
enum StreamScale { kStreamNone = 0, kStreamRow = 1, kStreamGroup = 2, kStreamHalfGroup = 3 };

struct StreamArgs {
    const char* A;        // [M, K] binary16, 16-byte aligned
    const char* W;        // [N, K] weights, 16-byte aligned
    const float* scales;  // FP8: per tensor, per row, or [N][groups_per_row]
    _Float16* C;          // [M, N]
    int M, N, K;
    int gs, groups_per_row;
    float* part;          // [splits][M][N] fp32 partials (gridDim.y > 1)
    int chunks_per_split; // K-split of blockIdx.y, in kStreamChunk steps
    const char* W2;       // gridDim.z = 2: a second product of the same tokens and shape
    const float* scales2; // (no K-split)
    _Float16* C2;
};

constexpr int kStreamChunk = 128;       // k per step of a wavefront
constexpr int kStreamMaxK = 1 << 23;    // byte offsets inside a workgroup's rows stay below 2^31

// What bounds it: the weight matrix from HBM, and the token rows, which every
// workgroup reads for its whole K range from L2 (measured at about 17-20 TB/s over
// the chip, so at 32 tokens they cost as much as the weights unless a workgroup
// covers several row tiles).  A read-only probe of the same 58.7 MB takes 11-12 us.
//
// Workgroup: 16*R weight rows x 16*MT tokens, NW wavefronts that take every NW-th
// chunk of 128 k of the workgroup's range, so together they read whole rows: a
// chunk of 16 rows is kLoads instructions of complete 128- or 256-byte row segments
// (16 rows x 64 bytes an instruction, the fragment shape, streamed 20-40% slower),
// and the chunk's token rows 4 rows x 256 bytes an instruction (1 to 9 us faster at
// 32 tokens than 16 rows x 64 bytes).  Both are re-laid into MFMA fragments through a
// wavefront-private LDS area, XOR-swizzled by row; one wavefront's LDS operations
// complete in order, so the loop has no barrier.  One chunk of loads is in flight
// while the one before is multiplied (two were 0-30% slower: a wavefront has 2-8
// chunks, and the loads past its last one cost issue slots).  The weights are the
// B operand, so a lane's sums belong to one weight row and take one scale each.
// The wavefronts' partial tiles are summed in LDS in wavefront order.
//
// Measured on MI355X, weights streamed from HBM, us per call against what ran
// before: FP8 E4M3 groups of 128, 24 tokens x 4096 x 14336 24.6 -> 19.9, 32 x 14336 x
// 4096 23.3 -> 19.2 (3.1 TB/s), 16 x 3072 x 2048 10.1 -> 5.1; binary16 (the library
// GEMM) 1 x 4096 x 4096 12.4 -> 8.2, 8 x 4096 x 14336 24.9 -> 21.5 (5.5 TB/s).
template <typename WP, int SK, int MT, int R, int NW>
__global__ __launch_bounds__(NW * kWave) void stream_gemm(StreamArgs p) {
    constexpr int NL = WP::kLoads;                    // 16-byte loads of a 16-row tile per step
    constexpr int kRowB = kStreamChunk * WP::kBytes;  // bytes of a row per step
    constexpr int kCols = kRowB / 16;                 // 16-byte slots of a row
    const int lane = threadIdx.x & (kWave - 1), wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
    const int j = lane & 15, q = lane >> 4;
    const int n0 = blockIdx.x * 16 * R;
    if (blockIdx.z) {
        p.W = p.W2;
        p.scales = p.scales2;
        p.C = p.C2;
    }
    const int rows = min(16 * R, p.N - n0);
    const uint32_t row_b = (uint32_t)p.K * WP::kBytes;
    // buffers that end at the workgroup's last weight row and the last token row:
    // loads past either end return zeros without touching memory
    const uint32_t w_end = (uint32_t)rows * row_b, a_end = 2u * (uint32_t)p.M * (uint32_t)p.K;
    const __amdgpu_buffer_rsrc_t rw = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<char*>(p.W + (size_t)n0 * row_b), (short)0, (int)w_end, 0x00020000);
    const __amdgpu_buffer_rsrc_t ra =
        __builtin_amdgcn_make_buffer_rsrc(const_cast<char*>(p.A), (short)0, (int)a_end, 0x00020000);
    // weights: instruction l covers kWave / kCols whole rows of the tile; tokens: 4 rows
    uint32_t woff[NL], aoff[4];
#pragma unroll
    for (int l = 0; l < NL; ++l) woff[l] = (uint32_t)((kWave / kCols) * l + lane / kCols) * row_b + 16u * (lane % kCols);
#pragma unroll
    for (int l = 0; l < 4; ++l) aoff[l] = 2u * (uint32_t)(4 * l + q) * (uint32_t)p.K + 16u * j;
    const uint32_t a_tile = 32u * (uint32_t)p.K;      // bytes of 16 token rows
    uint32_t soff[R];
#pragma unroll
    for (int r = 0; r < R; ++r) soff[r] = (uint32_t)min(n0 + 16 * r + j, p.N - 1) * (uint32_t)p.groups_per_row;

    constexpr int kTile = 16 * kCols, kTok = 16 * 16; // 16-byte slots of a weight tile and of a token tile
    constexpr int kWaveSlots = R * kTile > MT * kTok ? R * kTile : MT * kTok;
    constexpr int kTileB = NW * kWaveSlots * 16, kRedB = NW * R * MT * kWave * 16;
    __shared__ __align__(16) char smem[kTileB > kRedB ? kTileB : kRedB];
    u32x4* tile = reinterpret_cast<u32x4*>(smem) + wave * kWaveSlots;
    int wslot[NL], rslot[NL], twslot[4], trslot[4];
#pragma unroll
    for (int l = 0; l < NL; ++l) {
        const int row = (kWave / kCols) * l + lane / kCols;
        wslot[l] = row * kCols + WP::swizzle(row, lane % kCols);
        rslot[l] = j * kCols + WP::swizzle(j, 4 * l + q);
    }
#pragma unroll
    for (int l = 0; l < 4; ++l) {
        twslot[l] = (4 * l + q) * 16 + (j ^ (4 * l + q));
        trslot[l] = j * 16 + (WP::tok_slot(l, q) ^ j);
    }

    const int c0 = blockIdx.y * p.chunks_per_split;
    const int c1 = min(p.K / kStreamChunk, c0 + p.chunks_per_split);
    const int first = c0 + wave;
    u32x4 w[R][NL], a[MT][4];
    float s[R][2];
    // chunk c; past the split's end the loads return zeros (never used)
    auto load = [&](int c) __attribute__((always_inline)) {
        const uint32_t kw = c < c1 ? (uint32_t)c * kRowB : w_end;
        const uint32_t ka = c < c1 ? (uint32_t)c * (2u * kStreamChunk) : a_end;
#pragma unroll
        for (int r = 0; r < R; ++r)
#pragma unroll
            for (int l = 0; l < NL; ++l)
                w[r][l] = __builtin_amdgcn_raw_buffer_load_b128(rw, woff[l] + (uint32_t)(16 * r) * row_b + kw, 0, 2);
#pragma unroll
        for (int t = 0; t < MT; ++t)
#pragma unroll
            for (int l = 0; l < 4; ++l)
                a[t][l] = __builtin_amdgcn_raw_buffer_load_b128(ra, aoff[l] + (uint32_t)t * a_tile + ka, 0, 0);
        if constexpr (SK >= kStreamGroup) {
            const int k = min(c, c1 - 1) * kStreamChunk;
#pragma unroll
            for (int r = 0; r < R; ++r) {
                s[r][0] = p.scales[soff[r] + (uint32_t)(k / p.gs)];
                if constexpr (SK == kStreamHalfGroup) s[r][1] = p.scales[soff[r] + (uint32_t)((k + 64) / p.gs)];
            }
        }
    };
    sg_floatx4 acc[R][MT];
#pragma unroll
    for (int r = 0; r < R; ++r)
#pragma unroll
        for (int t = 0; t < MT; ++t) acc[r][t] = sg_floatx4{};
    if (first < c1) load(first);
    for (int c = first; c < c1; c += NW) {
        sg_half8 x[MT][4];
        float inv[R][2];
#pragma unroll
        for (int t = 0; t < MT; ++t)
#pragma unroll
            for (int l = 0; l < 4; ++l) tile[t * kTok + twslot[l]] = a[t][l];
        // orders the compiler only: one wavefront's LDS operations execute in order
        __builtin_amdgcn_wave_barrier();
#pragma unroll
        for (int t = 0; t < MT; ++t)
#pragma unroll
            for (int l = 0; l < 4; ++l) x[t][l] = __builtin_bit_cast(sg_half8, tile[t * kTok + trslot[l]]);
        __builtin_amdgcn_wave_barrier();
#pragma unroll
        for (int r = 0; r < R; ++r)
#pragma unroll
            for (int l = 0; l < NL; ++l) tile[r * kTile + wslot[l]] = w[r][l];
        if constexpr (SK >= kStreamGroup) {
#pragma unroll
            for (int r = 0; r < R; ++r) {
                inv[r][0] = 1.0f / s[r][0];
                if constexpr (SK == kStreamHalfGroup) inv[r][1] = 1.0f / s[r][1];
            }
        }
        load(c + NW);
        __builtin_amdgcn_wave_barrier();
#pragma unroll
        for (int r = 0; r < R; ++r) {
            u32x4 v[NL];
#pragma unroll
            for (int l = 0; l < NL; ++l) v[l] = tile[r * kTile + rslot[l]];
            sg_half8 b[4];
            WP::decode(v, b);
#pragma unroll
            for (int t = 0; t < MT; ++t) {
                if constexpr (SK >= kStreamGroup) {
                    // products of decoded codes, one multiply-add per output and group
                    sg_floatx4 g = sg_floatx4{};
#pragma unroll
                    for (int l = 0; l < 4; ++l) {
                        g = __builtin_amdgcn_mfma_f32_16x16x32_f16(x[t][l], b[l], g, 0, 0, 0);
                        if (l == 3 || (SK == kStreamHalfGroup && l == 1)) {
#pragma unroll
                            for (int i = 0; i < 4; ++i)
                                acc[r][t][i] = fmaf(g[i], inv[r][SK == kStreamHalfGroup ? l / 2 : 0], acc[r][t][i]);
                            g = sg_floatx4{};
                        }
                    }
                } else {
#pragma unroll
                    for (int l = 0; l < 4; ++l)
                        acc[r][t] = __builtin_amdgcn_mfma_f32_16x16x32_f16(x[t][l], b[l], acc[r][t], 0, 0, 0);
                }
            }
        }
        __builtin_amdgcn_wave_barrier();
    }
    // lane holds C[token 16t + 4q + i][row 16r + j]; sum the wavefronts in order
    __syncthreads();
    sg_floatx4* red = reinterpret_cast<sg_floatx4*>(smem);
#pragma unroll
    for (int r = 0; r < R; ++r)
#pragma unroll
        for (int t = 0; t < MT; ++t) red[(wave * R * MT + r * MT + t) * kWave + lane] = acc[r][t];
    __syncthreads();
#pragma unroll
    for (int it = 0; it < (R * MT + NW - 1) / NW; ++it) {
        const int u = it * NW + wave;   // wavefront-uniform
        if (u < R * MT) {
            const int r = u / MT, t = u - r * MT;
            sg_floatx4 sum = red[u * kWave + lane];
#pragma unroll
            for (int v = 1; v < NW; ++v) sum += red[(v * R * MT + u) * kWave + lane];
            const int row = n0 + 16 * r + j;
            if constexpr (SK == kStreamRow) {
                const float rs = 1.0f / p.scales[(size_t)min(row, p.N - 1) * p.groups_per_row];
#pragma unroll
                for (int i = 0; i < 4; ++i) sum[i] *= rs;
            }
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const int m = 16 * t + 4 * q + i;
                if (m < p.M && row < p.N) {
                    if (gridDim.y == 1) p.C[(size_t)m * p.N + row] = from_f32<_Float16>(sum[i]);
                    else p.part[((size_t)blockIdx.y * p.M + m) * p.N + row] = sum[i];
                }
            }
        }
    }
}

// binary16 weights: a lane's fragment of step l is its row's k = 32l + 8q .. +7
struct StreamF16 {
    static constexpr int kBytes = 2, kLoads = 4;
    static __device__ __forceinline__ constexpr int tok_slot(int l, int q) { return 4 * l + q; }
    static __device__ __forceinline__ int swizzle(int row, int col) { return col ^ row; }
    static __device__ __forceinline__ void decode(const u32x4 (&v)[4], sg_half8 (&b)[4]) {
#pragma unroll
        for (int l = 0; l < 4; ++l) b[l] = __builtin_bit_cast(sg_half8, v[l]);
    }
};

}  // namespace ql

// fp8_gemm_tile.hip -- FP8-weight GEMM for more than 64 token rows:
// C[M,N] = A[M,K] (dequant W[N,K])^T with the weights decoded between LDS and the
// matrix cores, so that no dequantized copy of W is written and read.
#include "fp8_decode.hpp"
#include "fp8_gemm_tile.hpp"
#include "quantlib_amd.h"

#include <type_traits>

namespace {

using namespace ql;

typedef float floatx4 __attribute__((ext_vector_type(4)));

constexpr int kBM = 128;       // token rows of a workgroup
constexpr int kBK = 64;        // k of a step
constexpr int kThreads = 256;  // 2 x 2 wavefronts of 64 tokens x BN / 2 weight rows

struct TileArgs {
    const char* A;
    const char* W;
    const float* scales;
    _Float16* C;
    float* part;
    int M, N, K, gs, groups_per_row;
    int steps_per_split;
    int m_tiles;
    int wide_store;   // C rows take 16-byte stores
};

// Lane l's 16 (4) bytes at src to dst + 16 (4) l in LDS, dst uniform over the wavefront.
__device__ __forceinline__ void to_lds16(const void* src, u32x4* dst) {
    __builtin_amdgcn_global_load_lds(src, (__attribute__((address_space(3))) void*)dst, 16, 0, 0);
}
__device__ __forceinline__ void to_lds4(const void* src, u32x4* dst) {
    __builtin_amdgcn_global_load_lds(src, (__attribute__((address_space(3))) void*)dst, 4, 0, 0);
}

__device__ __forceinline__ uint32_t lds_offset(const void* p) {
    return (uint32_t)(uintptr_t)(const __attribute__((address_space(3))) void*)p;
}

// s[n] = the float at LDS offset at + 256 n (rows 16 apart)
template <int NT>
__device__ __forceinline__ void lds_read_scales(uint32_t at, float (&s)[NT]) {
    static_assert(NT == 2 || NT == 4, "row tiles");
    if constexpr (NT == 2)
        asm volatile("ds_read_b32 %0, %2\n\tds_read_b32 %1, %2 offset:256\n\ts_waitcnt lgkmcnt(0)"
                     : "=&v"(s[0]), "=&v"(s[1]) : "v"(at) : "memory");
    else
        asm volatile("ds_read_b32 %0, %4\n\tds_read_b32 %1, %4 offset:256\n\tds_read_b32 %2, %4 offset:512\n\t"
                     "ds_read_b32 %3, %4 offset:768\n\ts_waitcnt lgkmcnt(0)"
                     : "=&v"(s[0]), "=&v"(s[1]), "=&v"(s[2]), "=&v"(s[3]) : "v"(at) : "memory");
}

// A workgroup computes 128 tokens x BN weight rows over its K range in steps of 64 k.
// Tokens (128-byte rows) and codes (64-byte rows) go straight from global memory into
// one of ST LDS stages, ST - 1 steps ahead (16-byte slots XOR-swizzled by row through
// the lanes' source addresses, conflict-free reads); a step waits for its own stage's
// loads only, then one barrier.  Group scales follow four groups at a time.  A lane's 16 codes of
// a row are two MFMA fragments (k = 16q + 8e .. +7 of the step), the token fragments
// follow the same order.  Codes are decoded exactly; GROUPS: the products of a group are
// summed apart and added once, times the group's inverse scale (v_rcp_f32, 1 ulp).
// Reference mode: each wavefront checks its half of the codes it multiplies for an
// exponent of 0 with a mantissa; those, and the NaN sums that |code| 0x7F gives, are
// the codes whose reference decode differs (the encoder writes them only for NaN
// inputs): a workgroup that met one computes its tile again with the checking decoder.
// Rows past M or N repeat the last row: their products are never stored.
template <int FMT, int MODE, bool GROUPS, int BN, int ST>
__global__ __launch_bounds__(kThreads, 2) void fp8_gemm_tile(TileArgs p) {
    constexpr int WN = BN / 2, NT = WN / 16;          // a wavefront's weight rows, in tiles
    constexpr int MT = 4;                              // its token tiles
    constexpr int AL = kBM / 32, WL = BN / 64;         // its 1 KiB loads of a step
    constexpr int kLoads = AL + WL;
    constexpr int kTokU4 = kBM * 8, kWtU4 = BN * 4;
    constexpr int kStageU4 = kTokU4 + kWtU4;
    static_assert(ST >= 2 && ST <= 4, "stages");
    __shared__ u32x4 s0[kStageU4];
    __shared__ u32x4 s1[kStageU4];
    __shared__ u32x4 s2[ST > 2 ? kStageU4 : 1];
    __shared__ u32x4 s3[ST > 3 ? kStageU4 : 1];
    __shared__ u32x4 scale_quads[GROUPS ? 2 * BN : 1];   // scales of 4 groups: [group / 4 % 2][row][group % 4]
    int* any_special = reinterpret_cast<int*>(s1);         // after the loop

    const int tid = threadIdx.x, lane = tid & (kWave - 1), wave = __builtin_amdgcn_readfirstlane(tid / kWave);
    const int j = lane & 15, q = lane >> 4;
    const int wm = wave & 1, wn = wave >> 1;
    // consecutive ids go to the 8 XCDs in turn: each XCD takes a contiguous run of tiles,
    // the token tiles of one weight tile side by side, so its weights are read once a XCD
    int m0, n0;
    {
        const int total = gridDim.x, x = blockIdx.x & 7, per = total >> 3, rem = total & 7;
        const int t = x * per + min(x, rem) + (int)(blockIdx.x >> 3);
        m0 = (t % p.m_tiles) * kBM;
        n0 = (t / p.m_tiles) * BN;
    }
    const int t0 = blockIdx.y * p.steps_per_split;
    const int n_steps = min(p.K / kBK - t0, p.steps_per_split);
    auto swz_a = [](int r) { return (r ^ ((r >> 3) & 1)) & 7; };
    auto swz_w = [](int r) { return (r >> 2) & 3; };
    // load l of a wavefront: token rows 8 (4 l + wave) + lane / 8, weight rows
    // 16 (4 l + wave) + lane / 4 of the workgroup's
    uint32_t aoff[AL], woff[WL];
#pragma unroll
    for (int l = 0; l < AL; ++l) {
        const int r = 8 * (4 * l + wave) + lane / 8;
        aoff[l] = 2u * (uint32_t)min(m0 + r, p.M - 1) * (uint32_t)p.K + 16u * ((lane & 7) ^ swz_a(r));
    }
#pragma unroll
    for (int l = 0; l < WL; ++l) {
        const int r = 16 * (4 * l + wave) + lane / 4;
        woff[l] = (uint32_t)min(r, p.N - 1 - n0) * (uint32_t)p.K + 16u * ((lane & 3) ^ swz_w(r));
    }
    const char* wbase = p.W + (size_t)n0 * (size_t)p.K;
    auto load = [&](u32x4* st, int i) __attribute__((always_inline)) {
        const int t = t0 + min(i, n_steps - 1);   // past the last step: repeated, never used
        const char* a = p.A + (size_t)t * (2 * kBK);
        const char* w = wbase + (size_t)t * kBK;
#pragma unroll
        for (int l = 0; l < AL; ++l) to_lds16(a + aoff[l], st + (4 * l + wave) * kWave);
#pragma unroll
        for (int l = 0; l < WL; ++l)
            to_lds16(w + woff[l], st + kTokU4 + (4 * l + wave) * kWave);
    };
    // scales of groups 4 quad .. 4 quad + 3: 16 rows x 16 bytes a load
    auto load_scales = [&](int quad) __attribute__((always_inline)) {
#pragma unroll
        for (int l = 0; l < WL; ++l) {
            const int r = 16 * (4 * l + wave);
            const size_t row = (size_t)min(n0 + r + lane / 4, p.N - 1);
            to_lds4(p.scales + row * (size_t)p.groups_per_row + min(4 * quad + (lane & 3), p.groups_per_row - 1),
                    scale_quads + (quad & 1) * BN + r);
        }
    };
    floatx4 acc[NT][MT], part[GROUPS ? NT : 1][MT];
    uint32_t special = 0;
    const int group_steps = GROUPS ? p.gs / kBK : 1;
    int left = 0, group = 0;   // steps left in the current group
    bool new_quad = false;
    auto fold = [&]() __attribute__((always_inline)) {
        if constexpr (GROUPS) {
            // read in assembly, with its wait: the compiler's wait before an ordinary read
            // of an array that loads go to would cover every load in flight.  The quad's
            // own loads were waited for at least a group ago.
            const uint32_t at = lds_offset(scale_quads) +
                                16u * (uint32_t)(((group >> 2) & 1) * BN + wn * WN + j) + 4u * (uint32_t)(group & 3);
            float sc[NT];
            lds_read_scales<NT>(at, sc);
#pragma unroll
            for (int n = 0; n < NT; ++n) {
                const float inv = __builtin_amdgcn_rcpf(sc[n]);
#pragma unroll
                for (int t = 0; t < MT; ++t) {
#pragma unroll
                    for (int e = 0; e < 4; ++e) acc[n][t][e] = fmaf(part[n][t][e], inv, acc[n][t][e]);
                    part[n][t] = floatx4{};
                }
            }
        }
    };
    auto compute = [&](const u32x4* st, auto checked) __attribute__((always_inline)) {
        const u32x4* wt = st + kTokU4;
        half8 x[MT][2];
#pragma unroll
        for (int t = 0; t < MT; ++t)
#pragma unroll
            for (int e = 0; e < 2; ++e) {
                const int row = wm * 64 + 16 * t + j;
                x[t][e] = __builtin_bit_cast(half8, st[row * 8 + ((2 * q + e) ^ swz_a(row))]);
            }
#pragma unroll
        for (int n = 0; n < NT; ++n) {
            const int row = wn * WN + 16 * n + j;
            const u32x4 v = wt[row * 4 + (q ^ swz_w(row))];
            half8 b[2];
            constexpr int kDec = decltype(checked)::value ? QL_FP8_MODE_REFERENCE : QL_FP8_MODE_OCP;
            dequant16<FMT, kDec, false>(uint4{v[0], v[1], v[2], v[3]}, 1.0f, b[0], b[1]);
            if constexpr (MODE == QL_FP8_MODE_REFERENCE && !decltype(checked)::value) {
                if ((n & 1) == wm) {
                    // bit 7 of a byte: its low 7 bits are 1..7 (no carry or borrow between bytes)
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        const uint32_t l = v[e] & 0x7F7F7F7Fu;
                        special |= (l + 0x7F7F7F7Fu) & (0x87878787u - l);
                    }
                }
            }
            floatx4 (&sum)[MT] = GROUPS ? part[GROUPS ? n : 0] : acc[n];
#pragma unroll
            for (int e = 0; e < 2; ++e)
#pragma unroll
                for (int t = 0; t < MT; ++t)
                    sum[t] = __builtin_amdgcn_mfma_f32_16x16x32_f16(x[t][e], b[e], sum[t], 0, 0, 0);
        }
        if constexpr (GROUPS) {
            if (--left == 0) {   // uniform: the group's last step
                left = group_steps;
                fold();
                new_quad = (++group & 3) == 0;
            }
        }
    };
    auto stage_of = [&](int s) __attribute__((always_inline)) { return s == 0 ? s0 : s == 1 ? s1 : s == 2 ? s2 : s3; };
    auto run = [&](auto checked) __attribute__((always_inline)) {
#pragma unroll
        for (int n = 0; n < NT; ++n)
#pragma unroll
            for (int t = 0; t < MT; ++t) {
                acc[n][t] = floatx4{};
                if constexpr (GROUPS) part[n][t] = floatx4{};
            }
        if constexpr (GROUPS) {
            group = t0 / group_steps;
            left = group_steps - t0 % group_steps;
            new_quad = false;
            load_scales(group / 4);
            load_scales(group / 4 + 1);
        }
#pragma unroll
        for (int s = 0; s < ST - 1; ++s) load(stage_of(s), s);
        auto step = [&](int s, int i) __attribute__((always_inline)) {
            // this wavefront's loads of step i have landed and its LDS reads of step i - 1
            // are done (vmcnt(kLeft), lgkmcnt(0), expcnt at its maximum), then every
            // wavefront's: the stage of step i - 1 is free
            constexpr int kLeft = (ST - 2) * kLoads;
            static_assert(kLeft < 64, "vmcnt");
            __builtin_amdgcn_s_waitcnt(0x0070 | (kLeft & 15) | ((kLeft >> 4) << 14));
            // a bare barrier: a release fence would wait for every load in flight to LDS
            asm volatile("s_barrier" ::: "memory");
            load(stage_of((s + ST - 1) % ST), i + ST - 1);
            if constexpr (GROUPS) {
                // every wavefront has read the quad before: its place takes the one after next
                if (new_quad) load_scales(group / 4 + 1);
                new_quad = false;
            }
            compute(stage_of(s), checked);
        };
        // whole rounds without a branch between the steps (at a join the compiler's own
        // waits before the LDS reads would cover every load in flight), then the rest
        int i0 = 0;
        for (; i0 + ST <= n_steps; i0 += ST) {
#pragma unroll
            for (int s = 0; s < ST; ++s) step(s, i0 + s);
        }
#pragma unroll
        for (int s = 0; s < ST - 1; ++s)
            if (i0 + s < n_steps) step(s, i0 + s);
        if (left != group_steps) fold();   // the split ends inside a group (uniform)
        __builtin_amdgcn_s_waitcnt(0x0F70);   // the repeated loads too: the stages are reused
        __syncthreads();
    };
    run(std::false_type{});
    if constexpr (MODE == QL_FP8_MODE_REFERENCE) {
        if (tid == 0) *any_special = 0;
        __syncthreads();
        bool nan = false;
#pragma unroll
        for (int n = 0; n < NT; ++n)
#pragma unroll
            for (int t = 0; t < MT; ++t)
#pragma unroll
                for (int e = 0; e < 4; ++e) nan |= acc[n][t][e] != acc[n][t][e];
        if ((special & 0x80808080u) || nan) *any_special = 1;
        __syncthreads();
        const bool again = *any_special != 0;
        __syncthreads();
        if (again) run(std::true_type{});   // uniform
    }
    // lane holds C[token m0 + 64 wm + 16 t + 4 q + e][row n0 + WN wn + 16 n + j]
    if constexpr (!GROUPS) {
#pragma unroll
        for (int n = 0; n < NT; ++n) {
            const float inv = 1.0f / p.scales[(size_t)min(n0 + wn * WN + 16 * n + j, p.N - 1) * p.groups_per_row];
#pragma unroll
            for (int t = 0; t < MT; ++t)
#pragma unroll
                for (int e = 0; e < 4; ++e) acc[n][t][e] *= inv;
        }
    }
    if (gridDim.y > 1) {
#pragma unroll
        for (int n = 0; n < NT; ++n) {
            const int row = n0 + wn * WN + 16 * n + j;
#pragma unroll
            for (int t = 0; t < MT; ++t)
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    const int m = m0 + wm * 64 + 16 * t + 4 * q + e;
                    if (m < p.M && row < p.N) p.part[((size_t)blockIdx.y * p.M + m) * p.N + row] = acc[n][t][e];
                }
        }
        return;
    }
    // through LDS, a wavefront's 16 tokens at a time, to rows of 16-byte stores
    constexpr int kPitch = WN + 8;
    static_assert(4 * 16 * kPitch * 2 <= (int)sizeof(s0), "output tile");
    _Float16* o = reinterpret_cast<_Float16*>(s0) + wave * 16 * kPitch;
#pragma unroll
    for (int t = 0; t < MT; ++t) {
#pragma unroll
        for (int n = 0; n < NT; ++n)
#pragma unroll
            for (int e = 0; e < 4; ++e) o[(4 * q + e) * kPitch + 16 * n + j] = from_f32<_Float16>(acc[n][t][e]);
        // orders the compiler only: one wavefront's LDS operations execute in order
        __builtin_amdgcn_wave_barrier();
#pragma unroll
        for (int i0 = 0; i0 < 16 * WN / 8; i0 += kWave) {
            const int i = i0 + lane, r = i / (WN / 8), c = i % (WN / 8) * 8;
            const half8 v = *reinterpret_cast<const half8*>(o + r * kPitch + c);
            const int m = m0 + wm * 64 + 16 * t + r, col = n0 + wn * WN + c;
            if (m < p.M) {
                _Float16* dst = p.C + (size_t)m * p.N + col;
                if (p.wide_store && col + 8 <= p.N) {
                    *reinterpret_cast<half8*>(dst) = v;
                } else {
#pragma unroll
                    for (int e = 0; e < 8; ++e)
                        if (col + e < p.N) dst[e] = v[e];
                }
            }
        }
        __builtin_amdgcn_wave_barrier();
    }
}

struct TilePlan {
    int bn, stages, splits, steps_per_split;
    double us;
};

// Step time of a CU that has `load` workgroups of the launch (us), from the sweeps
// below: the first two fill its wavefront slots, more of them queue.
double step_us(bool groups, int bn, double load) {
    if (groups) return bn == 64 ? (load <= 1 ? 0.54 : load <= 2 ? 0.72 : 0.37 * load)
                                : (load <= 1 ? 0.80 : load <= 2 ? 1.20 : 0.70 * load);
    return bn == 64 ? (load <= 1 ? 0.37 : load <= 2 ? 0.55 : 0.31 * load)
                    : (load <= 1 ? 0.51 : load <= 2 ? 0.85 : 0.53 * load);
}

// Tile width and K-split of the lowest estimated time.  Measured on MI355X, E4M3 in
// groups of 128 with the reference decode, us per call (bn x splits): 333 x 14336 x 4096
// 64x1 63.6, 128x1 73.6, 64x2 77.5; 512 rows 64x1 90.1, 128x1 77.5; 200 x 4096 x 14336
// 64x1 107.6, 64x4 46.9, 64x8 52.9, 128x4 54.3; 65 x 1024 x 8192 64x1 63.0, 64x4 21.6,
// 64x8 15.5.  Per row, 333 x 14336 x 4096: 64x1 54.4, 128x1 49.9.
TilePlan tile_plan(int M, int N, int K, bool groups, size_t part_bytes) {
    TilePlan best{0, 0, 0, 0, 0.0};
    const int steps = K / kBK;
    for (int bn : {64, 128}) {
        const double tiles = (double)qlh::blocks_for(M, kBM) * qlh::blocks_for(N, bn);
        for (int want = 1; want <= 8; ++want) {
            const int per = (steps + want - 1) / want, splits = (steps + per - 1) / per;
            const double part = (double)splits * M * N * sizeof(float);   // written and read again
            if (splits != want || (splits > 1 && (per < 8 || part > (double)part_bytes))) continue;
            const double load = tiles * splits / 256;
            const double us = 3 + per * step_us(groups, bn, load) + (splits > 1 ? 3.5 + 2 * part / 5e6 : 0);
            if (!best.bn || us < best.us) best = {bn, bn == 64 && groups && load > 2 ? 2 : 3, splits, per, us};
        }
    }
    return best;
}

// The dequantizing path: the copy at 3 bytes a weight, then the library GEMM, whose
// rate grows with its number of tiles (333 / 512 / 800 / 1500 x 14336 x 4096: 674 / 910 /
// 989 / 1108 TFLOP/s; x 4096 x 14336: 502 / 647 / 717 / 979).
double dequantized_us(int M, int N, int K) {
    const double x = (double)M * N / 49152;
    return 6 + 6e-7 * N * K + 2.0 * M * N * K / (1.3e9 * x / (x + 60));
}

template <int FMT, int MODE, bool GROUPS>
void launch_bn(const TileArgs& a, const TilePlan& pl, hipStream_t st) {
    const dim3 grid((unsigned)(qlh::blocks_for(a.N, pl.bn) * (unsigned)a.m_tiles), (unsigned)pl.splits), block(kThreads);
    if (pl.bn == 128) {
        hipLaunchKernelGGL((fp8_gemm_tile<FMT, MODE, GROUPS, 128, 3>), grid, block, 0, st, a);
    } else if (pl.stages == 3) {
        hipLaunchKernelGGL((fp8_gemm_tile<FMT, MODE, GROUPS, 64, 3>), grid, block, 0, st, a);
    } else {
        if constexpr (GROUPS) hipLaunchKernelGGL((fp8_gemm_tile<FMT, MODE, GROUPS, 64, 2>), grid, block, 0, st, a);
    }
}

template <int FMT, int MODE>
void launch_groups(const TileArgs& a, const TilePlan& pl, bool groups, hipStream_t st) {
    if (groups) launch_bn<FMT, MODE, true>(a, pl, st);
    else launch_bn<FMT, MODE, false>(a, pl, st);
}

}  // namespace

bool qlh::fp8_gemm_tile(const Fp8TileCall& c, int* splits, hipStream_t stream) {
    // 32-bit byte offsets into the token rows and a workgroup's weight rows
    if (c.K % kBK || 2ull * (uint64_t)c.M * (uint64_t)c.K >= (1ull << 32) || 128ull * (uint64_t)c.K >= (1ull << 32))
        return false;
    if (!qlh::aligned16(c.A) || !qlh::aligned16(c.W)) return false;
    if (c.format == QL_FP8_E5M2 && c.mode == QL_FP8_MODE_REFERENCE) return false;   // codes beyond the binary16 range
    if (c.gs != 0 && c.gs != c.K && (c.K % c.gs || c.gs % kBK)) return false;
    const bool groups = c.gs != 0 && c.gs != c.K;
    const TilePlan pl = tile_plan(c.M, c.N, c.K, groups, c.part_bytes);
    // 8% in hand for the estimates (at 1500 rows both are within 10% of each other)
    if (pl.us > 0.92 * dequantized_us(c.M, c.N, c.K)) return false;
    if ((long long)qlh::blocks_for(c.M, kBM) * qlh::blocks_for(c.N, pl.bn) > INT32_MAX) return false;
    TileArgs a{};
    a.A = reinterpret_cast<const char*>(c.A);
    a.W = reinterpret_cast<const char*>(c.W);
    a.scales = c.scales;
    a.C = reinterpret_cast<_Float16*>(c.C);
    a.part = c.part;
    a.M = c.M;
    a.N = c.N;
    a.K = c.K;
    a.gs = groups ? c.gs : c.K;
    a.groups_per_row = c.gs == 0 ? 0 : c.K / c.gs;
    a.steps_per_split = pl.steps_per_split;
    a.m_tiles = (int)qlh::blocks_for(c.M, kBM);
    a.wide_store = c.N % 8 == 0 && qlh::aligned16(c.C);
    *splits = pl.splits;
    if (c.format == QL_FP8_E5M2) launch_groups<QL_FP8_E5M2, QL_FP8_MODE_OCP>(a, pl, groups, stream);
    else if (c.mode == QL_FP8_MODE_REFERENCE) launch_groups<QL_FP8_E4M3, QL_FP8_MODE_REFERENCE>(a, pl, groups, stream);
    else launch_groups<QL_FP8_E4M3, QL_FP8_MODE_OCP>(a, pl, groups, stream);
    return true;
}

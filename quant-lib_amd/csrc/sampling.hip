// sampling.hip -- greedy token selection over rows of logits.
//
// argmax_kernel (src/continuous_batch.cu:12-25) picks, for one row, the first
// index whose value is strictly greater than every earlier one and than the
// start value -1e20f (:15); NaN never compares greater, and a row with nothing
// above -1e20f gives 0.  (The fp16 engine's argmax_kernel,
// src/fp16_forward.cu:259-283, starts from -FLT_MAX instead: the two agree on
// every row that holds a value above -1e20f, which every binary16 row with a
// finite value does.)  Here one workgroup handles one
// row of a batch: each lane keeps its first strict maximum over a strided pass of
// 16-byte loads, then (value, index) pairs are reduced
// preferring the larger value and, on equal values, the smaller index -- the
// same answer as the sequential scan.
#include "ql_common.hpp"
#include "quantlib_amd.h"

#include <math.h>
#include <limits.h>

namespace {

using namespace ql;

constexpr float kStart = -1e20f;   // src/continuous_batch.cu:15

__device__ __forceinline__ void better(float& v, int& i, float v2, int i2) {
    if (v2 > v || (v2 == v && i2 < i)) {
        v = v2;
        i = i2;
    }
}

constexpr int kArgBlock = 1024;   // threads of a row's workgroup
constexpr int kArgUnroll = 4;     // 16-byte loads of a thread in flight

// What bounds it: one CU streams a row (about 50 GB/s), so a row wants every load in
// flight it can have: 16 wavefronts x 4 loads of 16 bytes.  The vectors are the aligned
// ones that cover the row, whatever its offset; elements outside it never win.
// Measured on MI355X, binary16, us for the argmax and the embedding gather after it,
// against 256 threads with one load each (element-wise off 16-byte alignment):
// 5 x 137001 68 -> 14.7, 64 x 128256 38 -> 15.5, 128 x 160000 47.7 -> 18.1; 8 x 32000 is
// bound by the two launches (10.1-11.1 either way).
template <typename D>
__global__ __launch_bounds__(kArgBlock) void argmax_rows(const D* __restrict__ x, int cols, int64_t ld,
                                                         int32_t* __restrict__ out) {
    constexpr int W = vec16<D>();
    const uintptr_t row = reinterpret_cast<uintptr_t>(x + (size_t)blockIdx.x * (size_t)ld);
    const int skip = (int)((row & 15) / sizeof(D));   // elements of the first vector before the row
    typedef const __attribute__((address_space(1))) u32x4* GlobalU4Ptr;
    const GlobalU4Ptr vecs = (GlobalU4Ptr)(row & ~(uintptr_t)15);
    const int nv = (int)(((long long)skip + cols + W - 1) / W);
    float best = kStart;
    int idx = INT_MAX;   // none yet
    for (long long c0 = threadIdx.x; c0 < nv; c0 += kArgBlock * kArgUnroll) {
        Vec<D, W> v[kArgUnroll];
        // past the end: the last vector again (the same elements never beat themselves)
#pragma unroll
        for (int u = 0; u < kArgUnroll; ++u)
            v[u] = __builtin_bit_cast(Vec<D, W>, __builtin_nontemporal_load(vecs + min(c0 + u * kArgBlock, (long long)nv - 1)));
#pragma unroll
        for (int u = 0; u < kArgUnroll; ++u) {
            const long long first = min(c0 + u * kArgBlock, (long long)nv - 1) * W - skip;
#pragma unroll
            for (int e = 0; e < W; ++e) {
                const float f = to_f32(v[u].v[e]);
                const long long i = first + e;
                if (f > best && i >= 0 && i < cols) {
                    best = f;
                    idx = (int)i;
                }
            }
        }
    }
    // lanes that saw nothing above the start keep (kStart, INT_MAX) and never win a tie
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) {
        const float v2 = __shfl_xor(best, o, kWave);
        const int i2 = __shfl_xor(idx, o, kWave);
        better(best, idx, v2, i2);
    }
    constexpr int kWaves = kArgBlock / kWave;
    __shared__ float sv[kWaves];
    __shared__ int si[kWaves];
    const int wave = threadIdx.x / kWave;
    if ((threadIdx.x & (kWave - 1)) == 0) {
        sv[wave] = best;
        si[wave] = idx;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
#pragma unroll
        for (int w = 1; w < kWaves; ++w) better(best, idx, sv[w], si[w]);
        out[blockIdx.x] = idx == INT_MAX ? 0 : idx;
    }
}

template <typename D>
hipError_t argmax_launch(const D* x, int rows, int cols, int64_t ld, int32_t* out,
                         hipStream_t stream) {
    QL_CHECK_ARG(rows >= 0 && cols > 0 && ld >= cols && rows <= 0x7fffffff);
    if (rows == 0) return hipSuccess;
    QL_CHECK_ARG(x && out);
    hipLaunchKernelGGL((argmax_rows<D>), dim3(rows), dim3(kArgBlock), 0, stream, x, cols, ld, out);
    return hipGetLastError();
}

}  // namespace

extern "C" hipError_t ql_argmax_f32(const float* logits, int rows, int cols, int64_t ld,
                                    int32_t* out, hipStream_t stream) {
    return argmax_launch<float>(logits, rows, cols, ld, out, stream);
}

extern "C" hipError_t ql_argmax_f16(const uint16_t* logits, int rows, int cols, int64_t ld,
                                    int32_t* out, hipStream_t stream) {
    return argmax_launch<_Float16>(reinterpret_cast<const _Float16*>(logits), rows, cols, ld, out,
                                   stream);
}

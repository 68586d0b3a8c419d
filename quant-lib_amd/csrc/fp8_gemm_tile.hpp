// fp8_gemm_tile.hpp -- the tiled FP8-weight GEMM of fp8_gemm_tile.hip, called by ql_fp8_gemm_f16.
#pragma once

#include <hip/hip_runtime_api.h>
#include <stddef.h>
#include <stdint.h>

namespace qlh {

// C[M, N] = A[M, K] (dequant W[N, K])^T.  gs: group length (K: per row; 0: per tensor).
struct Fp8TileCall {
    const uint16_t* A;
    const uint8_t* W;
    const float* scales;
    uint16_t* C;
    int M, N, K, gs, format, mode;
    float* part;           // fp32 partials of K-splits
    size_t part_bytes;     // 0: no K-split
};

// Launches the tiled kernel where it applies (sizes, scales, alignment) and is expected
// to be faster than dequantizing W for the library GEMM; false: nothing was launched.
// *splits > 1: c.part holds that many partials to be summed into C.
bool fp8_gemm_tile(const Fp8TileCall& c, int* splits, hipStream_t stream);

}  // namespace qlh

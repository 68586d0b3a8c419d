// fp8_gemm_pair.hpp -- two FP8-weight products of the same token rows (fp8.hip), called
// by the layer engine for gate and up.
#pragma once

#include <hip/hip_runtime_api.h>
#include <stddef.h>
#include <stdint.h>

namespace qlh {

// ql_fp8_gemm_f16 by W into C and by W2 into C2, matrices of one shape and options: one
// launch where a few-row kernel takes both, else one call after the other.
hipError_t fp8_gemm_pair(const uint16_t* A, const uint8_t* W, const float* scales, uint16_t* C, const uint8_t* W2,
                         const float* scales2, uint16_t* C2, int M, int N, int K, int format, int granularity,
                         int group_size, int mode, void* workspace, size_t workspace_bytes, hipStream_t stream);

}  // namespace qlh

// gemm_stream.hpp -- the few-row binary16 GEMM of gemm_stream.hip, called by ql_gemm_f16.
#pragma once

#include <hip/hip_runtime_api.h>
#include <stdint.h>

namespace qlh {

// Whether the weight-stream kernel takes y[M, N] = x[M, K] w[N, K]^T.
bool stream_gemm_f16_applies(const uint16_t* x, const uint16_t* w, int M, int N, int K);
hipError_t stream_gemm_f16(const uint16_t* x, const uint16_t* w, uint16_t* y, int M, int N, int K, hipStream_t stream);

}  // namespace qlh

// gemm_stream.hpp -- the few-row binary16 GEMM of gemm_stream.hip, called by ql_gemm_f16,
// and two products of the same rows.
#pragma once

#include <hip/hip_runtime_api.h>
#include <stdint.h>

namespace qlh {

// Whether the weight-stream kernel takes y[M, N] = x[M, K] w[N, K]^T (pair: together
// with a second matrix).
bool stream_gemm_f16_applies(const uint16_t* x, const uint16_t* w, int M, int N, int K, bool pair = false);
// w2: a second matrix of the same shape, y2 = x w2^T in the same launch.
hipError_t stream_gemm_f16(const uint16_t* x, const uint16_t* w, uint16_t* y, int M, int N, int K, hipStream_t stream,
                           const uint16_t* w2 = nullptr, uint16_t* y2 = nullptr);

// ql_gemm_f16 of x by w and by w2 (gate and up): one launch where the weight-stream
// kernel takes both, else one after the other.
hipError_t gemm_pair_f16(const uint16_t* x, const uint16_t* w, uint16_t* y, const uint16_t* w2, uint16_t* y2, int M,
                         int N, int K, hipStream_t stream);

}  // namespace qlh

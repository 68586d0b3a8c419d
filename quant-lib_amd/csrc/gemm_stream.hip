// gemm_stream.hip -- ql_gemm_f16 for at most 16 token rows: the weight stream of
// stream_gemm.hpp on binary16 weights.
#include "gemm_stream.hpp"
#include "quantlib_amd.h"
#include "stream_gemm.hpp"

namespace {

using namespace ql;

constexpr int kMaxTokens = 16;   // 17-32 tokens: the library is 0-6% faster on most shapes,
constexpr int kManyRows = 16384; // but not on more weight rows than this in a launch

template <int R, int MT = 1, int NW = 8>
void launch(const StreamArgs& a, hipStream_t st) {
    const dim3 grid(qlh::blocks_for(a.N, 16 * R), 1, a.W2 ? 2 : 1), block(NW * kWave);
    hipLaunchKernelGGL((stream_gemm<StreamF16, kStreamNone, MT, R, NW>), grid, block, 0, st, a);
}

}  // namespace

// Measured on MI355X, weights streamed from HBM, us per call at 1 / 4 / 16 tokens
// (R row tiles of 16 per workgroup; last: the library):
//   4096 x 4096    R 1  8.2 /  8.4 /  9.4   R 2 11.2 / 11.4 / 12   (12.4 / 9.8 / 9.9)
//   4096 x 14336   R 1 21.0 / 21.2 / 24.2   R 2 25.2 / 26.4 / 30.6   (24.3 / 24.7 / 25.6)
//   8192 x 2048    R 2  8.9 /  9.2 /  9.5   R 1  9.8 / 10.1 / 10.7   (13.7 / 10.8 / 11.4)
//   12288 x 4096   R 1 18.8 / 19.1 / 20.3   R 4 20.7 / 21.0 / 21.5   (20.1 / 21.1 / 21.4)
//   14336 x 4096   R 1 22.4 / 22.5 / 24.8   R 4 22.3 / 22.7 / 23.1   (22.8 / 23.4 / 23.5)
// The library keeps K above 4096 with more than 4096 rows (8192 x 8192: 26.2 / 26.4
// / 27.1 against 28.5-29.8), and K above 8192 with fewer than 3072 rows, where its
// K-split over workgroups fills the chip (512 x 14336: 10.3 / 10.5 / 11.6 against
// 13.0 / 13.5 / 18.0).
// Two products of the same rows (gate and up) in one launch save one fill and drain of
// the chip, which turns 17-32 rows of large matrices in the kernel's favour: a decode
// step of 32 sequences, two layers of 4096 with FFN 14336 and logits, 398 -> 387 us (both in 44.9 us, 5.2 TB/s;
// the library on the 32000 x 4096 logits 59.2 us, 4.4 TB/s, which come here too).
bool qlh::stream_gemm_f16_applies(const uint16_t* x, const uint16_t* w, int M, int N, int K, bool pair) {
    if (M > ((pair ? 2 : 1) * (long long)N > kManyRows ? 2 : 1) * kMaxTokens || K % kStreamChunk || K > kStreamMaxK || !qlh::aligned16(x) || !qlh::aligned16(w)) return false;
    return N > 4096 ? K <= 4096 : K <= 8192 || N >= 3072;
}

hipError_t qlh::stream_gemm_f16(const uint16_t* x, const uint16_t* w, uint16_t* y, int M, int N, int K,
                                hipStream_t stream, const uint16_t* w2, uint16_t* y2) {
    StreamArgs a{};
    a.A = reinterpret_cast<const char*>(x);
    a.W = reinterpret_cast<const char*>(w);
    a.C = reinterpret_cast<_Float16*>(y);
    a.W2 = reinterpret_cast<const char*>(w2);
    a.C2 = reinterpret_cast<_Float16*>(y2);
    a.M = M;
    a.N = N;
    a.K = K;
    a.chunks_per_split = K / kStreamChunk;
    if (M > kMaxTokens) launch<4, 2, 4>(a, stream);
    else if (N > 4096 && K <= 2048) launch<2>(a, stream);
    else if (N > 12288 && M > 8) launch<4>(a, stream);
    else launch<1>(a, stream);
    return hipGetLastError();
}

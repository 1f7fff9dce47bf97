// Kernels for calls of few tokens (few_tokens.hip): what lmhead_kernels.hip launches there instead of its 256 x 256 tiles.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace lmhead {

constexpr int kDwH = 128, kDwV = 256;  // tile of the weight gradient: hidden columns, vocabulary rows

struct DwFewArgs {
  const uint16_t* Hd;  // hidden [T, ldh], the first H columns
  int ldh;
  const uint16_t* D;   // dz panel [T rounded up to 256, ldd]
  int ldd;
  int T;
  const int* T_dev;    // when not NULL: the number of tokens, <= T, as a value in device memory
  int H;
  // Vocabulary rows of the chunk, and its moved last group: row n at or beyond n_tail is row n - n_back, and the first n_back of
  // those belong to the group before it (VocabTail in gemm_core.hpp).
  int N, n_tail, n_back;
  float* Cf;
  uint16_t* Cb;        // dW rows of the chunk [.., H]: one of the two
};

inline int64_t dw_few_tiles(int64_t H, int64_t N) { return (N + kDwV - 1) / kDwV * ((H + kDwH - 1) / kDwH); }

hipError_t launch_bwd_dw_few(hipStream_t s, const DwFewArgs& a);

}  // namespace lmhead

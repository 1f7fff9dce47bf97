// Kernels for calls of few tokens (few_tokens.hip): what lmhead_kernels.hip launches there instead of its 256 x 256 tiles.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "logits_tile.hpp"

namespace lmhead {

constexpr int kDwH = 128, kDwV = 256;  // tile of the weight gradient: hidden columns, vocabulary rows
constexpr int kDwUnitH = 64;           // hidden columns of what the kernel for more tokens makes at once

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
  int ncu;             // CUs of the device
};

// Up to this many tokens, of which any number may have a gradient, dW is made in those tiles, behind it with dz in registers, which takes 118 to 122 us
// for whatever is below 130 tokens (H=1536, V=151936): 88 -> 121 at 20, 123 -> 119 at 64, 144 -> 118 at 96, 152 -> 118 at 128.  Not at the sizes
// of the tie, because half of the tokens and more are often masked.
constexpr int64_t kDwTileTokens = 96;
// Behind it, where the device finds out how many tokens have a gradient, it also chooses: up to this many, two steps of the tiles, are made in tiles, by
// a launch in front that returns at once if there are more.  Training pass, H=1536, V=151936, dz in registers -> the device's choice: 478 -> 459 us with 20
// tokens of 137, 479 -> 469 with 40 and with 60; 490 -> 468, 488 -> 477 and 491 -> 480 of 200; 599 -> 578 with 20 of 611, 601 -> 591 with 60; 994 -> 981
// with 50 of 300 at H=4096, V=128261.  With 20 known to the host it would be 444.  What the choice costs a call that has more: 493 -> 495 with 137 of 137, 848 ->
// 846 with 428 of 611.
constexpr int kDwTileActive = 64;
// Whether the call is one for resident dz.  A workgroup's new dz rows cost it 6 us, for a row of H / 64 units: with short rows that is more than is
// saved.  Tiles -> resident dz, us, 137, 300 and 768 tokens: H=256, V=248320 48 -> 59, 66 -> 77, 124 -> 143 (fp32 result 73 -> 83 and 148 -> 169 at
// 137 and 768); V=151936, 120, 300, 500 and 768 tokens: H=512 56 -> 50, 81 -> 80, 105 -> 109, 136 -> 144; H=576 64 -> 51, 95 -> 84, 123 -> 114, 161 -> 151;
// H=384 42 -> 39, 60 -> 65 at 300, 88 -> 99 at 600; H=448 52 -> 45, 101 -> 102 at 500.  Of what stands here 2 to 4 us go to the device's choice.
inline bool dw_resident(int64_t T, int64_t H) { return T > kDwTileTokens && (H > 512 || (H > 384 && T <= 128)); }
inline int64_t dw_few_tiles(int64_t H, int64_t N) { return (N + kDwV - 1) / kDwV * ((H + kDwH - 1) / kDwH); }

hipError_t launch_bwd_dw_few(hipStream_t s, const DwFewArgs& a);

// Whether the logits of a call, forward or backward, are made on half tiles (half_tile.hpp): where one of them holds all tokens.
// Forward / whole backward with dW, square -> half tiles, V=151936: H=512 57 -> 39 / 183 -> 157 us at T=16, 58 -> 42 / 207 -> 186 at
// T=128; H=896 84 -> 62 / 285 -> 258, 86 -> 67 / 327 -> 308; H=1536 144 -> 121 / 425 -> 407, 150 -> 133 / 488 -> 479; H=4096, V=128261
// 259 -> 219, 270 -> 238; H=1024, V=32000 29 -> 25 at both.  Two half tiles along the tokens instead of one square tile:
// 88 -> 98 us at T=137, H=896, 145 -> 177 at H=1536, 269 -> 374 at H=4096; 58 -> 57 at H=512.
constexpr int64_t kHalfTileTokens = 128;
inline bool half_tile_logits(int64_t T) { return T <= kHalfTileTokens; }

void launch_fwd_half_tiles(hipStream_t s, bool entropy, const uint16_t* W, int ldw, const uint16_t* Hd, int ldh, int T, int H, int V,
                           float rcp_temp, float* part_max, float* part_sum, float* part_pz);
hipError_t launch_bwd_half_dz(hipStream_t s, bool entgrad, const DzArgs& z);

}  // namespace lmhead

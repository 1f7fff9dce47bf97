// HIP kernels (gfx950) and C-ABI entry points of the fused LM-head log-probability path.
//
// Forward  (2*T*V*H flop):
//   lmhead_fwd_tiles   one 256(vocab) x 256(token) logits tile per workgroup: bf16 MFMA GEMM, then in registers
//                      scale by 1/temperature, per-token max / sum-exp / sum (z-max)*exp over the tile's vocab rows;
//                      writes one (max, sum, pz) partial per token per 128-row half tile, in blocks of 64 tokens.  Logits
//                      never leave VGPRs.
//                      (Up to 128 tokens, here and for the dz tiles: half tiles, few_tokens.hip.)
//   lmhead_fwd_merge   per 16 tokens: merges the partials (online log-sum-exp), gathers the label logit with an
//                      fp32 dot product hidden[t] . weight[label], writes logprob / entropy / lse / pz.
// Backward (6*T*V*H flop), looped over vocab chunks of `vocab_chunk` columns:
//   transpose_bf16     hidden^T once per call (and weight^T only for small vocabularies that are not multiples of 128).
//   lmhead_bwd_dz      recompute a logits tile, form dz in registers and write it (bf16) into one token-major panel of
//                      the chunk.
//   lmhead_bwd_gemm    dHidden (+)= dz . weight and dW[chunk] = dz^T . hidden with fp32 accumulation, both from that
//                      panel -- dW reads it K-major, dHidden reads the weight K-major in place -- through the transposing
//                      LDS read (gemm_core.hpp).
// Soft cross-entropy of a draft head against the policy (10*T*V*H flop): softce_pack_rows stacks the two hidden rows of every
//   token, softce_fwd_tiles is the forward tile with a paired third statistic, softce_dz_tiles the matching dz producer; merge
//   and dHidden GEMM are the kernels above.
// The per-token loss kernels and the packed-sequence index kernels live in loss_kernels.hip and packed_kernels.hip.
#include <hip/hip_runtime.h>
#include <math.h>
#include <stdint.h>

#include <algorithm>
#include <mutex>
#include <vector>

#include "../../include/skyrl_lmhead.h"
#include "../../include/skyrl_lmhead_bench.h"
#include "dh_split.hpp"
#include "few_tokens.hpp"
#include "gemm_core.hpp"
#include "logits_tile.hpp"
#include "topk_kernels.hpp"

using namespace lmhead;

namespace {

static_assert(BM == kSplitTile && BN == kSplitTile && 2 * BK == kSplitPair, "the tiles that dh_split.hpp rates");

// Timing-only ablations for skyrl_amd/bench_ablations.py (results are wrong with any of them; 0 in the product build):
//   1  forward tiles skip their statistics epilogue        2  dz tiles skip their epilogue (arithmetic, staging, stores)
//   4  dz tiles do everything but the global stores        8  forward and dz tiles read the operand panels of one 4 x 8 patch
//  16  the same for the gradient-GEMM tiles                   of tiles, so that every operand read hits the XCD's L2
//  32, 64  in gemm_core.hpp: the mainloop without its LDS fragment reads / without its global -> LDS copies
#ifndef LMHEAD_ABLATE
#define LMHEAD_ABLATE 0
#endif
// Scratch matrices get 64 extra elements (128 B) per row: with a power-of-two row pitch (T' = 16384 -> 32 KiB) the 256 rows of
// an operand tile would all start in the same L2 channel and set.
constexpr int kLdPad = 64;

__host__ __device__ inline int64_t round_up(int64_t x, int64_t m) { return (x + m - 1) / m * m; }
// An even number of k-tiles selects the accumulator-stationary mainloop (the EVEN instantiation of a tile kernel).
inline bool even_ktiles(int64_t contraction) { return (contraction / BK) % 2 == 0; }

// Whether a launch of tiles_m x ceil(T / 256) tiles makes others than square ones, and how many of them as short ones.  The branches to them
// are compiled into kernels of their own, because they cost every tile about half a k-tile's time (V=151936; T=8192, H=896, where they save
// 0.4 of 75 rounds: 1768 us without them, 1796 with; T=20608, H=1536: 6688 and 6692 to 6724).  What they save, 0.4 or 0.2 of a tile in the
// last token column (128 or 192 tokens) and 0.4 of a round at the end, has to be more than that; a square tile takes H / 64 + 5 k-tiles' time.
struct TileShapes {
  bool used;
  int split;
};
inline bool shapes_pay(int64_t tenths_saved, int64_t H, int64_t tiles) { return tenths_saved * (H / BK + 5) > 5 * tiles; }
inline TileShapes tile_shapes(int64_t T, int64_t H, int tiles_m, int ncu) {
  const int64_t tiles = (T + BN - 1) / BN * tiles_m, rest = T % BN;
  const int split = split_last_round((int)tiles, ncu);
  const int64_t tenths = (rest == 0 || rest > BN * 3 / 4 ? 0 : rest > BN / 2 ? 2 : 4) * tiles_m + (split > 0 ? 4 * ncu : 0);
  const bool used = shapes_pay(tenths, H, tiles);
  return TileShapes{used, used ? split : 0};
}
// The same for a count of tokens that only the device knows: it may leave any remainder, and any number of tiles up to these.  On the average
// over the remainders a quarter of a tile is saved in the last token column.
inline TileShapes tile_shapes_of_any_count(int64_t H, int tiles_m, int tiles, int ncu) {
  const bool used = shapes_pay(10 * tiles_m / 4, H, tiles);
  return TileShapes{used, !used ? 0 : tiles < ncu / 2 ? tiles : ncu / 2};
}
// pick(x, y, z) for the three flags as compile-time constants.
template <class Pick>
auto flagged_kernel(Pick pick, bool x, bool y, bool z) {
  const std::true_type t;
  const std::false_type f;
  if (x) return y ? (z ? pick(t, t, t) : pick(t, t, f)) : (z ? pick(t, f, t) : pick(t, f, f));
  return y ? (z ? pick(f, t, t) : pick(f, t, f)) : (z ? pick(f, f, t) : pick(f, f, f));
}

// Scratch of skyrl_lmhead_fwd_static_scratch, the entry point for callers that cannot allocate: one fixed array in every
// device's memory, held until the process ends.  In host code this name is only a handle for hipGetSymbolAddress (see
// static_scratch_of_current_device); kernels receive the looked-up address as an ordinary argument.
constexpr size_t kStaticScratchBytes = SKYRL_LMHEAD_STATIC_SCRATCH_BYTES;
static __device__ __align__(256) unsigned char static_scratch[kStaticScratchBytes];

// ------------------------------------------------------------------------------------------------------------
// Forward tile kernel.  M axis = vocab (A = weight), N axis = tokens (B = hidden).
// Online softmax statistics follow efficient_entropy_kernel_general_mainloop
// (fused_linear_logprob_triton.py:296-385): scale, running max, sum exp, sum z*exp (kept relative to the maximum here); vocab rows past V take no part.
// The label-logit gather of that kernel (:364-385) is done in lmhead_fwd_merge instead.
// ------------------------------------------------------------------------------------------------------------
// EVEN: H / 64 is even, which selects the accumulator-stationary mainloop (gemm_core.hpp).
// SHAPES: some tiles are not square (tile_shapes()); split: how many of them are made as short ones.
template <bool ENTROPY, bool PAIRED, bool EVEN, bool SHAPES>
__device__ __forceinline__ void fwd_tile(const uint16_t* __restrict__ W, int ldw, const uint16_t* __restrict__ Hd, int ldh, int T,
                                         int H, int V, float rcp_temp, float* __restrict__ part_max,
                                         float* __restrict__ part_sum, float* __restrict__ part_pz, int split, char* lds) {
  const int tiles_m = (V + BM - 1) / BM;
  const int tiles_n = (T + BN - 1) / BN;
  const Tile t = tile_of<false, SHAPES>(blockIdx.x, tiles_m, tiles_n, kGroupM, split);
  const int wave = threadIdx.x >> 6;
  auto tile = [&](auto shape, int v0) {  // the tile of that shape from vocabulary row v0 on
    constexpr int SHAPE = decltype(shape)::value;
    const int part = v0 / WM + wave / waves_n(SHAPE), t0 = t.tn * BN + wave % waves_n(SHAPE) * (wave_cols(SHAPE) * MT);
#if LMHEAD_ABLATE & 8
    const Operand a{W, ldw, (t.tm % 4) * BM, V}, b{Hd, ldh, (t.tn % 8) * BN, T};
#else
    // A part behind the vocabulary (the upper half of the last tile): its statistics are empty whatever row is multiplied.
    const Operand a{W, ldw, SHAPE == kShort && v0 >= V ? V - 1 : v0, V}, b{Hd, ldh, t.tn * BN, T};
#endif
    f32x4 acc[TM][wave_cols(SHAPE)];
    tile_product<SHAPE, EVEN>(a, b, H / BK, lds, acc);
#if !(LMHEAD_ABLATE & 1)
    fwd_epilogue<ENTROPY, PAIRED>(acc, part, tiles_m * WAVES_M, t0, T, V, rcp_temp, part_max, part_sum, part_pz);
#endif
  };
  if constexpr (SHAPES) {
    const int shape = shape_of_tile(t.tn, T);
    if (shape == kNarrow) {  // of the two workgroups of a split tile the first makes it
      if (t.half < 1) tile(std::integral_constant<int, kNarrow>{}, t.tm * BM);
      return;
    }
    if (t.half >= 0) return tile(std::integral_constant<int, kShort>{}, t.tm * BM + t.half * WM);
    if (shape == kMedium) return tile(std::integral_constant<int, kMedium>{}, t.tm * BM);
  }
  tile(std::integral_constant<int, kSquare>{}, t.tm * BM);
}

template <bool ENTROPY, bool EVEN, bool SHAPES>
__global__ __launch_bounds__(NTHREADS) void lmhead_fwd_tiles(const uint16_t* __restrict__ W, int ldw,
                                                             const uint16_t* __restrict__ Hd, int ldh, int T, int H, int V,
                                                             float rcp_temp, float* __restrict__ part_max,
                                                             float* __restrict__ part_sum, float* __restrict__ part_pz, int split) {
  __shared__ __attribute__((aligned(1024))) char lds[LDS_BYTES];
  fwd_tile<ENTROPY, false, EVEN, SHAPES>(W, ldw, Hd, ldh, T, H, V, rcp_temp, part_max, part_sum, part_pz, split, lds);
}

// ------------------------------------------------------------------------------------------------------------
// Forward merge.  One workgroup of 16 waves per 16 tokens: lane = (token, part mod 4), wave w merges parts 4w .. 4w + 3, then
// every 64th of them (a load is 64 contiguous bytes of four parts), the running triples meet in shuffles and in LDS.  Wave w
// also takes the label logit of token w, 64 lanes to the dot product.
// What bounds it: 12 bytes per part and token and two rows per label from HBM for many tokens, the chain of load and merge steps
// for few.  Sixty-four streams per token and BATCH parts a step, 24 or 30 loads in flight per lane, keep that chain at two steps for 1188
// parts (16 streams of 64-token blocks: 19), with one exponential per part, and the label's rows are loaded with the first step.  Between
// HIP events (which add about 4 us), V=151936, eight parts a step and the label's rows behind them -> this way: 11.2 -> 10.6 us at T=137, 14.0
// -> 12.3 at T=611, 14.5 -> 13.2 at T=2048 with entropy, 34 and 34 at T=8192, 81 and 82 at T=16384, H=3584 (5.8 TB/s).
// Merge algebra as in efficient_entropy_triton_kernel_epilogue (fused_linear_logprob_triton.py:417-467) except that
// the running max starts at -inf (that kernel starts it at 0, which loses rows whose logits are all << 0).
// Out-of-range labels give logprob 0 (model_utils.py:337; fused_linear_logprob_triton.py:1898-1905).
// ------------------------------------------------------------------------------------------------------------
constexpr int kMergeTokens = 16;
constexpr int kMergeThreads = 1024;
constexpr int kMergeWaves = kMergeThreads / 64;
constexpr int kMergeStreams = kMergeWaves * 4;  // of parts per token
static_assert(kMergeWaves == kMergeTokens && kPartTokens % kMergeTokens == 0, "one wave per token for the label logit");

// Partial triples (maximum, sum e^(z - max), third statistic) of one token become one.  RELATIVE: the third statistic is
// sum (z - max) e^(z - max) and moves with the maximum, e' = c (e + (max - max') s); otherwise it is sum y e^(z - max) of some y that
// does not depend on the maximum and only scales.  A part without a sum (no vocabulary row, or logits that are all -inf) must come
// in with a maximum of -inf and zeros, so that it raises no maximum; a NaN in a sum stays.
// One exponential per part, taken relative to the largest maximum of the batch: the parts of a batch do not wait for each
// other.  (2^(d log2 e) through v_exp_f32: its relative error grows with |d|, the part's weight falls faster; |d| e^d < 0.4.)
template <bool RELATIVE, int N>
__device__ __forceinline__ void merge_partials(float& M, float& S, float& E, const float (&m)[N], const float (&s)[N],
                                               const float (&e)[N]) {
  float top = M;
#pragma unroll
  for (int u = 0; u < N; ++u) top = fmaxf(top, m[u]);
  if (!(top > -INFINITY)) return;
  auto add = [&](float mu, float su, float eu, float& sum_s, float& sum_e) {
    const float d = fmaxf(mu - top, -1.0e30f);  // finite: an empty part has s = e = 0
    const float c = __builtin_amdgcn_exp2f(d * kLog2e);
    // Explicit fused multiply-adds: which products the compiler would contract is its choice, and it need not make the same one
    // in every build.
    sum_s = fmaf(su, c, sum_s);
    sum_e = fmaf(RELATIVE ? fmaf(d, su, eu) : eu, c, sum_e);
  };
  float sum_s = 0.f, sum_e = 0.f;
  add(M, S, E, sum_s, sum_e);
#pragma unroll
  for (int u = 0; u < N; ++u) add(m[u], s[u], e[u], sum_s, sum_e);
  M = top, S = sum_s, E = sum_e;
}

// The triple of lane ^ o joins this lane's.
template <bool RELATIVE>
__device__ __forceinline__ void merge_lanes(float& M, float& S, float& E, int o) {
  const float m[1] = {__shfl_xor(M, o, 64)}, s[1] = {__shfl_xor(S, o, 64)}, e[1] = {__shfl_xor(E, o, 64)};
  merge_partials<RELATIVE>(M, S, E, m, s, e);
}

template <bool RELATIVE, int BATCH>
__global__ __launch_bounds__(kMergeThreads) void lmhead_fwd_merge(const float* __restrict__ part_max,
                                                                  const float* __restrict__ part_sum,
                                                                  const float* __restrict__ part_pz, int nparts, int T,
                                                                  const uint16_t* __restrict__ Hd, int ldh,
                                                                  const uint16_t* __restrict__ W, int ldw,
                                                                  const int64_t* __restrict__ labels, int H, int V, float rcp_temp,
                                                                  float* __restrict__ logprobs, float* __restrict__ entropy,
                                                                  float* __restrict__ row_lse, float* __restrict__ row_pz) {
  __shared__ float sm_m[kMergeWaves][kMergeTokens], sm_s[kMergeWaves][kMergeTokens], sm_e[kMergeWaves][kMergeTokens];
  __shared__ float sm_dot[kMergeTokens];
  __shared__ int sm_has_label[kMergeTokens];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  // Four consecutive workgroups read the same cache lines (16 of a block's 64 tokens each): keep them on one XCD.
  const int t0 = xcd_contiguous(blockIdx.x, gridDim.x) * kMergeTokens;
  const int64_t y = (labels && t0 + wave < T) ? labels[t0 + wave] : (int64_t)-1;
  const int t = t0 + (lane & 15);
  const size_t base = part_index(0, t < T ? t : T - 1, nparts);
  const int first = wave * 4 + (lane >> 4);
  float m[BATCH], sv[BATCH], ev[BATCH];
  auto load_batch = [&](int p0) {  // parts p0, p0 + kMergeStreams, ...; behind the last one: part 0, dropped below
#pragma unroll
    for (int u = 0; u < BATCH; ++u) {
      const int p = p0 + u * kMergeStreams;
      const size_t idx = base + (size_t)(p < nparts ? p : 0) * kPartTokens;
      m[u] = part_max[idx];
      sv[u] = part_sum[idx];
      ev[u] = part_pz ? part_pz[idx] : 0.f;
    }
  };
  load_batch(first);
  // Label logit: 16-byte loads, fp32 accumulation.  Its two rows travel together with the first batch of the partials.
  float dot = 0.f;
  const bool has_label = y >= 0 && y < (int64_t)V;
  if (has_label) {
    const uint16_t* hp = Hd + (size_t)(t0 + wave) * (size_t)ldh;
    const uint16_t* wp = W + (size_t)y * (size_t)ldw;
#pragma unroll 4
    for (int c = lane * 8; c < H; c += 64 * 8) {
      const uint4 hv = *(const uint4*)(hp + c);
      const uint4 wv = *(const uint4*)(wp + c);
      const uint32_t hh[4] = {hv.x, hv.y, hv.z, hv.w};
      const uint32_t ww[4] = {wv.x, wv.y, wv.z, wv.w};
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        dot = fmaf(__uint_as_float(hh[k] << 16), __uint_as_float(ww[k] << 16), dot);
        dot = fmaf(__uint_as_float(hh[k] & 0xffff0000u), __uint_as_float(ww[k] & 0xffff0000u), dot);
      }
    }
  }
  {
    float M = -INFINITY, S = 0.f, E = 0.f;
    for (int p0 = first; p0 < nparts;) {
#pragma unroll
      for (int u = 0; u < BATCH; ++u)
        if (p0 + u * kMergeStreams >= nparts || sv[u] == 0.f) m[u] = -INFINITY, sv[u] = 0.f, ev[u] = 0.f;
      merge_partials<RELATIVE>(M, S, E, m, sv, ev);
      p0 += kMergeStreams * BATCH;
      if (p0 < nparts) load_batch(p0);
    }
    merge_lanes<RELATIVE>(M, S, E, 16);
    merge_lanes<RELATIVE>(M, S, E, 32);
    if (lane < kMergeTokens) sm_m[wave][lane] = M, sm_s[wave][lane] = S, sm_e[wave][lane] = E;
  }
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) dot += __shfl_xor(dot, o, 64);
  if (lane == 0) sm_dot[wave] = dot, sm_has_label[wave] = has_label;
  __syncthreads();
  if (wave != 0) return;
  const int tl = lane & 15;
  float M = -INFINITY, S = 0.f, E = 0.f;
  float wm[kMergeWaves / 4], ws[kMergeWaves / 4], we[kMergeWaves / 4];
#pragma unroll
  for (int u = 0; u < kMergeWaves / 4; ++u) {
    const int w = (lane >> 4) * (kMergeWaves / 4) + u;
    wm[u] = sm_m[w][tl], ws[u] = sm_s[w][tl], we[u] = sm_e[w][tl];
  }
  merge_partials<RELATIVE>(M, S, E, wm, ws, we);
  merge_lanes<RELATIVE>(M, S, E, 16);
  merge_lanes<RELATIVE>(M, S, E, 32);
  if (lane >= kMergeTokens || t >= T) return;
  const float log_s = logf(S), lse = M + log_s;
  // RELATIVE: the entropy itself, ln s - e / s, comes out of the sums, and sum p z is recovered as lse - entropy (exactly what
  // the absolute form subtracts the other way round).
  const float third = RELATIVE ? log_s - E / S : E / S;
  if (logprobs) logprobs[t] = sm_has_label[tl] ? sm_dot[tl] * rcp_temp - lse : 0.f;
  if (entropy) entropy[t] = RELATIVE ? third : lse - third;
  if (row_lse) row_lse[t] = lse;
  if (row_pz) row_pz[t] = RELATIVE ? lse - third : third;
}

// Ten parts a step where that saves the first or the second of the steps that eight take (lanes without a part of their own load and drop
// one): with ten instead of eight 8.5 -> 7.7 us at 137 tokens of V=80000 (ten parts per stream), 11.5 -> 10.6 at V=151936 (19), but 8.5 -> 9.2
// at V=100000 (13), 10.2 -> 10.8 at V=200064 (25), and 29 -> 38 at 32768 tokens of V=32000 (4).  The same for every number of tokens, so that
// a token's sums do not depend on it.
template <bool RELATIVE>
auto merge_kernel(int64_t nparts) {
  const int64_t n = (nparts + kMergeStreams - 1) / kMergeStreams;
  return n <= 20 && (n + 9) / 10 < (n + 7) / 8 ? &lmhead_fwd_merge<RELATIVE, 10> : &lmhead_fwd_merge<RELATIVE, 8>;
}

// The dz tiles (logits_tile.hpp) on products of any shape.
template <bool ENTGRAD, bool EVEN, bool SHAPES>
__device__ __forceinline__ void dz_square_tile(const DzArgs& z, int id, char* lds) {
  static_assert(NWAVES * WN * (kDzTokRow + kDzTokBytes) <= LDS_BYTES, "dz staging and per-token values do not fit LDS");
  int T;
  Tile t;
  if (!dz_tile_of<SHAPES>(z, id, BN, T, t)) return;
  auto tile = [&](auto shape, int col0) {
    constexpr int SHAPE = decltype(shape)::value;
    dz_tile<ENTGRAD, wave_cols(SHAPE), SHAPE == kShort>(
        z, T, col0, t.tn * BN, lds,
        [&](Operand a, Operand b, f32x4 (&acc)[TM][wave_cols(SHAPE)]) {
#if LMHEAD_ABLATE & 8
          a.row0 = z.vc0 + (t.tm % 4) * BM, b.row0 = (t.tn % 8) * BN;
#endif
          tile_product<SHAPE, EVEN>(a, b, z.H / BK, lds, acc);
          return !(LMHEAD_ABLATE & 2);
        },
        [](u32x4 v, u32x4* p) {
#if LMHEAD_ABLATE & 4
          asm volatile("" ::"v"(v), "v"(p));  // staged and read back, not stored
#else
          __builtin_nontemporal_store(v, p);
#endif
        });
  };
  if constexpr (SHAPES) {
    const int shape = shape_of_tile(t.tn, T);
    if (shape == kNarrow) {  // of the two workgroups of a split tile the first makes it
      if (t.half < 1) tile(std::integral_constant<int, kNarrow>{}, t.tm * BM);
      return;
    }
    if (t.half >= 0) return tile(std::integral_constant<int, kShort>{}, t.tm * BM + t.half * WM);
    if (shape == kMedium) return tile(std::integral_constant<int, kMedium>{}, t.tm * BM);
  }
  tile(std::integral_constant<int, kSquare>{}, t.tm * BM);
}

// ------------------------------------------------------------------------------------------------------------
// Soft cross-entropy from hidden states (the draft-head loss of multi-token prediction, skyrl/backends/skyrl_train/mtp/
// soft_ce.py:200-240):  loss[t] = -sum_v softmax(z_teacher[t])_v * log_softmax(z_student[t])_v = lse_student - E_teacher[z_student],
// both logits rows being products with the same (detached) output weight.  The reference materialises both [T, V] logits
// tensors and their fp32 softmaxes; here the two hidden rows of a token sit in one "stacked" operand so that one lane
// holds z_student and z_teacher of the same (token, vocab) pair, one accumulator block apart:
//   stacked row of token t:   student  (t / 16) * 32 + t % 16,   teacher  (t / 16) * 32 + 16 + t % 16
// i.e. a wave's token blocks are in turn 16 student rows and the 16 teacher rows of the same tokens, so that a tile of any shape
// holds whole pairs and calls of few tokens use them (V=151936, forward and backward, square tiles -> this: 389 -> 341 us at T=16, H=1536;
// 557 -> 521 at T=137, H=2048; 7.27 -> 7.23 ms at T=4096, where all tiles are square).  The forward
// is the ordinary tile kernel on the stacked rows with the paired third statistic; the backward recomputes a tile and writes
//   d loss / d z_student = g * (softmax(z_student) - softmax(z_teacher))  (soft_ce.py:146-151) for the student rows
// into the token-major dz panel, from which the ordinary dHidden GEMM runs.  The weight gets no gradient (it is detached
// in the reference, mtp/adapter.py:51-56), neither does the teacher.
// ------------------------------------------------------------------------------------------------------------
constexpr int kPairRows = MT;
__host__ __device__ inline int stacked_rows(int T) { return (T + kPairRows - 1) / kPairRows * (2 * kPairRows); }

__host__ __device__ inline int64_t stacked_row(int64_t t, bool teacher) {
  return (t / kPairRows) * (2 * kPairRows) + (teacher ? kPairRows : 0) + t % kPairRows;
}

// One workgroup per stacked row: copies the student's or the teacher's hidden row, zeros for the padding tokens.
// Teacher row of token t = b * seq_len + s is the teacher's hidden row b * seq_len + (s + shift) mod seq_len: the roll of
// build_teacher_logits (soft_ce.py:22-34) applied to the hidden states instead of the logits.
__device__ __forceinline__ const uint16_t* softce_source_row(int t, bool is_teacher, const uint16_t* student, int lds_,
                                                             const uint16_t* teacher, int ldt, int seq_len, int shift) {
  if (!is_teacher) return student + (size_t)t * (size_t)lds_;
  const int b = t / seq_len, sft = (t % seq_len + shift) % seq_len;
  return teacher + (size_t)(b * seq_len + sft) * (size_t)ldt;
}

__global__ __launch_bounds__(256) void softce_pack_rows(const uint16_t* __restrict__ student, int lds_,
                                                        const uint16_t* __restrict__ teacher, int ldt, int T, int seq_len,
                                                        int shift, int H, uint16_t* __restrict__ stacked) {
  const int r = blockIdx.x;
  const bool is_teacher = (r / kPairRows) & 1;
  const int t = r / (2 * kPairRows) * kPairRows + r % kPairRows;
  const uint16_t* src = t < T ? softce_source_row(t, is_teacher, student, lds_, teacher, ldt, seq_len, shift) : nullptr;
  uint16_t* dst = stacked + (size_t)r * (size_t)H;
  for (int c = threadIdx.x * 8; c < H; c += 256 * 8)
    *(uint4*)(dst + c) = src ? *(const uint4*)(src + c) : make_uint4(0, 0, 0, 0);
}

// The same for the backward, which runs on the tokens with an upstream gradient only (compact_active_rows: idx, counts): stacked
// rows and per-token inputs of compacted token t are those of token idx[t].  Rows beyond the last 16 tokens that hold one are
// not written.  As student row, token t also clears d_student[t]; active tokens get their row from the dHidden GEMM.
__global__ __launch_bounds__(256) void softce_gather_rows(const uint16_t* __restrict__ student, int lds_,
                                                          const uint16_t* __restrict__ teacher, int ldt, int T, int seq_len,
                                                          int shift, int H, const int* __restrict__ idx,
                                                          const int* __restrict__ counts, const float* __restrict__ lse_student,
                                                          const float* __restrict__ lse_teacher, const float* __restrict__ dloss,
                                                          uint16_t* __restrict__ stacked, float* __restrict__ lse_student_c,
                                                          float* __restrict__ lse_teacher_c, float* __restrict__ dloss_c,
                                                          uint16_t* __restrict__ d_student) {
  const int r = blockIdx.x;
  const bool is_teacher = (r / kPairRows) & 1;
  const int t = r / (2 * kPairRows) * kPairRows + r % kPairRows, n = counts[0];
  if (!is_teacher && t < T) {
    uint16_t* zero_row = d_student + (size_t)t * (size_t)H;
    for (int c = threadIdx.x * 8; c < H; c += 256 * 8) *(uint4*)(zero_row + c) = make_uint4(0, 0, 0, 0);
  }
  if (r >= stacked_rows(n)) return;
  const uint16_t* src = nullptr;
  if (t < n) {
    const int token = idx[t];
    src = softce_source_row(token, is_teacher, student, lds_, teacher, ldt, seq_len, shift);
    if (!is_teacher && threadIdx.x == 0)
      lse_student_c[t] = lse_student[token], lse_teacher_c[t] = lse_teacher[token], dloss_c[t] = dloss[token];
  }
  uint16_t* dst = stacked + (size_t)r * (size_t)H;
  for (int c = threadIdx.x * 8; c < H; c += 256 * 8)
    *(uint4*)(dst + c) = src ? *(const uint4*)(src + c) : make_uint4(0, 0, 0, 0);
}

template <bool EVEN, bool SHAPES>
__global__ __launch_bounds__(NTHREADS) void softce_fwd_tiles(const uint16_t* __restrict__ W, int ldw,
                                                             const uint16_t* __restrict__ Hd, int ldh, int T, int H, int V,
                                                             float rcp_temp, float* __restrict__ part_max,
                                                             float* __restrict__ part_sum, float* __restrict__ part_pz, int split) {
  __shared__ __attribute__((aligned(1024))) char lds[LDS_BYTES];
  fwd_tile<true, true, EVEN, SHAPES>(W, ldw, Hd, ldh, T, H, V, rcp_temp, part_max, part_sum, part_pz, split, lds);
}

// Per token: the merged statistics of its two stacked rows -> loss and the two log-sum-exps the backward needs.
__global__ __launch_bounds__(256) void softce_finish(const float* __restrict__ row_lse, const float* __restrict__ row_pz, int T,
                                                     float* __restrict__ loss, float* __restrict__ lse_student,
                                                     float* __restrict__ lse_teacher) {
  const int t = blockIdx.x * 256 + threadIdx.x;
  if (t >= T) return;
  const int64_t rs = stacked_row(t, false), rt = stacked_row(t, true);
  const float ls = row_lse[rs];
  loss[t] = ls - row_pz[rt];  // row_pz of a teacher row is E_teacher[z_student]
  lse_student[t] = ls;
  lse_teacher[t] = row_lse[rt];
}

struct SoftCeDzArgs {
  const uint16_t* W;
  int ldw;
  const uint16_t* S;  // stacked hidden rows [stacked_rows(tokens), H]
  int H, V;
  const int* T_dev;   // the number of tokens, counted on the device; token tiles beyond it return at once
  float rcp_temp;
  const float* lse_student;
  const float* lse_teacher;
  const float* dloss;
  int vc0, tiles_m, tiles_n;  // first vocab row of the chunk; tiles along the chunk's vocab rows and the stacked rows
  VocabTail tail;
  uint16_t* D;                // [tokens rounded up to 128, ldd]  dz of the student rows, token-major; rows behind the last tile are not written
  int ldd;
  int ncu;
};

// The tile of SHAPE from panel column col0 and token tok0 on, of T >= 1.
template <bool EVEN, int SHAPE>
__device__ __forceinline__ void softce_dz_tile(const SoftCeDzArgs& z, int T, int col0, int tok0, char* lds) {
  constexpr int N = wave_cols(SHAPE), PAIRS = N / 2;  // a wave's token blocks, and those of its student rows
  const uint16_t* __restrict__ W = z.W;
  const int V = z.V, vc0 = z.vc0, ldd = z.ldd;
  uint16_t* __restrict__ D = z.D;

  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int wm = wave / waves_n(SHAPE), wn = wave % waves_n(SHAPE);
  const int lrow = lane & 15, kq = lane >> 4;
  const int vloc_base = col0 + wm * WM;
  const WaveRows rows = wave_vocab_rows(vc0 + vloc_base, V, z.tail);
  const int tokbase = tok0 + wn * (PAIRS * MT);  // first token of this wave
  const bool full = rows.lo == 0 && rows.hi == WM;
  const float scale2 = z.rcp_temp * kLog2e;

  // Per-token inputs: unconditional loads from a clamped index, issued before the mainloop and first touched behind it (as
  // in dz_tile: a load under `t < T` is a branch with its own wait in front of the first copy).
  float gs_[PAIRS], ls2_[PAIRS], lt2_[PAIRS];
#pragma unroll
  for (int j = 0; j < PAIRS; ++j) {
    const int t = tokbase + j * MT + lrow;
    const int tc = t < T ? t : T - 1;
    gs_[j] = z.dloss[tc];
    ls2_[j] = z.lse_student[tc];
    lt2_[j] = z.lse_teacher[tc];
  }

  Operand a = dz_weight_rows(W, z.ldw, vc0 + col0, V, z.tail);
  if (SHAPE == kShort && a.row0 >= V) a.row0 = V - 1;  // as in dz_tile
  const Operand b{z.S, z.H, 2 * tok0, stacked_rows(T)};
  f32x4 acc[TM][N];
  tile_product<SHAPE, EVEN>(a, b, z.H / BK, lds, acc);
#pragma unroll
  for (int j = 0; j < PAIRS; ++j) {
    const bool valid = tokbase + j * MT + lrow < T;
    gs_[j] = valid ? gs_[j] * z.rcp_temp : 0.f;
    ls2_[j] = valid ? ls2_[j] * kLog2e : INFINITY;
    lt2_[j] = valid ? lt2_[j] * kLog2e : INFINITY;
  }

  // Staging as in dz_tile: a private region per wave, its token rows of 128 vocab columns, then 16-byte non-temporal stores.
  constexpr int kTokRow = WM * 2 + 16;
  constexpr int kStage = PAIRS * MT * kTokRow;
  char* stage = lds + wave * kStage;
  auto flush_block = [&](int j) {  // as in dz_tile: a finished token block leaves while the next one is computed
#pragma unroll
    for (int it = 0; it < 4; ++it) {
      const int idx = it * 64 + lane;
      const int n = j * MT + (idx >> 4), c = idx & 15;
      const u32x4 v = *(const u32x4*)(stage + n * kTokRow + c * 16);
      __builtin_nontemporal_store(v, (u32x4*)(D + (size_t)(tokbase + n) * (size_t)ldd + vloc_base + c * 8));
    }
  };
#pragma unroll
  for (int j = 0; j < PAIRS; ++j) {
    const float gs = gs_[j], ls2 = ls2_[j], lt2 = lt2_[j];
#pragma unroll
    for (int i = 0; i < TM; ++i) {
      float d[4];
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const float q = __builtin_amdgcn_exp2f(fmaf(acc[i][2 * j][r], scale2, -ls2));
        const float p = __builtin_amdgcn_exp2f(fmaf(acc[i][2 * j + 1][r], scale2, -lt2));
        d[r] = gs * (q - p);
      }
      const int vl = i * MT + kq * 4;
      if (!full) {
#pragma unroll
        for (int r = 0; r < 4; ++r)
          if (vl + r < rows.lo || vl + r >= rows.hi) d[r] = 0.f;
      }
      f32x4 v4 = {d[0], d[1], d[2], d[3]};
      const bf16x4 b4 = __builtin_convertvector(v4, bf16x4);
      *(uint2*)(stage + (j * MT + lrow) * kTokRow + vl * 2) = *(const uint2*)&b4;
      if (i == TM / 2 - 1 && j > 0) flush_block(j - 1);
    }
  }
  flush_block(PAIRS - 1);
}

template <bool EVEN, bool SHAPES>
__global__ __launch_bounds__(NTHREADS) void softce_dz_tiles(const SoftCeDzArgs z) {
  __shared__ __attribute__((aligned(1024))) char lds[LDS_BYTES];
  const int T = __builtin_amdgcn_readfirstlane(*z.T_dev);
  const int tiles_n = (T + BN / 2 - 1) / (BN / 2);
  const int split = SHAPES ? split_last_round(z.tiles_m * tiles_n, z.ncu) : 0;
  if ((int)blockIdx.x >= z.tiles_m * tiles_n + split) return;
  const Tile t = tile_of<true, SHAPES>(blockIdx.x, z.tiles_m, tiles_n, kGroupM, split);  // as in dz_tile_of
  const int tok0 = t.tn * (BN / 2);
  if constexpr (SHAPES) {
    const int shape = shape_of_tile(t.tn, stacked_rows(T));
    if (shape == kNarrow) {  // of the two workgroups of a split tile the first makes it
      if (t.half < 1) softce_dz_tile<EVEN, kNarrow>(z, T, t.tm * BM, tok0, lds);
      return;
    }
    if (t.half >= 0) return softce_dz_tile<EVEN, kShort>(z, T, t.tm * BM + t.half * WM, tok0, lds);
    if (shape == kMedium) return softce_dz_tile<EVEN, kMedium>(z, T, t.tm * BM, tok0, lds);
  }
  softce_dz_tile<EVEN, kSquare>(z, T, t.tm * BM, tok0, lds);
}

// ------------------------------------------------------------------------------------------------------------
// Plain NT GEMM with an fp32 / bf16 store epilogue:  C[N,M] (+)= B[N,K] . A[M,K]^T, i.e. C[n][m] = sum_k A[m][k] B[n][k]:
// the MFMA M axis (rows of A) runs along the contiguous dimension of C, because a lane's four accumulator values are
// consecutive along M -- one 16-byte fp32 (8-byte bf16) store.  M must be a multiple of 4.
//   Cin != 0   add the existing fp32 C before storing (accumulation across micro-batches)
//   Cf  != 0   store fp32;   Cb != 0  store bf16 (round-to-nearest-even)
// One launch carries up to two independent problems (workgroups [0, tiles0) work on p0, the rest on p1): the dHidden
// and dWeight products of a vocab chunk have no dependency on each other, and together they fill the 256 CUs in whole
// rounds where each alone leaves a partial last round.
// ------------------------------------------------------------------------------------------------------------
constexpr int kSlabWaveFloats = TM * TN * 64 * 4;            // one wave's accumulators
constexpr int64_t kSlabTileFloats = NWAVES * kSlabWaveFloats;  // one tile's: 256 KiB
struct GemmArgs {
  const uint16_t* A;
  int lda, a_rows;
  const uint16_t* B;
  int ldb, b_rows;  // K-major B: b_rows is the number of valid columns (n) of the stored matrix
  int b_kmajor;     // B is stored K-major, B[k * ldb + n]
  int c_rows_m;     // the bf16 output is C[m * ldc + n] (n contiguous) instead of C[n * ldc + m]
  int nk, M, N;
  const float* Cin;
  float* Cf;
  uint16_t* Cb;
  int ldc;
  // Partial sums that leave a launch (dHidden: from vocab chunk to vocab chunk, and from the splits of its contraction) live in
  // "accumulator order": split by split, tile by tile, wave by wave, MFMA block by MFMA block, each lane's 4 registers
  // contiguous.  Reading and writing them is 16 bytes per lane and 1 KiB contiguous per wave instruction, with no address
  // arithmetic beyond a constant offset.  p_first: nothing to add yet; p_last: the sum is complete with this launch, and without
  // splits it leaves as C.
  float* P;
  int p_first, p_last;
  // Number of splits of the contraction: workgroups per C tile, each with its share of the k-tile pairs and its own slab of P,
  // summed by lmhead_dh_reduce; in lmhead_bwd_dh_shares a code of Shares.  splits_dev, when not NULL, replaces it (what compact_active_rows chose for its token count).
  int splits;
  const int* splits_dev;
  // When not NULL: row m of the bf16 output is row row_map[m] of C.
  const int* row_map;
  // When not NULL: a token count in device memory that replaces one extent of the problem, chosen by t_role: the rows M
  // (kTokensOnM), the columns N (kTokensOnN) or the contraction length, nk = ceil(count / 64) (kTokensOnK).  The host-side
  // value of that extent is an upper bound that sizes the grid and the scratch; tiles beyond the count return at once.
  const int* T_dev;
  int t_role;
  // The moved last group of a vocabulary that is not a multiple of 128 (VocabTail), relative to the chunk.  dHidden contracts
  // over it: the last pair of its k-tiles reads the weight k_back rows earlier.  dW has it as output rows: row n at or beyond
  // n_tail is row n - n_back, and the first n_back of those belong to the group before it.
  int k_back, n_tail, n_back;
};
enum { kTokensOnM = 1, kTokensOnN = 2, kTokensOnK = 3 };

// BKM: the B operand is K-major.  The two variants are separate instantiations of the whole tile (mainloop and
// epilogue) so that their accumulators never meet at a join, where the register allocator would shuffle all 256 of them.
// Tile (tm, tn), its k-tiles k0 .. k0 + nk - 1, the slab `slot` of P; partial: the sum stays there.
template <bool BKM>
__device__ __forceinline__ void gemm_tile_at(const GemmArgs& p, int M, int N, int tm, int tn, int k0, int nk, int k_back, size_t slot, bool partial, char* lds);

template <bool BKM>
__device__ __forceinline__ void gemm_tile(const GemmArgs& p, int bid, char* lds) {
  int M = p.M, N = p.N, nk = p.nk;
  if (p.T_dev) {
    const int count = __builtin_amdgcn_readfirstlane(*p.T_dev);
    if (p.t_role == kTokensOnM) M = count;
    else if (p.t_role == kTokensOnN) N = count;
    else nk = (count + kTokenGroup - 1) / kTokenGroup * 2;  // whole pairs of k-tiles: the panel's rows up to the next kTokenGroup are zeros
    // Nothing to contract: C += 0 needs no work; a C that is overwritten or converted still goes through the epilogue.
    if (nk == 0 && !p.Cb && p.Cin == p.Cf) return;
  }
  const int splits = p.splits_dev ? __builtin_amdgcn_readfirstlane(*p.splits_dev) : p.splits;
  // Tiles of the extents in force: with a device-side count the tiles that hold tokens are numbered from 0, so that the
  // round-robin of workgroup ids over the XCDs spreads exactly those, and the rest of the (static) grid returns at once.  The
  // partial sums that cross vocab chunks are laid out by the same numbering (the count does not change between chunks).
  const int tiles_m = (M + BM - 1) / BM;
  const int tiles_n = (N + BN - 1) / BN;
  const int tiles = tiles_m * tiles_n;
  if (bid >= tiles * splits) return;
  int tm, tn, k0 = 0, k_back = p.k_back, split = 0;
  int logical = xcd_contiguous(bid, tiles * splits);
  if (splits > 1) {  // split by split, so that the workgroups resident on an XCD read the same range of both operands
    split = logical / tiles;
    logical -= split * tiles;
    const int pairs = nk / 2, p0 = pairs * split / splits, p1 = pairs * (split + 1) / splits;
    k0 = __builtin_amdgcn_readfirstlane(2 * p0), nk = __builtin_amdgcn_readfirstlane(2 * (p1 - p0));
    if (split != splits - 1) k_back = 0;
    if (nk == 0 && !p.p_first) return;  // a narrow last chunk: this split adds nothing to its slab
  }
  banded_tile(logical, tiles_m, tiles_n, kGroupM, tm, tn);
  gemm_tile_at<BKM>(p, M, N, tm, tn, k0, nk, k_back, (size_t)(split * tiles + tm * tiles_n + tn), !p.p_last || splits > 1, lds);
}

template <bool BKM>
__device__ __forceinline__ void gemm_tile_at(const GemmArgs& p, int M, int N, int tm, int tn, int k0, int nk, int k_back, size_t slot, bool partial, char* lds) {
#if LMHEAD_ABLATE & 16
  Operand a{p.A, p.lda, (tm % 4) * BM, p.a_rows};
  Operand b{p.B, p.ldb, (tn % 8) * BN, p.b_rows};
#else
  Operand a{p.A, p.lda, tm * BM, p.a_rows};
  Operand b{p.B, p.ldb, tn * BN, p.b_rows, 0, k_back};
#endif
  acc_t acc;
  if (nk > 0) prefetch_first_tiles<BKM>(a, b, k0 * BK, nk, lds);
  zero_acc(acc);
  if (nk > 0) {
    mainloop<BKM, true>(a, b, k0 * BK, nk, lds, acc);  // nk is even for every gradient GEMM (make_gemm checks)
  }

  const float* __restrict__ Cin = p.Cin;
  float* __restrict__ Cf = p.Cf;
  uint16_t* __restrict__ Cb = p.Cb;
  const int ldc = p.ldc;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int wm = wave / WAVES_N, wn = wave % WAVES_N;
  const int lrow = lane & 15, kq = lane >> 4;

  if (p.P) {
    float* part = p.P + (slot * NWAVES + wave) * kSlabWaveFloats + (size_t)lane * 4;
    if (!p.p_first) {  // sixteen loads in flight at a time: one at a time costs a round trip to HBM each (36 us per tile)
#pragma unroll
      for (int i = 0; i < TM; i += 2) {
        f32x4 t[2 * TN];
#pragma unroll
        for (int x = 0; x < 2 * TN; ++x) t[x] = *(const f32x4*)(part + (size_t)(i * TN + x) * (64 * 4));
#pragma unroll
        for (int x = 0; x < 2 * TN; ++x) acc[i + x / TN][x % TN] += t[x];
      }
    }
    if (partial) {
#pragma unroll
      for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j) *(f32x4*)(part + (size_t)(i * TN + j) * (64 * 4)) = acc[i][j];
      return;
    }
  }

  if (Cb && !Cin && !Cf) {
    // bf16 rows leave through LDS: in the accumulator layout a store instruction writes 32 contiguous bytes of sixteen rows (c_rows_m:
    // two bytes per lane), staged it writes 256 of four: 1110 -> 1046 us for a whole training pass at T=611, H=1536, V=151936,
    // whose dW tiles have eight k-tiles each.  The mainloop has left LDS free and every wave uses a region of its
    // own, so no barrier is needed.  Staged rows run along M with c_rows_m (the tokens of dHidden), along N otherwise.
    constexpr int kRow = WM * 2 + 16;
    static_assert(WM == WN && NWAVES * WN * kRow <= LDS_BYTES, "output staging does not fit LDS");
    char* stage = lds + wave * (WN * kRow);
    const bool along_m = BKM && p.c_rows_m;
    if (along_m) {
#pragma unroll
      for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j) {
          const bf16x4 b4 = __builtin_convertvector(acc[i][j], bf16x4);
          const uint16_t* h4 = (const uint16_t*)&b4;
#pragma unroll
          for (int r = 0; r < 4; ++r) *(uint16_t*)(stage + (i * MT + kq * 4 + r) * kRow + (j * MT + lrow) * 2) = h4[r];
        }
    } else {
#pragma unroll
      for (int j = 0; j < TN; ++j)
#pragma unroll
        for (int i = 0; i < TM; ++i) {
          const bf16x4 b4 = __builtin_convertvector(acc[i][j], bf16x4);
          *(uint2*)(stage + (j * MT + lrow) * kRow + (i * MT + kq * 4) * 2) = *(const uint2*)&b4;
        }
    }
    const int row0 = along_m ? tm * BM + wm * WM : tn * BN + wn * WN, rows = along_m ? M : N;
    const int col = (along_m ? tn * BN + wn * WN : tm * BM + wm * WM) + lrow * 8, cols = along_m ? N : M;
    if (col >= cols) return;  // whole 16-byte pieces: both extents that run along rows are multiples of 64
#pragma unroll
    for (int it = 0; it < WN / 4; ++it) {
      const u32x4 v = *(const u32x4*)(stage + (it * 4 + kq) * kRow + lrow * 16);
      int r = row0 + it * 4 + kq;
      if (r >= rows) continue;
      if (r >= p.n_tail) {
        r -= p.n_back;
        if (r < p.n_tail) continue;
      }
      if (p.row_map) r = p.row_map[r];
      *(u32x4*)(Cb + (size_t)r * (size_t)ldc + col) = v;
    }
    return;
  }

#pragma unroll
  for (int j = 0; j < TN; ++j) {
    int n = tn * BN + wn * WN + j * MT + lrow;
    if (n >= N) continue;
    if (n >= p.n_tail) {
      n -= p.n_back;
      if (n < p.n_tail) continue;
    }
#pragma unroll
    for (int i = 0; i < TM; ++i) {
      const int m = tm * BM + wm * WM + i * MT + kq * 4;  // this lane holds m .. m+3
      if (m < M) {
        const size_t idx = (size_t)n * (size_t)ldc + m;
        f32x4 v = acc[i][j];
        if (Cin) v += *(const f32x4*)(Cin + idx);
        if (Cf) *(f32x4*)(Cf + idx) = v;
        if (Cb) {
          const bf16x4 b4 = __builtin_convertvector(v, bf16x4);
          *(uint2*)(Cb + idx) = *(const uint2*)&b4;
        }
      }
    }
  }
}

// The two kinds of backward launch per vocab chunk, as kernels of their own so that a kernel trace tells them apart:
// the dz tiles of the chunk, then its two gradient GEMMs in one launch (workgroups [0, tiles0) work on p0, the rest on p1).
template <bool ENTGRAD, bool EVEN, bool SHAPES>
__global__ __launch_bounds__(NTHREADS) void lmhead_bwd_dz(const DzArgs z) {
  __shared__ __attribute__((aligned(1024))) char lds[LDS_BYTES];
  dz_square_tile<ENTGRAD, EVEN, SHAPES>(z, blockIdx.x, lds);
}

__global__ __launch_bounds__(NTHREADS) void lmhead_bwd_gemm(const GemmArgs p0, const GemmArgs p1, int tiles0) {
  __shared__ __attribute__((aligned(1024))) char lds[LDS_BYTES];
  const int id = blockIdx.x;
  // With a device-side token count the dW tiles start right behind the dHidden tiles in force; what is left of the (static) grid
  // returns at once.
  if (p0.T_dev) {
    const int count = __builtin_amdgcn_readfirstlane(*p0.T_dev);
    const int other = p0.t_role == kTokensOnM ? p0.N : p0.M;
    tiles0 = (count + BM - 1) / BM * ((other + BN - 1) / BN) *
             (p0.splits_dev ? __builtin_amdgcn_readfirstlane(*p0.splits_dev) : p0.splits);
  }
  // dW always reads the dz panel K-major (K = tokens); dHidden either reads the weight itself K-major (K = vocab) or,
  // for a small vocabulary that is not a multiple of two k-tiles, a transposed, zero-padded copy of it with K contiguous.
  const bool second = id >= tiles0;
  if (second || p0.b_kmajor) gemm_tile<true>(second ? p1 : p0, second ? id - tiles0 : id, lds);
  else gemm_tile<false>(p0, id, lds);
}

// dHidden alone (a frozen weight, the draft loss, a dW launch of its own): its tiles in equal shares (Shares; B K-major, tokens along M).
__global__ __launch_bounds__(NTHREADS) void lmhead_bwd_dh_shares(const GemmArgs p) {
  __shared__ __attribute__((aligned(1024))) char lds[LDS_BYTES];
  const int M = p.T_dev ? __builtin_amdgcn_readfirstlane(*p.T_dev) : p.M;
  const int tiles_m = (M + BM - 1) / BM, tiles_n = (p.N + BN - 1) / BN, tiles = tiles_m * tiles_n;
  Shares s = shares_of(p.splits_dev ? __builtin_amdgcn_readfirstlane(*p.splits_dev) : p.splits, tiles);
  s.groups = __builtin_amdgcn_readfirstlane(s.groups);
  if ((int)blockIdx.x >= s.workgroups()) return;
  const int id = xcd_contiguous(blockIdx.x, s.workgroups());
  // All of this in scalar registers: the mainloop leaves no vector register to hold it.
  const int j = __builtin_amdgcn_readfirstlane(id / s.groups), g = id - j * s.groups;
  int bg = 1, first = 0, last = 0;
  if (s.b > 1) {  // splits need none of these divisions, and calls of few tokens would notice them
    bg = __builtin_amdgcn_readfirstlane(s.tiles_of(g, tiles));
    first = __builtin_amdgcn_readfirstlane(s.first_tile(j, bg)), last = __builtin_amdgcn_readfirstlane(s.last_tile(j, bg));
  }
  const int pairs = p.nk / 2;
  const int from = __builtin_amdgcn_readfirstlane(s.begin(j, bg, pairs)), to = __builtin_amdgcn_readfirstlane(s.begin(j + 1, bg, pairs));
  for (int i = first; i <= last; ++i) {
    const int k0 = from > i * pairs ? from - i * pairs : 0, k1 = to < (i + 1) * pairs ? to - i * pairs : pairs;
    const int nk = 2 * (k1 - k0);
    if (nk == 0 && !p.p_first) continue;  // a narrow last chunk: nothing to add to this slab
    if (i > first) __syncthreads();  // every wave has taken its rows of the tile before from LDS
    int tm, tn;
    banded_tile(i * s.groups + g, tiles_m, tiles_n, kGroupM, tm, tn);
    bool alone = s.u == 1;
    if (s.b > 1) alone = __builtin_amdgcn_readfirstlane(s.first_workgroup(i, bg)) == __builtin_amdgcn_readfirstlane(s.last_workgroup(i, bg));
    // The lanes' copy offsets and LDS addresses formed once for all tiles would be vector registers that the mainloop does not have.
    GemmArgs q = p;
    int lds_at = 0;
    asm volatile("" : "+s"(q.lda), "+s"(q.ldb), "+s"(q.ldc), "+s"(lds_at));
    gemm_tile_at<true>(q, M, p.N, tm, tn, 2 * k0, nk, k1 == pairs ? p.k_back : 0, (size_t)(s.b > 1 ? s.slot(g, i, j) : j * tiles + tm * tiles_n + tn), !p.p_last || !alone, lds + lds_at);
  }
}

// dHidden rows from the slabs of a split contraction: C[m, n] = bf16(sum of the slabs), added in split order.  One workgroup per
// 16 tokens x 128 columns (an MFMA row block of a wave): 16-byte loads of contiguous slab pieces, 16-byte row pieces out
// through LDS.  HBM-bound, splits x tokens x H x 4 bytes: 8 us at 240 slab tiles (60 MB).  SHARES: of a launch that may have been cut in shares; the
// code for these costs calls of few tokens, which bring it from memory each time: 6.9 -> 8.4 us at 20 tokens, H=1536, 10.0 -> 12.1 at 300, H=512,
// 8.6 -> 11.4 in the draft loss of 20 tokens, H=896, V=246016.
struct DhReduceArgs {
  const float* P;
  int M, H, splits;
  const int *T_dev, *splits_dev, *row_map;  // as in GemmArgs
  uint16_t* C;
  int ldc;
};
constexpr int kReduceGroups = NWAVES * TM;  // workgroups per tile

template <bool SHARES>
__global__ __launch_bounds__(256) void lmhead_dh_reduce(const DhReduceArgs a) {
  __shared__ __attribute__((aligned(16))) uint16_t rows[MT][WN + 8];
  const int splits = a.splits_dev ? *a.splits_dev : a.splits;
  const int M = a.T_dev ? *a.T_dev : a.M;
  const int tiles_m = (M + BM - 1) / BM, tiles_n = (a.H + BN - 1) / BN, tiles = tiles_m * tiles_n;
  const int tile = blockIdx.x / kReduceGroups, wave = blockIdx.x / TM % NWAVES, i = blockIdx.x % TM;
  if (splits < 2 || tile >= tiles) return;  // without splits the GEMM epilogue has written C
  // Splits: the slabs of a tile stand `tiles` apart, in row order; shares: `groups` apart, in the launch's order.
  int tm = tile / tiles_n, tn = tile % tiles_n, count = splits, step = tiles, slot = tile;
  if (SHARES && splits >= 256) {
    const Shares sh = shares_of(splits, tiles);
    const int in_group = tile / sh.groups, g = tile - in_group * sh.groups, bg = sh.tiles_of(g, tiles), first = sh.first_workgroup(in_group, bg);
    count = __builtin_amdgcn_readfirstlane(sh.last_workgroup(in_group, bg) - first + 1), step = __builtin_amdgcn_readfirstlane(sh.groups);
    slot = __builtin_amdgcn_readfirstlane(sh.slot(g, in_group, first));
    if (count < 2) return;  // one workgroup made the tile, and its epilogue has written C
    banded_tile(tile, tiles_m, tiles_n, kGroupM, tm, tn);
  }
  const int m0 = tm * BM + wave / WAVES_N * WM + i * MT;
  const int n0 = tn * BN + wave % WAVES_N * WN;
  if (m0 >= M || n0 >= a.H) return;
  const int tid = threadIdx.x;
  const float* part = a.P + ((size_t)slot * NWAVES + wave) * kSlabWaveFloats + (size_t)(i * TN) * (64 * 4) + (size_t)tid * 4;
  const size_t slab = (size_t)step * kSlabTileFloats;
  f32x4 sum[2] = {*(const f32x4*)part, *(const f32x4*)(part + 1024)};
#pragma unroll 4
  for (int s = 1; s < count; ++s) {
    sum[0] += *(const f32x4*)(part + (size_t)s * slab);
    sum[1] += *(const f32x4*)(part + (size_t)s * slab + 1024);
  }
  const int lane = tid & 63, lrow = lane & 15, kq = lane >> 4;
#pragma unroll
  for (int u = 0; u < 2; ++u) {
    const bf16x4 b4 = __builtin_convertvector(sum[u], bf16x4);
    const uint16_t* h4 = (const uint16_t*)&b4;
#pragma unroll
    for (int r = 0; r < 4; ++r) rows[kq * 4 + r][(u * 4 + (tid >> 6)) * MT + lrow] = h4[r];
  }
  __syncthreads();
  const int r = tid >> 4, c = (tid & 15) * 8, m = m0 + r;
  if (m < M && n0 + c < a.H)
    *(uint4*)(a.C + (size_t)(a.row_map ? a.row_map[m] : m) * (size_t)a.ldc + n0 + c) = *(const uint4*)&rows[r][c];
}

// Measurement aid: the mainloop's MFMA sequence (two 32-k steps of 64 MFMAs, same order, accumulators in AGPRs) with
// register-resident operands and nothing else in the loop -- what the matrix pipe sustains on a given kind of data.
__global__ __launch_bounds__(NTHREADS) void mfma_probe(const bf16x8* __restrict__ operands, int iters, float* __restrict__ sink) {
  bf16x8 af[2][TM], bfr[2][TN];
#pragma unroll
  for (int s = 0; s < 2; ++s)
#pragma unroll
    for (int i = 0; i < TM; ++i) {
      af[s][i] = operands[((s * TM + i) * 2 + 0) * NTHREADS + threadIdx.x];
      bfr[s][i] = operands[((s * TM + i) * 2 + 1) * NTHREADS + threadIdx.x];
    }
  acc_t acc;
  zero_acc(acc);
  for (int it = 0; it < iters; ++it) {
#pragma unroll
    for (int ks = 0; ks < KSTEPS; ++ks)
#pragma unroll
      for (int x = 0; x < TM * TN; ++x) {
        const int i = mfma_row<>(x), j = mfma_col<>(x);
        mfma_16x16x32(acc[i][j], af[ks][i], bfr[ks][j]);
      }
  }
  asm volatile("s_nop 15\n\ts_nop 15" ::: "memory");
  float sum = 0.f;
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j) {
      asm volatile("" : "+a"(acc[i][j]));
      sum += acc[i][j][0] + acc[i][j][1] + acc[i][j][2] + acc[i][j][3];
    }
  sink[blockIdx.x * NTHREADS + threadIdx.x] = sum;
}

// Measurement aid: the fp32 atomic traffic of a fully fused backward (efficient_entropy_backward_kernel_general_mainloop_MN,
// fused_linear_logprob_triton.py:807-996) and nothing else.  Such a kernel forms the dz tile of 256 vocab rows x 256 tokens and
// has to add its contribution to dW[256, H] and to dHidden[256, H] in memory, because no workgroup can hold a [256, H]
// accumulator.  One workgroup per (vocab tile, token tile) issues exactly those adds -- in the accumulator layout, a lane's
// four values contiguous -- with no logits recompute and no MFMA: a lower bound of what the fused variant costs.
__global__ __launch_bounds__(NTHREADS) void atomic_floor_probe(float* __restrict__ dW, float* __restrict__ dH, int tiles_v, int H) {
  const int tv = blockIdx.x % tiles_v, tt = blockIdx.x / tiles_v;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int wm = wave / WAVES_N, wn = wave % WAVES_N, lrow = lane & 15, kq = lane >> 4;
  for (int c0 = 0; c0 < H; c0 += BN) {
#pragma unroll
    for (int half = 0; half < 2; ++half) {
      float* dst = half ? dH + (size_t)tt * BM * (size_t)H : dW + (size_t)tv * BM * (size_t)H;
#pragma unroll 4
      for (int x = 0; x < TM * TN; ++x) {
        const int i = x / TN, j = x % TN;
        const int n = c0 + wn * WN + j * MT + lrow;          // column of the [256, H] slice
        if (n >= H) continue;
        const int m = wm * WM + i * MT + kq * 4;             // this lane adds rows m .. m+3
#pragma unroll
        for (int r = 0; r < 4; ++r) atomicAdd(dst + (size_t)(m + r) * (size_t)H + n, 1.0f);
      }
    }
  }
}

// dst[c, r] = src[r, c] for r < R, c < C;  dst[c, r] = 0 for R <= r < Rpad.  bf16 bits, 64 x 64 tiles.
// R_dev (may be NULL): the number of valid source rows as a value in device memory, <= R.
__global__ __launch_bounds__(256) void transpose_bf16(const uint16_t* __restrict__ src, int lds_src, int R, int C,
                                                      uint16_t* __restrict__ dst, int ld_dst, int Rpad,
                                                      const int* __restrict__ R_dev) {
  __shared__ uint16_t tile[64][66];
  if (R_dev) R = *R_dev;
  const int r0 = blockIdx.x * 64, c0 = blockIdx.y * 64;
  const int tid = threadIdx.x;
#pragma unroll
  for (int it = 0; it < 2; ++it) {
    const int idx = it * 256 + tid;  // 512 chunks of 8 elements
    const int rr = idx >> 3, cc = (idx & 7) * 8;
    const int r = r0 + rr, c = c0 + cc;
    uint16_t v[8] = {0, 0, 0, 0, 0, 0, 0, 0};
    if (r < R) {
      if (c + 8 <= C) {
        const uint4 q = *(const uint4*)(src + (size_t)r * (size_t)lds_src + c);
        const uint32_t w[4] = {q.x, q.y, q.z, q.w};
#pragma unroll
        for (int k = 0; k < 4; ++k) {
          v[2 * k] = (uint16_t)(w[k] & 0xffffu);
          v[2 * k + 1] = (uint16_t)(w[k] >> 16);
        }
      } else {
        for (int k = 0; k < 8; ++k)
          if (c + k < C) v[k] = src[(size_t)r * (size_t)lds_src + c + k];
      }
    }
#pragma unroll
    for (int k = 0; k < 8; ++k) tile[rr][cc + k] = v[k];
  }
  __syncthreads();
#pragma unroll
  for (int it = 0; it < 2; ++it) {
    const int idx = it * 256 + tid;
    const int cc = idx >> 3, rr = (idx & 7) * 8;  // output row = source column
    const int c = c0 + cc, r = r0 + rr;
    if (c < C && r < Rpad) {
      uint32_t w[4];
#pragma unroll
      for (int k = 0; k < 4; ++k) w[k] = (uint32_t)tile[rr + 2 * k][cc] | ((uint32_t)tile[rr + 2 * k + 1][cc] << 16);
      *(uint4*)(dst + (size_t)c * (size_t)ld_dst + r) = make_uint4(w[0], w[1], w[2], w[3]);
    }
  }
}

// ------------------------------------------------------------------------------------------------------------
// fp32 operands on the bf16 matrix pipe.  An fp32 value is the sum of bf16 terms, x = hi + lo (+ 2^-17 |x|), hi = bf16(x),
// lo = bf16(x - hi), and a product of sums is a sum of products: stacking the terms along the contraction axis,
//     weight fp32, hidden bf16:   [w_hi | w_lo] . [h | h]^T           = h . (w_hi + w_lo)
//     weight fp32, hidden fp32:   [w_hi | w_lo | w_hi] . [h_hi | h_hi | h_lo]^T = h_hi . w_hi + h_hi . w_lo + h_lo . w_hi
// turns the fp32 logits GEMM (model_utils.py:328-333: hidden is cast to the weight's dtype, the product is fp32) into the
// ordinary bf16 GEMM with two or three times the contraction length; the MFMA accumulates all terms in fp32.  What is dropped
// is below 2^-16 of each product.  This kernel writes one stacked operand: segment s of row r holds the hi (code 0) or lo
// (code 1) terms of the row.
// ------------------------------------------------------------------------------------------------------------
__device__ __forceinline__ uint16_t bf16_rne(float x) {
  const uint32_t u = __float_as_uint(x);
  if ((u & 0x7fffffffu) > 0x7f800000u) return (uint16_t)((u >> 16) | 0x40u);  // NaN stays NaN
  return (uint16_t)((u + 0x7fffu + ((u >> 16) & 1u)) >> 16);
}

template <bool SRC_FP32>
__global__ __launch_bounds__(256) void split_operand_rows(const void* __restrict__ src, int64_t ld_src, int H, int terms, int code0,
                                                          int code1, int code2, uint16_t* __restrict__ dst, int64_t ld_dst) {
  const int64_t r = blockIdx.x;
  const int codes[3] = {code0, code1, code2};
  for (int c = threadIdx.x * 4; c < H; c += 256 * 4) {
    uint16_t hi[4], lo[4];
    if (SRC_FP32) {
      const float4 v = *(const float4*)((const float*)src + r * ld_src + c);
      const float x[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        hi[k] = bf16_rne(x[k]);
        lo[k] = bf16_rne(x[k] - __uint_as_float((uint32_t)hi[k] << 16));
      }
    } else {
      const uint2 v = *(const uint2*)((const uint16_t*)src + r * ld_src + c);
      hi[0] = (uint16_t)(v.x & 0xffffu), hi[1] = (uint16_t)(v.x >> 16), hi[2] = (uint16_t)(v.y & 0xffffu), hi[3] = (uint16_t)(v.y >> 16);
      lo[0] = lo[1] = lo[2] = lo[3] = 0;
    }
    for (int s = 0; s < terms; ++s) {
      const uint16_t* t = codes[s] ? lo : hi;
      *(uint2*)(dst + r * ld_dst + (int64_t)s * H + c) =
          make_uint2((uint32_t)t[0] | ((uint32_t)t[1] << 16), (uint32_t)t[2] | ((uint32_t)t[3] << 16));
    }
  }
}

// ------------------------------------------------------------------------------------------------------------
// Row compaction for the backward.  A token whose upstream gradients are both zero has a zero dz row: it adds nothing to
// dW and its dHidden row is zero.  In RL micro-batches those are the prompt and padding tokens the loss mask removes, often
// more than half of the batch.  Two small kernels let the backward run on the remaining rows without the host ever
// learning how many there are (no synchronisation, so the call can be captured in a HIP graph):
//   compact_active_rows   one workgroup: idx[i] = i-th token with g != 0 or q != 0 (ascending), counts[0] = their number n,
//                         counts[1 + b] = how many of them fall into block b of `block` compacted rows,
//                         counts[1 + nblocks + b] = how that block's dHidden contraction is cut: the number of splits, or, where
//                         SplitProblem::shares admits it, a code of Shares, which only lmhead_bwd_dh_shares and lmhead_dh_reduce read
//   gather_active_rows    compacted copies of hidden rows and of the per-token inputs; zero dHidden rows for the inactive
// The GEMM kernels take the counts from device memory (T_dev), run on the static upper-bound grid and write the dHidden rows
// through the index list.
// ------------------------------------------------------------------------------------------------------------
constexpr int kCompactThreads = 1024;

template <int TOKENS>  // per thread and step
__global__ __launch_bounds__(kCompactThreads) void compact_active_rows(const float* __restrict__ g, const float* __restrict__ q,
                                                                       int T, int block, int nblocks, SplitProblem split,
                                                                       int* __restrict__ idx, int* __restrict__ counts) {
  // A step takes four tokens per thread: their loads travel together, and every wave scans the 64 counts of the step by itself, so that one
  // barrier stands between the counts and the list.  What bounds it is that chain: with a token per thread and the counts added up by one thread
  // 12.1 -> 7.7 us at T=8192, 6.7 -> 5.4 at 4096, 6.6 -> 5.2 at 2100.  Up to 1024 tokens, where it is the code that has to be fetched first, a
  // token per thread: 4.1 -> 3.6 us at T=137, 4.3 -> 3.7 at 300.
  constexpr int kCounts = TOKENS * kCompactThreads / 64;
  static_assert(kCounts <= 64, "one lane per count");
  __shared__ int count[2][kCounts];  // of tokens t0 + k * kCompactThreads + wave * 64 .. + 63: k * 16 + wave; steps take turns
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  int n = 0;
  for (int t0 = 0, turn = 0; t0 < T; t0 += TOKENS * kCompactThreads, turn ^= 1) {
    unsigned long long ballot[TOKENS];
#pragma unroll
    for (int k = 0; k < TOKENS; ++k) {
      const int t = t0 + k * kCompactThreads + tid;
      const int tc = t < T ? t : T - 1;
      const float gv = g[tc], qv = q ? q[tc] : 0.f;
      ballot[k] = __ballot(t < T && (gv != 0.f || qv != 0.f));
    }
#pragma unroll
    for (int k = 0; k < TOKENS; ++k)
      if (lane == 0) count[turn][k * (kCompactThreads / 64) + wave] = __popcll(ballot[k]);
    __syncthreads();
    const int mine = lane < kCounts ? count[turn][lane] : 0;
    int upto = mine;
#pragma unroll
    for (int o = 1; o < kCounts; o <<= 1) {
      const int below = __shfl_up(upto, o, 64);
      upto += lane >= o ? below : 0;
    }
#pragma unroll
    for (int k = 0; k < TOKENS; ++k) {
      const int base = n + __shfl(upto - mine, k * (kCompactThreads / 64) + wave, 64);
      if (ballot[k] >> lane & 1) idx[base + __popcll(ballot[k] & ((1ull << lane) - 1ull))] = t0 + k * kCompactThreads + tid;
    }
    n += __shfl(upto, kCounts - 1, 64);
  }
  for (int b = tid; b <= nblocks; b += kCompactThreads) {
    if (b == 0) {
      counts[0] = n;
    } else {
      const long long left = (long long)n - (long long)(b - 1) * block;
      counts[b] = left < 0 ? 0 : (left > block ? block : (int)left);
    }
  }
  for (int b = wave; b < nblocks; b += kCompactThreads / 64) {  // lane l rates l + 1 splits and groups of l + 2 tiles; the cheapest, of equals the fewest, wins
    const long long left = (long long)n - (long long)b * block;
    const int tokens = left < 0 ? 0 : (left > block ? block : (int)left);
    long long best = split_cost(split, tokens, lane + 1);
    int splits = lane + 1;
    if (split.shares) {
      int code = 0;
      const long long shared = lane < kMaxGroup - 1 ? share_cost(split, tokens, lane + 2, code) : INT64_MAX;
      if (shared < best) best = shared, splits = code;
    }
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) {
      const long long c = __shfl_xor(best, o, 64);
      const int k = __shfl_xor(splits, o, 64);
      if (c < best || (c == best && k < splits)) best = c, splits = k;
    }
    if (lane == 0) counts[1 + nblocks + b] = splits;
  }
}

inline auto compact_kernel(int64_t T) { return T <= kCompactThreads ? compact_active_rows<1> : compact_active_rows<4>; }

// One workgroup per row r < T: as compacted row r (when r < n) it copies the inputs of token idx[r]; as token r it clears
// d_hidden[r] -- active tokens get their row from the dHidden GEMM (or the sum over its splits) afterwards.
__global__ __launch_bounds__(256) void gather_active_rows(const int* __restrict__ idx, const int* __restrict__ counts,
                                                          const uint16_t* __restrict__ hidden, int ldh, int Hk, int H,
                                                          const int64_t* __restrict__ labels, const float* __restrict__ lse,
                                                          const float* __restrict__ pz, const float* __restrict__ g,
                                                          const float* __restrict__ q, uint16_t* __restrict__ hidden_c,
                                                          int64_t* __restrict__ labels_c, float* __restrict__ lse_c,
                                                          float* __restrict__ pz_c, float* __restrict__ g_c,
                                                          float* __restrict__ q_c, uint16_t* __restrict__ d_hidden) {
  const int r = blockIdx.x;
  uint16_t* zero_row = d_hidden + (size_t)r * (size_t)H;
  for (int c = threadIdx.x * 8; c < H; c += 256 * 8) *(uint4*)(zero_row + c) = make_uint4(0, 0, 0, 0);
  if (r >= counts[0]) return;
  const int t = idx[r];
  const uint16_t* src = hidden + (size_t)t * (size_t)ldh;
  uint16_t* dst = hidden_c + (size_t)r * (size_t)Hk;
  for (int c = threadIdx.x * 8; c < Hk; c += 256 * 8) *(uint4*)(dst + c) = *(const uint4*)(src + c);
  if (threadIdx.x == 0) {
    labels_c[r] = labels[t];
    lse_c[r] = lse[t];
    g_c[r] = g[t];
    if (q) q_c[r] = q[t], pz_c[r] = pz[t];
  }
}

// What the bf16 product dropped of the label's dz value d (see DzArgs::label_resid), added to the weight gradient in fp32:
//     dW[label_t, :] += (d - bf16(d)) * h_hi[t, :]  +  d * h_lo[t, :]
// h_lo is the third segment of a stacked fp32 hidden row (lo_offset = 2 * H) and absent (lo_offset = 0) for a bf16 hidden.
// One workgroup per token; fp32 atomic adds, because several tokens may share a label (their order, and with it the last
// bit of those rows, is not fixed).
__global__ __launch_bounds__(256) void label_residual_update(const float* __restrict__ label_dz, const int64_t* __restrict__ labels,
                                                             const uint16_t* __restrict__ hidden, int ldh, int H, int lo_offset,
                                                             int V, const int* __restrict__ T_dev, float* __restrict__ dW) {
  const int t = blockIdx.x;
  if (T_dev && t >= *T_dev) return;
  const float d = label_dz[t];
  const int64_t y = labels[t];
  if (d == 0.f || y < 0 || y >= (int64_t)V) return;
  const float r = d - __uint_as_float((uint32_t)bf16_rne(d) << 16);
  const uint16_t* hp = hidden + (size_t)t * (size_t)ldh;
  float* wp = dW + (size_t)y * (size_t)H;
  for (int c = threadIdx.x; c < H; c += 256) {
    float add = r * __uint_as_float((uint32_t)hp[c] << 16);
    if (lo_offset) add = fmaf(d, __uint_as_float((uint32_t)hp[lo_offset + c] << 16), add);
    atomicAdd(wp + c, add);
  }
}

__global__ __launch_bounds__(256) void zero_f32(float* __restrict__ p, int n) {
  const int i = blockIdx.x * 256 + threadIdx.x;
  if (i < n) p[i] = 0.f;
}

// ------------------------------------------------------------------------------------------------------------
// Host side
// ------------------------------------------------------------------------------------------------------------
// Optional per-kernel timing: while a profile is open on the calling thread every launch below is bracketed by a pair of
// HIP events on the launch stream.  Closed profiles cost one thread-local load per launch.
// A kind is a task: lmhead_bwd_gemm the gradient products of a chunk, in the kernel of that name or in lmhead_bwd_dh_shares; lmhead_bwd_dw_few dW of few
// tokens, in tiles or with resident dz.
enum KernelKind {
  kFwdTiles = 0, kFwdMerge, kTranspose, kBwdChunkDz, kBwdChunkGemm, kSoftCePack, kSoftCeFwdTiles, kSoftCeFinish, kSoftCeDz,
  kCompactRows, kSplitOperand, kTopkFilter, kTopkSelect, kTopkRows, kTopkBwdRows, kDhReduce, kBwdDwFew,
  kNumKernelKinds
};
const char* const kKernelNames[kNumKernelKinds] = {"lmhead_fwd_tiles", "lmhead_fwd_merge", "transpose_bf16",
                                                   "lmhead_bwd_dz", "lmhead_bwd_gemm", "softce_pack_rows",
                                                   "softce_fwd_tiles", "softce_finish", "softce_dz_tiles",
                                                   "active_rows[compact+gather]", "split_operand_rows",
                                                   "topk_filter_tiles", "topk_select", "topk_softce_rows",
                                                   "topk_softce_bwd_rows", "lmhead_dh_reduce", "lmhead_bwd_dw_few"};
struct Profile {
  struct Rec {
    int kind;
    hipEvent_t a, b;
  };
  std::vector<Rec> recs;
};
thread_local Profile* tl_profile = nullptr;

struct Timed {
  int kind;
  hipStream_t s;
  hipEvent_t a = nullptr, b = nullptr;
  Timed(int k, hipStream_t st) : kind(k), s(st) {
    if (tl_profile && hipEventCreate(&a) == hipSuccess && hipEventCreate(&b) == hipSuccess) (void)hipEventRecord(a, s);
  }
  ~Timed() {
    if (tl_profile && a && b) {
      (void)hipEventRecord(b, s);
      tl_profile->recs.push_back({kind, a, b});
    }
  }
};

struct Carver {
  char* base;
  size_t off = 0;
  explicit Carver(void* p) : base((char*)p) {}
  template <typename T>
  T* take(size_t count) {
    off = (size_t)round_up((int64_t)off, 256);
    T* p = base ? (T*)(base + off) : nullptr;
    off += count * sizeof(T);
    return p;
  }
};

inline bool aligned16(const void* p) { return ((uintptr_t)p & 15u) == 0; }

// Largest T, H or V any entry point accepts (row pitches are limited to kMaxRowPitch, far below it); the workspace queries
// answer 0 beyond it instead of computing with sizes that no call would accept.
constexpr int64_t kMaxExtent = (int64_t)1 << 30;

// The two bf16 operands of every entry point: hidden rows [T, H] and weight rows [V, H].
// Matrices may be of any size: the copy plan addresses a tile with 32-bit offsets from the tile's own first row, so only
// the row pitch is limited (256 rows must span less than 4 GiB: kMaxRowPitch elements).
int check_operands(const void* hidden, int64_t ldh, const void* weight, int64_t ldw, int64_t T, int64_t H, int64_t V,
                   float rcp_temperature, bool hidden_in_blocks = false) {
  if (!hidden || !weight) return SKYRL_LMHEAD_ERR_NULL;
  if (T < 1 || V < 1 || H < BK || H % BK != 0 || ldh < H || ldw < H) return SKYRL_LMHEAD_ERR_SHAPE;
  if (T > kMaxExtent || V > kMaxExtent) return SKYRL_LMHEAD_ERR_SHAPE;
  (void)hidden_in_blocks;
  if (ldh > kMaxRowPitch || ldw > kMaxRowPitch) return SKYRL_LMHEAD_ERR_SHAPE;
  if (!aligned16(hidden) || !aligned16(weight) || ldh % 8 != 0 || ldw % 8 != 0) return SKYRL_LMHEAD_ERR_ALIGN;
  if (!(rcp_temperature > 0.f) || !isfinite(rcp_temperature)) return SKYRL_LMHEAD_ERR_ARG;
  return SKYRL_LMHEAD_OK;
}

int check_common(const void* hidden, int64_t ldh, const void* weight, int64_t ldw, const int64_t* labels, int64_t T,
                 int64_t H, int64_t V, float rcp_temperature, bool hidden_in_blocks = false) {
  if (!hidden || !weight || !labels) return SKYRL_LMHEAD_ERR_NULL;
  const int st = check_operands(hidden, ldh, weight, ldw, T, H, V, rcp_temperature, hidden_in_blocks);
  if (st == SKYRL_LMHEAD_ERR_SHAPE) return st;  // shape errors are reported before alignment errors, labels included
  if ((uintptr_t)labels & 7u) return SKYRL_LMHEAD_ERR_ALIGN;
  return st;
}

// Compute units of the current device (256 on an MI355X); 256 when no device answers, so that the workspace query gives
// the same figure on a machine without a GPU.
int compute_units() {
  int dev = 0, n = 0;
  if (hipGetDevice(&dev) != hipSuccess || hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess ||
      n < 1) {
    (void)hipGetLastError();
    return 256;
  }
  return n;
}

// Estimated duration, in k-tiles of mainloop per CU, of `count_a` tiles of length `len_a` followed by `count_b` tiles of
// length `len_b` handed to `ncu` CUs in order, each CU taking the next tile when it is free (what the dispatcher does with
// one workgroup per CU).  Closed form: the first kind fills whole rounds plus one partial round; the second kind then
// runs back to back on CUs that became free at one of two times, so the end is the smallest time by which those CUs can
// have completed count_b tiles.
int64_t list_schedule(int64_t count_a, int64_t len_a, int64_t count_b, int64_t len_b, int64_t ncu) {
  const int64_t rounds = count_a / ncu, late = count_a % ncu, early = ncu - late;
  const int64_t t_early = rounds * len_a, t_late = late ? (rounds + 1) * len_a : t_early;
  if (count_b == 0) return t_late;
  auto done_by = [&](int64_t t) {
    return early * (t > t_early ? (t - t_early) / len_b : 0) + late * (t > t_late ? (t - t_late) / len_b : 0);
  };
  // the end is t_early + m * len_b or t_late + m * len_b for some m >= 1: take the smallest that suffices
  int64_t best = -1;
  for (const int64_t t0 : {t_early, t_late}) {
    int64_t lo = 1, hi = count_b;  // m = count_b always suffices (one CU alone)
    while (lo < hi) {
      const int64_t mid = (lo + hi) / 2;
      if (done_by(t0 + mid * len_b) >= count_b) hi = mid; else lo = mid + 1;
    }
    const int64_t t = t0 + lo * len_b;
    if (best < 0 || t < best) best = t;
  }
  return best > t_late ? best : t_late;
}

// Width of the dz panel in vocab columns when the caller does not choose one.  Wider chunks mean fewer launches (every
// launch ends with CUs idling for part of a tile), fewer read-modify-write passes over the dHidden partial sums and a
// larger panel; what matters most is whether the tiles of a launch divide evenly over the CUs.  The candidates
// (multiples of 2048 columns whose panel holds at most 1.5 GiB of dz values) are rated with a small model of the two launches per
// chunk -- dz tiles of H/64 k-tiles plus an epilogue, then dHidden tiles of chunk/64 and dW tiles of T'/64 k-tiles,
// list-scheduled over the CUs, plus a fixed cost per launch -- and the cheapest wins.  At the 7B shape (T = 16384, H = 3584)
// that is 49152 columns: 4096 x 3 dz tiles and 896 + 2688 GEMM tiles per launch, both multiples of 256 CUs.
int64_t default_vocab_chunk(int64_t T, int64_t H, int64_t V) {
  const int64_t Tpad = round_up(T, 256), Vpad = round_up(V, 256), Hpad = round_up(H, 256);
  const int ncu = compute_units();
  const int64_t tiles_t = Tpad / 256, tiles_h = Hpad / 256;
  const int64_t kDzEpilogue = 8, kGemmEpilogue = 6, kLaunch = 24;  // in k-tiles (about 1.3 us each)
  const int64_t kMaxPanelBytes = (int64_t)3 << 29;  // of dz values, before the row padding
  // Few dHidden tiles: their contraction is split over the CUs (split_cost), whole rounds no longer depend on the width, and the
  // fewest chunks are the cheapest.
  if (tiles_h * tiles_t < kSplitBelowTiles) {
    const int64_t widest = kMaxPanelBytes / (Tpad * 2) / 2048 * 2048, chunks = (Vpad + widest - 1) / widest;
    return round_up((Vpad + chunks - 1) / chunks, 256);
  }
  int64_t best_vc = 0, best_cost = 0;
  for (int64_t vc = 2048;; vc += 2048) {
    if (vc > Vpad) vc = Vpad;
    const bool fits = Tpad * vc * 2 <= kMaxPanelBytes;
    if (fits || best_vc == 0) {
      auto chunk_cost = [&](int64_t w) {  // the two launches of a chunk of w columns
        return list_schedule(w / 256 * tiles_t, H / BK + kDzEpilogue, 0, 0, ncu) + kLaunch +
               list_schedule(tiles_h * tiles_t, w / BK + kGemmEpilogue, tiles_h * (w / 256), Tpad / BK + kGemmEpilogue, ncu) + kLaunch;
      };
      const int64_t full = Vpad / vc, rest = Vpad % vc;  // all chunks but the last have the same width
      const int64_t cost = full * chunk_cost(vc) + (rest ? chunk_cost(rest) : 0);
      if (best_vc == 0 || cost < best_cost) best_vc = vc, best_cost = cost;
    }
    if (vc >= Vpad || !fits) break;
  }
  return best_vc;
}

// Scratch that is `missing` bytes smaller than the query's.  A width of the library's own choice makes room first, in the dz panel of `rows`
// rows (2048 columns are the narrowest it chooses), because splits save more than wide chunks; then the slabs: `wanted` floats of them
// become what fits, but no fewer than the `least`, one per dHidden tile.  Backward with dW, V=151936, whole scratch / half of it, narrower
// chunks / whole chunk, one slab per tile: 868 / 968 / 3163 us at T=611, H=1536, 2229 / 2270 / 3544 at T=2048, 397 / 539 / 2697 at T=300, H=896.
int64_t fitting_chunk(int64_t vc, int64_t rows, int64_t V, size_t missing) {
  const int64_t Vpad = round_up(V, 256), least = Vpad < 2048 ? Vpad : 2048;
  const int64_t fits = (vc - (int64_t)(missing / (size_t)(2 * rows)) - 1) / 256 * 256;
  if (fits < least) return least;
  const int64_t chunks = (Vpad + fits - 1) / fits;
  return round_up((Vpad + chunks - 1) / chunks, 256);
}
int64_t fitting_slabs(int64_t wanted, int64_t least, size_t missing) {
  const int64_t fits = wanted - (int64_t)((missing + 255) / 256 * 64);
  return fits > least ? fits : least;
}

// Forward scratch: three arrays of per-part statistics for `tokens` tokens.
size_t fwd_partials_bytes(int64_t tokens, int64_t V) {
  const size_t nparts = (size_t)((V + BM - 1) / BM) * WAVES_M;
  Carver c(nullptr);
  c.take<float>(part_elems(nparts, tokens));
  c.take<float>(part_elems(nparts, tokens));
  c.take<float>(part_elems(nparts, tokens));
  return (size_t)round_up((int64_t)c.off, 256);
}

// The forward walks the tokens in blocks: tokens are independent, so a block is a complete forward problem on a slice of
// hidden / labels / outputs, and the partials of one block are merged before the next block overwrites them (launches on
// one stream run in order).  The scratch is therefore sized by the block, not by T.  Block boundaries are multiples of the
// 256-token tile, so every token sees the same tiles, in the same order, as in an unblocked run: results are bit-identical
// for any block size.
constexpr int64_t kFwdTokenBlock = 32768;


// Tokens per block: what the caller's scratch allows, at least one 256-token tile.
int64_t fwd_block_tokens(int64_t wanted, int64_t ld_hidden) {
  (void)ld_hidden;
  return wanted < BN ? BN : wanted;
}

int fwd_token_blocks(const void* hidden, int64_t ld_hidden, const void* weight, int64_t ld_weight, const int64_t* labels,
                     int64_t T, int64_t H, int64_t V, float rcp_temperature, float* logprobs, float* entropy, float* row_lse,
                     float* row_pz, void* scratch, int64_t block_tokens, hipStream_t s) {
  const int tiles_m = (int)((V + BM - 1) / BM);
  const size_t nparts = (size_t)tiles_m * WAVES_M;
  const bool want_pz = entropy || row_pz;
  const uint16_t* Wp = (const uint16_t*)weight;
  for (int64_t t0 = 0; t0 < T; t0 += block_tokens) {
    const int64_t Tb = (T - t0) < block_tokens ? (T - t0) : block_tokens;
    const bool half = half_tile_logits(Tb);
    const int tiles_n = (int)((Tb + BN - 1) / BN);
    Carver c(scratch);
    float* pmax = c.take<float>(part_elems(nparts, Tb));
    float* psum = c.take<float>(part_elems(nparts, Tb));
    float* ppz = c.take<float>(part_elems(nparts, Tb));
    const uint16_t* Hp = (const uint16_t*)hidden + (size_t)t0 * (size_t)ld_hidden;
    const TileShapes shapes = tile_shapes(Tb, H, tiles_m, compute_units());
    const dim3 grid((unsigned)(tiles_m * tiles_n + shapes.split)), block(NTHREADS);
    {
      Timed timed(kFwdTiles, s);
      auto kernel = flagged_kernel(
          [](auto pz, auto even, auto others) { return &lmhead_fwd_tiles<pz.value, even.value, others.value>; }, want_pz, even_ktiles(H),
          shapes.used);
      if (half)
        launch_fwd_half_tiles(s, want_pz, Wp, (int)ld_weight, Hp, (int)ld_hidden, (int)Tb, (int)H, (int)V, rcp_temperature, pmax, psum, ppz);
      else
        hipLaunchKernelGGL(kernel, grid, block, 0, s, Wp, (int)ld_weight, Hp, (int)ld_hidden, (int)Tb, (int)H, (int)V,
                         rcp_temperature, pmax, psum, ppz, shapes.split);
    }
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return (int)e;
    Timed timed(kFwdMerge, s);
    hipLaunchKernelGGL(merge_kernel<true>(nparts), dim3((unsigned)((Tb + kMergeTokens - 1) / kMergeTokens)), dim3(kMergeThreads), 0, s, pmax,
                       psum, want_pz ? ppz : (float*)nullptr, (int)nparts, (int)Tb, Hp, (int)ld_hidden, Wp, (int)ld_weight,
                       labels + t0, (int)H, (int)V, rcp_temperature, logprobs + t0, entropy ? entropy + t0 : (float*)nullptr,
                       row_lse ? row_lse + t0 : (float*)nullptr, row_pz ? row_pz + t0 : (float*)nullptr);
    if ((e = hipGetLastError()) != hipSuccess) return (int)e;
  }
  return SKYRL_LMHEAD_OK;
}

// Address of this device's copy of the static scratch array.  Every device holds its own copy of a __device__ array at
// its own address, so the address is looked up once per device, with that device current, and kept.
constexpr int kMaxDevices = 64;
void* g_static_scratch_ptr[kMaxDevices];
std::mutex g_static_scratch_mutex;

int static_scratch_of_current_device(void** out) {
  int dev = -1;
  hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess) return (int)e;
  if (dev < 0 || dev >= kMaxDevices) return SKYRL_LMHEAD_ERR_ARG;
  std::lock_guard<std::mutex> lock(g_static_scratch_mutex);
  if (!g_static_scratch_ptr[dev]) {
    void* p = nullptr;
    e = hipGetSymbolAddress(&p, HIP_SYMBOL(static_scratch));
    if (e != hipSuccess) return (int)e;
    if (!p || ((uintptr_t)p & 255u)) return SKYRL_LMHEAD_ERR_ALIGN;
    g_static_scratch_ptr[dev] = p;
  }
  *out = g_static_scratch_ptr[dev];
  return SKYRL_LMHEAD_OK;
}

// The backward, like the forward, walks the tokens in blocks: dHidden rows are complete within their block, dW is summed
// over the blocks (the first block stores or adds as the caller's dw_mode says, the later ones add), and every scratch
// matrix is sized by the block.  One block for T <= 32768, which covers every shape whose step time is quoted anywhere.
constexpr int64_t kBwdTokenBlock = 32768;

struct BwdWorkspace {
  uint16_t *Wt, *Ht, *D;
  float *dHacc, *dWsum, *label_resid;
  // only with row compaction (skyrl_lmhead_bwd_active_rows):
  uint16_t* hidden_c;
  int64_t* labels_c;
  float *lse_c, *pz_c, *g_c, *q_c;
  int *idx, *counts;
  int64_t slots;  // slab tiles dHacc holds
  size_t bytes;
};

// The dHidden GEMM contracts over the vocabulary, in whole pairs of k-tiles, and reads the weight rows where they are
// (K-major B operand); the last, incomplete group of a vocabulary that is not a multiple of 128 is moved back (VocabTail).
// A transposed, zero-padded copy in the workspace stays below 1024 rows only: a vocabulary below 128 has no group to move
// back, and there the copy is the cheaper side -- whole backward, copy against in place: 42.3 / 44.0 us at T=300, H=128,
// V=1000; 60.7 / 59.4 at T=512, H=1024, V=1000; 79.8 / 75.9 at V=2001; 515 / 499 at V=32001.  A pass over the weight saved:
// 0.38 of 5.9 ms at T=2654, H=4096, V=128261.
constexpr int64_t kInPlaceMinVocab = 1024;
inline bool reads_weight_in_place(int64_t V) { return V % (2 * BK) == 0 || V >= kInPlaceMinVocab; }
inline VocabTail vocab_tail(int64_t V) {
  const int64_t rest = V % (2 * BK);
  if (rest == 0 || !reads_weight_in_place(V)) return VocabTail{0x7fffffff, 0};
  return VocabTail{(int)(V - rest), (int)(2 * BK - rest)};
}

inline int64_t bwd_block_tokens(int64_t T) { return T < kBwdTokenBlock ? T : kBwdTokenBlock; }
inline int64_t bwd_num_blocks(int64_t T) { return (T + kBwdTokenBlock - 1) / kBwdTokenBlock; }

// vc: chunk width for a block of bwd_block_tokens(T) tokens.  compact: the buffers of the row-compacting entry point.
// Hk: length of the logits contraction, a multiple of H when the operands are stacked bf16 terms of fp32 values.
BwdWorkspace lay_out_bwd(void* ws, int64_t T, int64_t H, int64_t Hk, int64_t V, int64_t vc, bool compact, int64_t slab_floats) {
  const int64_t Tb = bwd_block_tokens(T), Tpad = round_up(Tb, 256), Vpad = round_up(V, 256);
  Carver c(ws);
  BwdWorkspace w{};
  w.Wt = reads_weight_in_place(V) ? nullptr : c.take<uint16_t>((size_t)H * (Vpad + kLdPad));
  w.Ht = c.take<uint16_t>((size_t)H * (Tpad + kLdPad));
  w.slots = slab_floats / kSlabTileFloats;
  w.dHacc = c.take<float>((size_t)slab_floats);  // dHidden partial sums in accumulator order, whole tiles
  w.D = c.take<uint16_t>((size_t)Tpad * (vc + kLdPad));
  // Several blocks and a bf16 dW: the sum over the blocks is kept in fp32 here and rounded once, by the last block.
  w.dWsum = bwd_num_blocks(T) > 1 ? c.take<float>((size_t)V * (size_t)H) : nullptr;
  w.label_resid = Hk > H ? c.take<float>((size_t)Tpad) : nullptr;  // stacked terms: fp32 operands
  if (compact) {
    w.hidden_c = c.take<uint16_t>((size_t)T * (size_t)Hk);
    w.labels_c = c.take<int64_t>((size_t)T);
    w.lse_c = c.take<float>((size_t)T);
    w.pz_c = c.take<float>((size_t)T);
    w.g_c = c.take<float>((size_t)T);
    w.q_c = c.take<float>((size_t)T);
    w.idx = c.take<int>((size_t)T);
    w.counts = c.take<int>((size_t)bwd_num_blocks(T) * 2 + 1);
  }
  w.bytes = (size_t)round_up((int64_t)c.off, 256);
  return w;
}

// The row-compacting entry point has more room for slabs: its token count, and with it the number of tiles, may be far below T.
// A result whose `bytes` exceed ws_bytes does not fit.  own_chunk: the library's choice of vc, which leaves a caller nothing to size by
// but a query, for this call or a longer one; the latter's has at least 1 MiB more, and less than that of slabs stays as it is.
BwdWorkspace carve_bwd(void* ws, int64_t T, int64_t H, int64_t Hk, int64_t V, int64_t vc, bool compact, size_t ws_bytes, bool own_chunk) {
  const int64_t Tb = bwd_block_tokens(T), more = compact ? T * H / 2 : 0;
  const int64_t wanted = slab_slots(Tb, H, vc) * kSlabTileFloats + more, least = dh_tiles(Tb, H) * kSlabTileFloats + more;
  const BwdWorkspace w = lay_out_bwd(ws, T, H, Hk, V, vc, compact, wanted);
  if (w.bytes <= ws_bytes || (own_chunk && wanted - least < 4 * kSlabTileFloats)) return w;
  return lay_out_bwd(ws, T, H, Hk, V, vc, compact, fitting_slabs(wanted, least, w.bytes - ws_bytes));
}

GemmArgs make_gemm(const uint16_t* A, int64_t lda, int64_t a_rows, const uint16_t* B, int64_t ldb, int64_t b_rows, bool b_kmajor,
                   bool c_rows_m, int64_t nk, int64_t M, int64_t N, const float* Cin, float* Cf, uint16_t* Cb, int64_t ldc,
                   const int* T_dev = nullptr, int t_role = 0) {
  GemmArgs g{};
  g.A = A, g.lda = (int)lda, g.a_rows = (int)a_rows, g.B = B, g.ldb = (int)ldb, g.b_rows = (int)b_rows;
  g.b_kmajor = b_kmajor ? 1 : 0, g.c_rows_m = c_rows_m ? 1 : 0, g.nk = (int)nk, g.M = (int)M, g.N = (int)N;
  g.Cin = Cin, g.Cf = Cf, g.Cb = Cb, g.ldc = (int)ldc;
  g.splits = 1, g.T_dev = T_dev, g.t_role = t_role, g.n_tail = 0x7fffffff;
  return g;
}

unsigned gemm_tiles(const GemmArgs& g) { return (unsigned)(((g.M + BM - 1) / BM) * ((g.N + BN - 1) / BN)); }

// dHidden of one vocab chunk, C[t, h] (+)= sum_v D[t, v] . weight[vc0 + v, h].  In place: A = D rows (K = vocab, contiguous), B =
// weight rows vc0.. read K-major; the k extent stops at the end of V's last group of 128.  Otherwise (a small vocabulary with a
// transposed copy): C[h, t] with A = weight^T rows, B = D rows, and no splits.
GemmArgs dhidden_gemm(const uint16_t* D, int64_t ldd, int64_t d_rows, const uint16_t* W, int64_t ldw, const uint16_t* Wt,
                      int64_t ldwt, int64_t vc0, int64_t vcw, int64_t V, int64_t T, int64_t H, uint16_t* d_hidden, float* slabs,
                      bool first, bool last, const int* T_dev) {
  const VocabTail tail = vocab_tail(V);
  const int64_t kext = round_up((V - vc0) < vcw ? (V - vc0) : vcw, 2 * BK);
  GemmArgs g = Wt ? make_gemm(Wt + vc0, ldwt, H, D, ldd, d_rows, false, false, vcw / BK, H, T, nullptr, nullptr, d_hidden, H, T_dev,
                              kTokensOnN)
                  : make_gemm(D, ldd, d_rows, W + (size_t)vc0 * (size_t)ldw, ldw, H, true, true, kext / BK, T, H, nullptr, nullptr,
                              d_hidden, H, T_dev, kTokensOnM);
  g.P = slabs, g.p_first = first, g.p_last = last;
  if (last) g.k_back = tail.back;
  return g;
}

hipError_t launch_bwd_dz(hipStream_t s, bool entgrad, DzArgs z) {
  Timed timed(kBwdChunkDz, s);
  if (half_tile_logits(z.T)) {
    z.tiles_n = 1;
    return launch_bwd_half_dz(s, entgrad, z);
  }
  z.tiles_n = (z.T + BN - 1) / BN;
  const int tiles = z.tiles_m * z.tiles_n;
  const TileShapes shapes = z.T_dev ? tile_shapes_of_any_count(z.H, z.tiles_m, tiles, z.ncu) : tile_shapes(z.T, z.H, z.tiles_m, z.ncu);
  auto kernel = flagged_kernel([](auto ent, auto even, auto others) { return &lmhead_bwd_dz<ent.value, even.value, others.value>; },
                               entgrad, even_ktiles(z.H), shapes.used);
  hipLaunchKernelGGL(kernel, dim3((unsigned)(tiles + shapes.split)), dim3(NTHREADS), 0, s, z);
  return hipGetLastError();
}

// Both problems (p1 may be empty) must have an even number of k-tiles: every caller contracts over padded extents that
// are multiples of 256, or over vocabulary rows that reads_weight_in_place() admits.
// split: the problem that p0's splits are chosen with, here or on the device.
hipError_t launch_bwd_gemm(hipStream_t s, const GemmArgs& p0, const GemmArgs& p1, const SplitProblem& split) {
  if ((p0.nk & 1) || (p1.nk & 1)) return hipErrorInvalidValue;
  const unsigned t1 = gemm_tiles(p1);
  const DhLaunch launch = dh_launch(split, (int)gemm_tiles(p0), p0.splits, p0.splits_dev != nullptr);
  const unsigned t0 = (unsigned)launch.workgroups;
  Timed timed(kBwdChunkGemm, s);
  if (launch.shares && p0.b_kmajor) {  // a transposed copy of the weight (b_kmajor 0) is never split
    if (t1 != 0) return hipErrorInvalidValue;
    hipLaunchKernelGGL(lmhead_bwd_dh_shares, dim3(t0), dim3(NTHREADS), 0, s, p0);
    return hipGetLastError();
  }
  hipLaunchKernelGGL(lmhead_bwd_gemm, dim3(t0 + t1), dim3(NTHREADS), 0, s, p0, p1, (int)t0);
  return hipGetLastError();
}

// Whether dW of a call has a launch of its own, launch_bwd_dw_few(), rather than 256 x 256 tiles next to the dHidden tiles.  Both sides of
// the line, all launches behind the dz tiles, tiles in one launch -> own launch: T=137 248 -> 177 us at H=896, 375 -> 276 at H=1536
// (V=151936), 860 -> 604 at H=4096, V=128261; T=400 554 -> 451 and 1315 -> 1080; T=768, H=3584, V=152064 1760 -> 1630; T=1024 947 -> 883
// and 2017 -> 2037; T=1400, H=4096 2776 -> 3074.  Below three rounds of two tiles per CU the second launch costs what it gains: 1000
// tiles (V=32000, H=1024) 75 -> 85 us at T=256, 2000 tiles (V=32000, H=2048) 114 -> 108.
constexpr int64_t kDwFewTokens = 768, kDwFewTiles = 1536;
inline bool few_token_dw(bool want_dw, bool adds, int64_t T, int64_t H, int64_t V) {
  return want_dw && !adds && T <= kDwFewTokens && dw_few_tiles(H, V) >= kDwFewTiles;
}

// The sum over the slabs of a split dHidden contraction; g is the GEMM of the last chunk, split the problem that its splits are chosen with.
hipError_t launch_dh_reduce(hipStream_t s, const GemmArgs& g, const SplitProblem& split) {
  if (!g.splits_dev && g.splits < 2) return hipSuccess;
  // a problem with more tiles than slots is never split, and without shares none with more than half as many
  const int64_t tiles = gemm_tiles(g), slots = split.shares ? split.slots : split.slots / 2, most = g.splits_dev && slots < tiles ? slots : tiles;
  if (most < 1) return hipSuccess;
  Timed timed(kDhReduce, s);
  hipLaunchKernelGGL(split.shares ? lmhead_dh_reduce<true> : lmhead_dh_reduce<false>, dim3((unsigned)(most * kReduceGroups)), dim3(256), 0, s,
                     DhReduceArgs{g.P, g.M, g.N, g.splits, g.T_dev, g.splits_dev, g.row_map, g.Cb, g.ldc});
  return hipGetLastError();
}

// Workspaces of the soft cross-entropy: the stacked hidden rows first in both.
constexpr int64_t kPairTile = BN / 2;  // tokens per workgroup tile of stacked rows

struct SoftCeFwdWorkspace {
  uint16_t* S;
  float *pmax, *psum, *ppz, *row_lse, *row_pz;
  size_t nparts, bytes;
};

SoftCeFwdWorkspace carve_softce_fwd(void* ws, int64_t T, int64_t H, int64_t V) {
  const int64_t Tp = round_up(T, kPairTile);
  Carver c(ws);
  SoftCeFwdWorkspace w;
  w.nparts = (size_t)((V + BM - 1) / BM) * WAVES_M;
  w.S = c.take<uint16_t>((size_t)(2 * Tp) * (size_t)H);
  w.pmax = c.take<float>(part_elems(w.nparts, 2 * Tp));
  w.psum = c.take<float>(part_elems(w.nparts, 2 * Tp));
  w.ppz = c.take<float>(part_elems(w.nparts, 2 * Tp));
  w.row_lse = c.take<float>((size_t)(2 * Tp));
  w.row_pz = c.take<float>((size_t)(2 * Tp));
  w.bytes = (size_t)round_up((int64_t)c.off, 256);
  return w;
}

struct SoftCeBwdWorkspace {
  uint16_t *S, *Wt, *D;
  float *dHacc, *lse_student, *lse_teacher, *dloss;  // the latter three: of the tokens with an upstream gradient
  int *idx, *counts;
  int64_t slots;
  size_t bytes;
};

SoftCeBwdWorkspace lay_out_softce_bwd(void* ws, int64_t T, int64_t H, int64_t V, int64_t vc, int64_t slab_floats) {
  const int64_t Tp = round_up(T, kPairTile), Vpad = round_up(V, 256);
  Carver c(ws);
  SoftCeBwdWorkspace w;
  w.S = c.take<uint16_t>((size_t)(2 * Tp) * (size_t)H);
  w.Wt = reads_weight_in_place(V) ? nullptr : c.take<uint16_t>((size_t)H * (Vpad + kLdPad));
  w.slots = slab_floats / kSlabTileFloats;
  w.dHacc = c.take<float>((size_t)slab_floats);
  w.D = c.take<uint16_t>((size_t)Tp * (vc + kLdPad));
  w.lse_student = c.take<float>((size_t)T);
  w.lse_teacher = c.take<float>((size_t)T);
  w.dloss = c.take<float>((size_t)T);
  w.idx = c.take<int>((size_t)T);
  w.counts = c.take<int>(3);
  w.bytes = (size_t)round_up((int64_t)c.off, 256);
  return w;
}

// As carve_bwd; a quarter more slabs let a batch with few active tokens split further, and 64 MiB at least of more lets dHidden tiles that fill
// whole rounds and a part of one go in equal shares.
SoftCeBwdWorkspace carve_softce_bwd(void* ws, int64_t T, int64_t H, int64_t V, int64_t vc, size_t ws_bytes) {
  const int64_t slots = slab_slots(T, H, vc), more = dh_tiles(T, H) >= kSplitBelowTiles && slots < 4 * 256 ? 256 : slots / 4;
  const int64_t wanted = (slots + more) * kSlabTileFloats;
  const SoftCeBwdWorkspace w = lay_out_softce_bwd(ws, T, H, V, vc, wanted);
  if (w.bytes <= ws_bytes) return w;
  return lay_out_softce_bwd(ws, T, H, V, vc, fitting_slabs(wanted, dh_tiles(T, H) * kSlabTileFloats, w.bytes - ws_bytes));
}

int check_softce(const void* student, int64_t lds_, const void* teacher, int64_t ldt, const void* weight, int64_t ldw, int64_t T,
                 int64_t seq_len, int64_t shift, int64_t H, int64_t V, float rcp_temperature) {
  if (!teacher) return SKYRL_LMHEAD_ERR_NULL;
  int st = check_operands(student, lds_, weight, ldw, T, H, V, rcp_temperature);
  if (st) return st;
  if (ldt < H || ldt > kMaxRowPitch) return SKYRL_LMHEAD_ERR_SHAPE;
  if (seq_len < 1 || T % seq_len != 0 || shift < 0) return SKYRL_LMHEAD_ERR_SHAPE;
  if (!aligned16(teacher) || ldt % 8 != 0) return SKYRL_LMHEAD_ERR_ALIGN;
  return SKYRL_LMHEAD_OK;
}

hipError_t launch_softce_pack(hipStream_t s, const void* student, int64_t lds_, const void* teacher, int64_t ldt, int64_t T,
                              int64_t seq_len, int64_t shift, int64_t H, uint16_t* S) {
  Timed timed(kSoftCePack, s);
  hipLaunchKernelGGL(softce_pack_rows, dim3((unsigned)stacked_rows((int)T)), dim3(256), 0, s, (const uint16_t*)student,
                     (int)lds_, (const uint16_t*)teacher, (int)ldt, (int)T, (int)seq_len, (int)(shift % seq_len), (int)H, S);
  return hipGetLastError();
}


// Top-k logits from hidden states.  Tokens are walked in blocks of at most 16384, the vocabulary in chunks.  The first chunk's
// logits are stored and searched (topk_init); from then on a logit passes with probability k / (columns seen so far) on
// exchangeable columns, so a later chunk may be 512 / k times as wide as what was seen before it and still leaves half a bulk
// round to topk_select.  A candidate list holds a whole chunk (cap columns per token), which makes the filter exact for any
// data: in the worst case -- logits ascending with the column -- every logit is a candidate and the select kernel does all the
// work.  What the lists may take, 1 GiB, is shared by the tokens of a block: few tokens mean few, wide chunks and so few launches
// whose tiles fill whole rounds of the CUs (T=1800, H=2048, V=151936, k=32: 21 chunks, 1.20 + 0.30 ms of tiles and selection -> 3 chunks, 1.11 + 0.08 ms).
constexpr int64_t kTopkTokenBlock = 16384;
constexpr int64_t kTopkListColumns = 8192;  // per token of a full block
constexpr int64_t kTopkDenseMin = 8192, kTopkDenseMax = 1024 * topk::kInitLogits;

struct TopkWorkspace {
  unsigned *cnt, *have;
  float* thr;
  topk::key_t *best, *cand;
  int64_t block_tokens, cap;
  size_t bytes;
};

// The columns of a list: as many as the scratch holds, at most what the 1 GiB allows and at least kTopkListColumns, which any block can
// have.  A narrower list means more chunks and launches, and the same results.
TopkWorkspace carve_topk(void* ws, int64_t T, int64_t V, int64_t k, size_t ws_bytes) {
  TopkWorkspace w;
  w.block_tokens = T < kTopkTokenBlock ? T : kTopkTokenBlock;
  const int64_t vpad = round_up(V, 256), room = kTopkTokenBlock * kTopkListColumns / w.block_tokens / 256 * 256;
  const int64_t widest = vpad < room ? vpad : room, narrowest = vpad < kTopkListColumns ? vpad : kTopkListColumns;
  Carver c(ws);
  w.cnt = c.take<unsigned>((size_t)w.block_tokens);
  w.have = c.take<unsigned>((size_t)w.block_tokens);
  w.thr = c.take<float>((size_t)w.block_tokens);
  w.best = c.take<topk::key_t>((size_t)w.block_tokens * (size_t)k);
  const size_t column = (size_t)w.block_tokens * sizeof(topk::key_t), fixed = (size_t)round_up((int64_t)c.off, 256);
  const size_t fits = ws_bytes > fixed ? (ws_bytes - fixed) / column : 0;
  w.cap = fits < (size_t)widest ? (int64_t)fits / 256 * 256 : widest;
  if (w.cap < narrowest) w.cap = narrowest;
  w.cand = c.take<topk::key_t>((size_t)w.block_tokens * (size_t)w.cap);
  w.bytes = (size_t)round_up((int64_t)c.off, 256);
  return w;
}

size_t bwd_workspace_bytes(int64_t T, int64_t H, int64_t V, int64_t vocab_chunk, bool compact, int64_t terms = 1) {
  if (T < 1 || V < 1 || H < 1 || vocab_chunk < 0 || vocab_chunk % 256 != 0 || terms < 1 || terms > 3) return 0;
  if (T > kMaxExtent || V > kMaxExtent || H > kMaxExtent / 4 || vocab_chunk > kMaxExtent) return 0;
  int64_t vc = vocab_chunk ? vocab_chunk : default_vocab_chunk(bwd_block_tokens(T), H, V);
  if (vc > round_up(V, 256)) vc = round_up(V, 256);
  return carve_bwd(nullptr, T, H, terms * H, V, vc, compact, SIZE_MAX, false).bytes;
}

// One token block of the backward: the vocab-chunk loop.  Hk is the contraction length of the logits recompute (H, or a
// multiple of it for stacked bf16 terms, in which case the two gradient GEMMs use the leading H columns: the hi terms).  `Tb` tokens (an upper bound when `T_dev` points at the block's
// count in device memory and `splits_dev` at what `rated` made of it), per-token inputs and d_hidden already offset to the block.  dW of every chunk leaves the GEMM
// epilogue as  (Cin ? Cin : 0) + product  ->  Cf (fp32) and / or Cb (bf16), each a [V, H] matrix or NULL.
int bwd_token_block(const uint16_t* Hp, int64_t ld_hidden, const uint16_t* Wp, int64_t ld_weight, const int64_t* labels,
                    const float* row_lse, const float* row_pz, const float* dlogprobs, const float* dentropy, int64_t Tb,
                    const int* T_dev, const int* splits_dev, const SplitProblem& rated, const int* row_map, int64_t H, int64_t Hk, int64_t V,
                    float rcp_temperature, uint16_t* d_hidden, bool want_dw,
                    const float* dw_in, float* dw_f32, uint16_t* dw_bf16, int64_t vc, const BwdWorkspace& w, float p_shift,
                    hipStream_t s) {
  const int64_t Tpad = round_up(Tb, 256), Vpad = round_up(V, 256);
  const int ncu = compute_units();
  const bool w_in_place = reads_weight_in_place(V);
  hipError_t e;
  const bool few = few_token_dw(want_dw, dw_in != nullptr, Tb, H, V);
  if (want_dw && !few) {  // only the dW product reads hidden^T [H, Tpad]; zero in the padding columns
    Timed timed(kTranspose, s);
    hipLaunchKernelGGL(transpose_bf16, dim3((unsigned)(Tpad / 64), (unsigned)(H / 64)), dim3(256), 0, s, Hp, (int)ld_hidden,
                       (int)Tb, (int)H, w.Ht, (int)(Tpad + kLdPad), (int)Tpad, T_dev);
    if ((e = hipGetLastError()) != hipSuccess) return (int)e;
  }
  // fp32 operands (stacked terms) with an fp32 dW: the label's dz value keeps fp32 accuracy through a residual (DzArgs).
  float* resid = (Hk > H && want_dw && dw_f32) ? w.label_resid : nullptr;
  if (resid) {
    hipLaunchKernelGGL(zero_f32, dim3((unsigned)(Tpad / 256)), dim3(256), 0, s, resid, (int)Tpad);
    if ((e = hipGetLastError()) != hipSuccess) return (int)e;
  }
  const VocabTail tail = vocab_tail(V);
  // The splits are those of a full chunk: the slabs are carried from chunk to chunk.
  const SplitProblem split = T_dev ? rated : split_problem(Tb, H, vc < Vpad ? vc : Vpad, want_dw && !few, w.slots, ncu);
  const int splits = !T_dev && w_in_place ? best_splits(split, Tb) : 1;
  const int64_t nchunks = (Vpad + vc - 1) / vc;
  auto chunk_width = [&](int64_t ci) { return (Vpad - ci * vc) < vc ? (Vpad - ci * vc) : vc; };  // multiple of 256
  const GemmArgs none{};
  for (int64_t ci = 0; ci < nchunks; ++ci) {
    // dz panel of this chunk, then the two gradient GEMMs that consume it (one launch, they are independent).
    // Carrying the next chunk's dz tiles in the GEMM launch (to fill its tail) was measured: no gain at the default chunk
    // width, and it needs a second panel.
    const int64_t vc0 = ci * vc, vcw = chunk_width(ci);
    const DzArgs z{Wp, (int)ld_weight, Hp, (int)ld_hidden, (int)Tb, (int)Hk, (int)V, rcp_temperature, labels, row_lse, row_pz,
                   dlogprobs, dentropy, (int)vc0, (int)(vcw / 256), 0, tail, w.D, (int)(vcw + kLdPad), T_dev, resid, p_shift, ncu};
    e = launch_bwd_dz(s, dentropy != nullptr, z);
    if (e != hipSuccess) return (int)e;
    // dHidden[t, h] (+)= sum_v D[t, v] . weight^T[h, vc0 + v]        (A = weight^T rows at k offset vc0, B = D rows)
    // dW[vc0 + v, h]  (+)= sum_t D[t, v] . hidden^T[h, t]             (A = hidden^T rows, B = D read K-major)
    const bool first = ci == 0, last = ci == nchunks - 1;
    const int64_t rows = (V - vc0) < vcw ? (V - vc0) : vcw;
    // dW rows are complete within their chunk (for this token block), so they can leave the GEMM epilogue in either precision.
    const size_t dw_off = (size_t)vc0 * (size_t)H;
    GemmArgs gh = dhidden_gemm(w.D, vcw + kLdPad, Tpad, Wp, ld_weight, w_in_place ? nullptr : w.Wt, Vpad + kLdPad, vc0, vcw, V, Tb, H,
                               d_hidden, w.dHacc, first, last, T_dev);
    gh.splits = splits, gh.splits_dev = w_in_place ? splits_dev : nullptr, gh.row_map = row_map;
    // A frozen LM head needs no dW: the launch then carries the dHidden tiles alone.
    const bool moved = last && tail.back > 0;  // the chunk ends with a moved group
    const int64_t n_rows = moved ? round_up(rows, 2 * BK) : rows;
    const float* const cin = dw_in ? dw_in + dw_off : nullptr;
    float* const cf = dw_f32 ? dw_f32 + dw_off : nullptr;
    uint16_t* const cb = dw_bf16 ? dw_bf16 + dw_off : nullptr;
    GemmArgs gw = want_dw && !few ? make_gemm(w.Ht, Tpad + kLdPad, H, w.D, vcw + kLdPad, vcw, true, false, round_up(Tb, 2 * BK) / BK, H, n_rows, cin,
                                              cf, cb, H, T_dev, kTokensOnK)
                                  : none;
    if (moved) gw.n_tail = (int)(tail.from - vc0), gw.n_back = tail.back;
    if (few) {
      Timed timed(kBwdDwFew, s);
      e = launch_bwd_dw_few(s, DwFewArgs{Hp, (int)ld_hidden, w.D, (int)(vcw + kLdPad), (int)Tb, T_dev, (int)H, (int)n_rows,
                                         moved ? gw.n_tail : 0x7fffffff, gw.n_back, cf, cb, ncu});
      if (e != hipSuccess) return (int)e;
    }
    e = launch_bwd_gemm(s, gh, gw, split);
    if (e == hipSuccess && last) e = launch_dh_reduce(s, gh, split);
    if (e != hipSuccess) return (int)e;
  }
  if (resid) {
    hipLaunchKernelGGL(label_residual_update, dim3((unsigned)Tb), dim3(256), 0, s, (const float*)resid, labels, Hp, (int)ld_hidden,
                       (int)H, Hk == 3 * H ? (int)(2 * H) : 0, (int)V, T_dev, dw_f32);
    if ((e = hipGetLastError()) != hipSuccess) return (int)e;
  }
  return SKYRL_LMHEAD_OK;
}

int bwd_entry(const void* hidden, int64_t ld_hidden, const void* weight, int64_t ld_weight, const int64_t* labels,
              const float* row_lse, const float* row_pz, const float* dlogprobs, const float* dentropy, int64_t T, int64_t H,
              int64_t V, float rcp_temperature, void* d_hidden, void* d_weight, int dw_mode, int64_t vocab_chunk,
              void* workspace, size_t workspace_bytes, hipStream_t s, bool compact, int64_t terms = 1) {
  if (terms < 1 || terms > 3 || H < 1 || H > kMaxExtent / 4) return SKYRL_LMHEAD_ERR_ARG;
  // dw_mode carries one option bit next to the mode: softmax probabilities below 2^-24 count as zero in dz.
  const float p_shift = (dw_mode & SKYRL_BWD_FLUSH_TINY_DZ) ? 126.f - 24.f : 0.f;
  if (dw_mode >= 0) dw_mode &= ~SKYRL_BWD_FLUSH_TINY_DZ;
  const int64_t Hk = terms * H;
  int st = check_common(hidden, ld_hidden, weight, ld_weight, labels, T, Hk, V, rcp_temperature, true);
  if (st) return st;
  if (H % BK != 0) return SKYRL_LMHEAD_ERR_SHAPE;
  if (!row_lse || !dlogprobs || !d_hidden) return SKYRL_LMHEAD_ERR_NULL;
  if (dentropy && !row_pz) return SKYRL_LMHEAD_ERR_NULL;
  if (!aligned16(d_hidden) || !aligned16(d_weight)) return SKYRL_LMHEAD_ERR_ALIGN;  // d_weight NULL: no dW wanted
  if (dw_mode < SKYRL_DW_FP32 || dw_mode > SKYRL_DW_BF16) return SKYRL_LMHEAD_ERR_ARG;
  if (vocab_chunk < 0 || vocab_chunk % 256 != 0) return SKYRL_LMHEAD_ERR_ARG;
  if (compact && T >= ((int64_t)1 << 31)) return SKYRL_LMHEAD_ERR_SHAPE;  // the row index list is 32-bit
  const int64_t Tb = bwd_block_tokens(T), Tbpad = round_up(Tb, 256), Vpad = round_up(V, 256);
  int64_t vc = vocab_chunk ? vocab_chunk : default_vocab_chunk(Tb, H, V);
  if (vc > Vpad) vc = Vpad;
  // Row pitches of the scratch matrices (weight^T, hidden^T, the dz panel) under the copy plan's limit; Hk <= ld_hidden is.
  if ((!reads_weight_in_place(V) && Vpad + kLdPad > kMaxRowPitch) || Tbpad + kLdPad > kMaxRowPitch || vc + kLdPad > kMaxRowPitch)
    return SKYRL_LMHEAD_ERR_SHAPE;
  const size_t full = bwd_workspace_bytes(T, H, V, vc, compact, terms);
  if (!vocab_chunk && workspace_bytes < full) vc = fitting_chunk(vc, Tbpad, V, full - workspace_bytes);
  const BwdWorkspace w = carve_bwd(workspace, T, H, Hk, V, vc, compact, workspace_bytes, !vocab_chunk);
  if (!workspace || workspace_bytes < w.bytes) return SKYRL_LMHEAD_ERR_WORKSPACE;
  if ((uintptr_t)workspace & 255u) return SKYRL_LMHEAD_ERR_ALIGN;

  const uint16_t* Wp = (const uint16_t*)weight;
  const uint16_t* Hp = (const uint16_t*)hidden;
  const int64_t nblocks = bwd_num_blocks(T);
  hipError_t e;

  // dW in the launch of the dHidden tiles (bwd_token_block decides the same way)
  const bool dw_in_gemm = d_weight && !few_token_dw(true, dw_mode == SKYRL_DW_FP32_ACCUMULATE || nblocks > 1, Tb, H, V);
  const SplitProblem rated = split_problem(Tb, H, vc, dw_in_gemm, w.slots, compute_units());
  if (compact) {
    Timed timed(kCompactRows, s);
    hipLaunchKernelGGL(compact_kernel(T), dim3(1), dim3(kCompactThreads), 0, s, dlogprobs, dentropy, (int)T, (int)Tb,
                       (int)nblocks, rated, w.idx, w.counts);
    hipLaunchKernelGGL(gather_active_rows, dim3((unsigned)T), dim3(256), 0, s, (const int*)w.idx, (const int*)w.counts, Hp,
                       (int)ld_hidden, (int)Hk, (int)H, labels, row_lse, row_pz, dlogprobs, dentropy, w.hidden_c, w.labels_c,
                       w.lse_c, w.pz_c, w.g_c, w.q_c, (uint16_t*)d_hidden);
    if ((e = hipGetLastError()) != hipSuccess) return (int)e;
  }
  if (!reads_weight_in_place(V)) {  // weight^T [H, Vpad], zero in the padding columns
    Timed timed(kTranspose, s);
    hipLaunchKernelGGL(transpose_bf16, dim3((unsigned)(Vpad / 64), (unsigned)(H / 64)), dim3(256), 0, s, Wp, (int)ld_weight,
                       (int)V, (int)H, w.Wt, (int)(Vpad + kLdPad), (int)Vpad, (const int*)nullptr);
    if ((e = hipGetLastError()) != hipSuccess) return (int)e;
  }

  for (int64_t b = 0; b < nblocks; ++b) {
    const int64_t t0 = b * Tb, Tcur = (T - t0) < Tb ? (T - t0) : Tb;
    // Where dW of this block comes from and goes to.  One block: straight to the caller's matrix as dw_mode says.  Several
    // blocks: fp32 modes add every later block to the caller's matrix; the bf16 mode sums in the fp32 scratch matrix and
    // the last block rounds the sum into the caller's.
    const float* dw_in = nullptr;
    float* dw_f32 = nullptr;
    uint16_t* dw_bf16 = nullptr;
    if (d_weight) {
      const bool first = b == 0, last = b == nblocks - 1;
      if (dw_mode == SKYRL_DW_BF16) {
        if (nblocks == 1) {
          dw_bf16 = (uint16_t*)d_weight;
        } else {
          dw_in = first ? nullptr : w.dWsum;
          if (last) dw_bf16 = (uint16_t*)d_weight; else dw_f32 = w.dWsum;
        }
      } else {
        dw_f32 = (float*)d_weight;
        dw_in = (dw_mode == SKYRL_DW_FP32_ACCUMULATE || !first) ? (const float*)d_weight : nullptr;
      }
    }
    if (compact) {
      st = bwd_token_block(w.hidden_c + (size_t)t0 * (size_t)Hk, Hk, Wp, ld_weight, w.labels_c + t0, w.lse_c + t0,
                           dentropy ? w.pz_c + t0 : nullptr, w.g_c + t0, dentropy ? w.q_c + t0 : nullptr, Tcur,
                           w.counts + 1 + b, w.counts + 1 + nblocks + b, rated, w.idx + t0, H, Hk, V, rcp_temperature, (uint16_t*)d_hidden,
                           d_weight != nullptr, dw_in, dw_f32, dw_bf16, vc, w, p_shift, s);
    } else {
      st = bwd_token_block(Hp + (size_t)t0 * (size_t)ld_hidden, ld_hidden, Wp, ld_weight, labels + t0, row_lse + t0,
                           row_pz ? row_pz + t0 : nullptr, dlogprobs + t0, dentropy ? dentropy + t0 : nullptr, Tcur, nullptr,
                           nullptr, rated, nullptr, H, Hk, V, rcp_temperature, (uint16_t*)d_hidden + (size_t)t0 * (size_t)H, d_weight != nullptr, dw_in, dw_f32,
                           dw_bf16, vc, w, p_shift, s);
    }
    if (st) return st;
  }
  return SKYRL_LMHEAD_OK;
}

}  // namespace

extern "C" {

int skyrl_lmhead_version(void) { return 20; }

const char* skyrl_lmhead_strerror(int status) {
  switch (status) {
    case SKYRL_LMHEAD_OK: return "ok";
    case SKYRL_LMHEAD_ERR_NULL: return "a required pointer is NULL (or only some of seg_row, seg_col, seg_len are given)";
    case SKYRL_LMHEAD_ERR_SHAPE:
      return "bad shape: need T >= 1, V >= 1, H a positive multiple of 64, leading dimensions >= H and at most 4194304 elements; "
             "packed-sequence calls: counts >= 0, rows == num_seqs with an attention mask";
    case SKYRL_LMHEAD_ERR_ALIGN: return "bad alignment: pointers must be 16-byte aligned, leading dimensions multiples of 8";
    case SKYRL_LMHEAD_ERR_WORKSPACE: return "workspace is NULL or too small";
    case SKYRL_LMHEAD_ERR_TOO_LARGE:
      return "too large for the entry point that uses the library's fixed scratch array: V exceeds "
             "SKYRL_LMHEAD_STATIC_SCRATCH_MAX_V; use skyrl_lmhead_fwd with a caller-provided workspace";
    case SKYRL_LMHEAD_ERR_ARG:
      return "bad argument: rcp_temperature must be finite and > 0, vocab_chunk a multiple of 256; packed-sequence calls take "
             "sub-sequence arrays or an attention mask, not both";
    default: break;
  }
  if (status > 0) return hipGetErrorString((hipError_t)status);
  return "unknown skyrl_lmhead status";
}

size_t skyrl_lmhead_fwd_workspace_bytes(int64_t T, int64_t H, int64_t V) {
  (void)H;
  if (T < 1 || V < 1 || T > kMaxExtent || V > kMaxExtent) return 0;
  return fwd_partials_bytes(T < kFwdTokenBlock ? T : kFwdTokenBlock, V);
}

size_t skyrl_lmhead_bwd_workspace_bytes(int64_t T, int64_t H, int64_t V, int64_t vocab_chunk) {
  return bwd_workspace_bytes(T, H, V, vocab_chunk, false);
}

size_t skyrl_lmhead_bwd_active_rows_workspace_bytes(int64_t T, int64_t H, int64_t V, int64_t vocab_chunk) {
  return bwd_workspace_bytes(T, H, V, vocab_chunk, true);
}

int skyrl_lmhead_fwd(const void* hidden, int64_t ld_hidden, const void* weight, int64_t ld_weight, const int64_t* labels,
                     int64_t T, int64_t H, int64_t V, float rcp_temperature, float* logprobs, float* entropy,
                     float* row_lse, float* row_pz, void* workspace, size_t workspace_bytes, void* stream) {
  int st = check_common(hidden, ld_hidden, weight, ld_weight, labels, T, H, V, rcp_temperature, true);
  if (st) return st;
  if (!logprobs) return SKYRL_LMHEAD_ERR_NULL;
  if (!workspace || workspace_bytes < skyrl_lmhead_fwd_workspace_bytes(T, H, V)) return SKYRL_LMHEAD_ERR_WORKSPACE;
  if ((uintptr_t)workspace & 255u) return SKYRL_LMHEAD_ERR_ALIGN;
  return fwd_token_blocks(hidden, ld_hidden, weight, ld_weight, labels, T, H, V, rcp_temperature, logprobs, entropy, row_lse,
                          row_pz, workspace, fwd_block_tokens(kFwdTokenBlock, ld_hidden), (hipStream_t)stream);
}

int skyrl_lmhead_fwd_static_scratch(const void* hidden, int64_t ld_hidden, const void* weight, int64_t ld_weight,
                                    const int64_t* labels, int64_t T, int64_t H, int64_t V, float rcp_temperature,
                                    float* logprobs, float* entropy, float* row_lse, float* row_pz, void* stream) {
  int st = check_common(hidden, ld_hidden, weight, ld_weight, labels, T, H, V, rcp_temperature, true);
  if (st) return st;
  if (!logprobs) return SKYRL_LMHEAD_ERR_NULL;
  // Token block: the most 256-token tiles whose partials fit the static array.
  const int64_t block = (int64_t)(kStaticScratchBytes / fwd_partials_bytes(BN, V)) * BN;
  if (V > SKYRL_LMHEAD_STATIC_SCRATCH_MAX_V || block < BN) return SKYRL_LMHEAD_ERR_TOO_LARGE;
  void* scratch_ptr = nullptr;
  if ((st = static_scratch_of_current_device(&scratch_ptr)) != SKYRL_LMHEAD_OK) return st;
  return fwd_token_blocks(hidden, ld_hidden, weight, ld_weight, labels, T, H, V, rcp_temperature, logprobs, entropy, row_lse,
                          row_pz, scratch_ptr, fwd_block_tokens(block, ld_hidden), (hipStream_t)stream);
}

size_t skyrl_lmhead_static_scratch_bytes(void) { return kStaticScratchBytes; }

int skyrl_lmhead_bwd(const void* hidden, int64_t ld_hidden, const void* weight, int64_t ld_weight, const int64_t* labels,
                     const float* row_lse, const float* row_pz, const float* dlogprobs, const float* dentropy, int64_t T,
                     int64_t H, int64_t V, float rcp_temperature, void* d_hidden, void* d_weight, int dw_mode,
                     int64_t vocab_chunk, void* workspace, size_t workspace_bytes, void* stream) {
  return bwd_entry(hidden, ld_hidden, weight, ld_weight, labels, row_lse, row_pz, dlogprobs, dentropy, T, H, V, rcp_temperature,
                   d_hidden, d_weight, dw_mode, vocab_chunk, workspace, workspace_bytes, (hipStream_t)stream, false);
}

int skyrl_lmhead_bwd_active_rows(const void* hidden, int64_t ld_hidden, const void* weight, int64_t ld_weight,
                                 const int64_t* labels, const float* row_lse, const float* row_pz, const float* dlogprobs,
                                 const float* dentropy, int64_t T, int64_t H, int64_t V, float rcp_temperature, void* d_hidden,
                                 void* d_weight, int dw_mode, int64_t vocab_chunk, void* workspace, size_t workspace_bytes,
                                 void* stream) {
  return bwd_entry(hidden, ld_hidden, weight, ld_weight, labels, row_lse, row_pz, dlogprobs, dentropy, T, H, V, rcp_temperature,
                   d_hidden, d_weight, dw_mode, vocab_chunk, workspace, workspace_bytes, (hipStream_t)stream, true);
}

size_t skyrl_lmhead_bwd_split_workspace_bytes(int64_t T, int64_t H, int64_t terms, int64_t V, int64_t vocab_chunk,
                                              int active_rows) {
  return bwd_workspace_bytes(T, H, V, vocab_chunk, active_rows != 0, terms);
}

int skyrl_lmhead_bwd_split(const void* hidden_terms, int64_t ld_hidden, const void* weight_terms, int64_t ld_weight,
                           const int64_t* labels, const float* row_lse, const float* row_pz, const float* dlogprobs,
                           const float* dentropy, int64_t T, int64_t H, int64_t terms, int64_t V, float rcp_temperature,
                           void* d_hidden, void* d_weight, int dw_mode, int64_t vocab_chunk, int active_rows, void* workspace,
                           size_t workspace_bytes, void* stream) {
  return bwd_entry(hidden_terms, ld_hidden, weight_terms, ld_weight, labels, row_lse, row_pz, dlogprobs, dentropy, T, H, V,
                   rcp_temperature, d_hidden, d_weight, dw_mode, vocab_chunk, workspace, workspace_bytes, (hipStream_t)stream,
                   active_rows != 0, terms);
}

int skyrl_lmhead_split_operand(const void* src, int src_is_fp32, int64_t ld_src, int64_t rows, int64_t H, int layout, void* dst,
                               int64_t ld_dst, void* stream) {
  if (!src || !dst) return SKYRL_LMHEAD_ERR_NULL;
  int terms, codes[3] = {0, 0, 0};
  switch (layout) {
    case SKYRL_SPLIT_HI_LO: terms = 2, codes[1] = 1; break;
    case SKYRL_SPLIT_HI_HI: terms = 2; break;
    case SKYRL_SPLIT_HI_LO_HI: terms = 3, codes[1] = 1; break;
    case SKYRL_SPLIT_HI_HI_LO: terms = 3, codes[2] = 1; break;
    default: return SKYRL_LMHEAD_ERR_ARG;
  }
  if (rows < 1 || rows > kMaxExtent || H < 4 || H % 4 != 0 || H > kMaxExtent / 4 || ld_src < H || ld_dst < terms * H ||
      ld_src > kMaxExtent || ld_dst > kMaxExtent)
    return SKYRL_LMHEAD_ERR_SHAPE;
  if (!aligned16(src) || !aligned16(dst) || ld_src % 4 != 0 || ld_dst % 8 != 0) return SKYRL_LMHEAD_ERR_ALIGN;
  hipStream_t s = (hipStream_t)stream;
  Timed timed(kSplitOperand, s);
  if (src_is_fp32)
    hipLaunchKernelGGL(split_operand_rows<true>, dim3((unsigned)rows), dim3(256), 0, s, src, ld_src, (int)H, terms, codes[0],
                       codes[1], codes[2], (uint16_t*)dst, ld_dst);
  else
    hipLaunchKernelGGL(split_operand_rows<false>, dim3((unsigned)rows), dim3(256), 0, s, src, ld_src, (int)H, terms, codes[0],
                       codes[1], codes[2], (uint16_t*)dst, ld_dst);
  const hipError_t e = hipGetLastError();
  return e == hipSuccess ? SKYRL_LMHEAD_OK : (int)e;
}

size_t skyrl_softce_fwd_workspace_bytes(int64_t T, int64_t H, int64_t V) {
  if (T < 1 || V < 1 || H < 1 || T > kMaxExtent || V > kMaxExtent || H > kMaxExtent) return 0;
  return carve_softce_fwd(nullptr, T, H, V).bytes;
}

size_t skyrl_softce_bwd_workspace_bytes(int64_t T, int64_t H, int64_t V, int64_t vocab_chunk) {
  if (T < 1 || V < 1 || H < 1 || vocab_chunk < 0 || vocab_chunk % 256 != 0) return 0;
  if (T > kMaxExtent || V > kMaxExtent || H > kMaxExtent || vocab_chunk > kMaxExtent) return 0;
  int64_t vc = vocab_chunk ? vocab_chunk : default_vocab_chunk(T, H, V);
  if (vc > round_up(V, 256)) vc = round_up(V, 256);
  return carve_softce_bwd(nullptr, T, H, V, vc, SIZE_MAX).bytes;
}

int skyrl_softce_fwd(const void* student_hidden, int64_t ld_student, const void* teacher_hidden, int64_t ld_teacher,
                     const void* weight, int64_t ld_weight, int64_t T, int64_t seq_len, int64_t shift, int64_t H, int64_t V,
                     float rcp_temperature, float* loss, float* lse_student, float* lse_teacher, void* workspace,
                     size_t workspace_bytes, void* stream) {
  int st = check_softce(student_hidden, ld_student, teacher_hidden, ld_teacher, weight, ld_weight, T, seq_len, shift, H, V,
                        rcp_temperature);
  if (st) return st;
  if (!loss || !lse_student || !lse_teacher) return SKYRL_LMHEAD_ERR_NULL;
  if (!workspace || workspace_bytes < skyrl_softce_fwd_workspace_bytes(T, H, V)) return SKYRL_LMHEAD_ERR_WORKSPACE;
  if ((uintptr_t)workspace & 255u) return SKYRL_LMHEAD_ERR_ALIGN;

  hipStream_t s = (hipStream_t)stream;
  const SoftCeFwdWorkspace w = carve_softce_fwd(workspace, T, H, V);
  const int64_t rows = stacked_rows((int)T);
  const uint16_t* Wp = (const uint16_t*)weight;
  hipError_t e = launch_softce_pack(s, student_hidden, ld_student, teacher_hidden, ld_teacher, T, seq_len, shift, H, w.S);
  if (e != hipSuccess) return (int)e;
  const int tiles_m = (int)((V + BM - 1) / BM), tiles_n = (int)((rows + BN - 1) / BN);
  const TileShapes shapes = tile_shapes(rows, H, tiles_m, compute_units());
  {
    Timed timed(kSoftCeFwdTiles, s);
    auto kernel = flagged_kernel([](auto, auto even, auto others) { return &softce_fwd_tiles<even.value, others.value>; }, true,
                                 even_ktiles(H), shapes.used);
    hipLaunchKernelGGL(kernel, dim3((unsigned)(tiles_m * tiles_n + shapes.split)), dim3(NTHREADS), 0, s, Wp, (int)ld_weight, w.S, (int)H,
                       (int)rows, (int)H, (int)V, rcp_temperature, w.pmax, w.psum, w.ppz, shapes.split);
  }
  if ((e = hipGetLastError()) != hipSuccess) return (int)e;
  {
    Timed timed(kFwdMerge, s);
    hipLaunchKernelGGL(merge_kernel<false>(w.nparts), dim3((unsigned)((rows + kMergeTokens - 1) / kMergeTokens)), dim3(kMergeThreads), 0, s, w.pmax,
                       w.psum, w.ppz, (int)w.nparts, (int)rows, w.S, (int)H, Wp, (int)ld_weight, (const int64_t*)nullptr, (int)H,
                       (int)V, rcp_temperature, (float*)nullptr, (float*)nullptr, w.row_lse, w.row_pz);
  }
  if ((e = hipGetLastError()) != hipSuccess) return (int)e;
  Timed timed(kSoftCeFinish, s);
  hipLaunchKernelGGL(softce_finish, dim3((unsigned)((T + 255) / 256)), dim3(256), 0, s, w.row_lse, w.row_pz, (int)T, loss,
                     lse_student, lse_teacher);
  e = hipGetLastError();
  return e == hipSuccess ? SKYRL_LMHEAD_OK : (int)e;
}

int skyrl_softce_bwd(const void* student_hidden, int64_t ld_student, const void* teacher_hidden, int64_t ld_teacher,
                     const void* weight, int64_t ld_weight, const float* lse_student, const float* lse_teacher,
                     const float* dloss, int64_t T, int64_t seq_len, int64_t shift, int64_t H, int64_t V, float rcp_temperature,
                     void* d_student_hidden, int64_t vocab_chunk, void* workspace, size_t workspace_bytes, void* stream) {
  int st = check_softce(student_hidden, ld_student, teacher_hidden, ld_teacher, weight, ld_weight, T, seq_len, shift, H, V,
                        rcp_temperature);
  if (st) return st;
  if (!lse_student || !lse_teacher || !dloss || !d_student_hidden) return SKYRL_LMHEAD_ERR_NULL;
  if (!aligned16(d_student_hidden)) return SKYRL_LMHEAD_ERR_ALIGN;
  if (vocab_chunk < 0 || vocab_chunk % 256 != 0) return SKYRL_LMHEAD_ERR_ARG;
  const int64_t Tp = round_up(T, kPairTile), Vpad = round_up(V, 256);
  int64_t vc = vocab_chunk ? vocab_chunk : default_vocab_chunk(T, H, V);
  if (vc > Vpad) vc = Vpad;
  if ((!reads_weight_in_place(V) && Vpad + kLdPad > kMaxRowPitch) || vc + kLdPad > kMaxRowPitch) return SKYRL_LMHEAD_ERR_SHAPE;
  const size_t full = skyrl_softce_bwd_workspace_bytes(T, H, V, vc);
  if (!vocab_chunk && workspace_bytes < full) vc = fitting_chunk(vc, Tp, V, full - workspace_bytes);
  SoftCeBwdWorkspace w = carve_softce_bwd(workspace, T, H, V, vc, workspace_bytes);
  // The inputs of the listed tokens (16 bytes each) came to the sums and the panel: where the scratch holds only those, 256 columns of
  // the panel (512 bytes per token) make way.
  if (workspace_bytes < w.bytes && vc > BM) {
    vc -= BM;
    w = carve_softce_bwd(workspace, T, H, V, vc, workspace_bytes);
  }
  if (!workspace || workspace_bytes < w.bytes) return SKYRL_LMHEAD_ERR_WORKSPACE;
  if ((uintptr_t)workspace & 255u) return SKYRL_LMHEAD_ERR_ALIGN;

  hipStream_t s = (hipStream_t)stream;
  const uint16_t* Wp = (const uint16_t*)weight;
  hipError_t e;
  const bool w_in_place = reads_weight_in_place(V);
  const VocabTail tail = vocab_tail(V);
  const int ncu = compute_units();
  const SplitProblem split = split_problem(T, H, vc, false, w.slots, ncu);
  {  // tokens without an upstream gradient (what the supervision mask removes) have a zero row and take no part
    Timed timed(kCompactRows, s);
    hipLaunchKernelGGL(compact_kernel(T), dim3(1), dim3(kCompactThreads), 0, s, dloss, (const float*)nullptr, (int)T, (int)T, 1,
                       split, w.idx, w.counts);
  }
  if ((e = hipGetLastError()) != hipSuccess) return (int)e;
  {
    Timed timed(kSoftCePack, s);
    hipLaunchKernelGGL(softce_gather_rows, dim3((unsigned)stacked_rows((int)T)), dim3(256), 0, s, (const uint16_t*)student_hidden, (int)ld_student,
                       (const uint16_t*)teacher_hidden, (int)ld_teacher, (int)T, (int)seq_len, (int)(shift % seq_len), (int)H,
                       (const int*)w.idx, (const int*)w.counts, lse_student, lse_teacher, dloss, w.S, w.lse_student, w.lse_teacher,
                       w.dloss, (uint16_t*)d_student_hidden);
  }
  if ((e = hipGetLastError()) != hipSuccess) return (int)e;
  if (!w_in_place) {
    Timed timed(kTranspose, s);
    hipLaunchKernelGGL(transpose_bf16, dim3((unsigned)(Vpad / 64), (unsigned)(H / 64)), dim3(256), 0, s, Wp, (int)ld_weight,
                       (int)V, (int)H, w.Wt, (int)(Vpad + kLdPad), (int)Vpad, (const int*)nullptr);
    if ((e = hipGetLastError()) != hipSuccess) return (int)e;
  }
  const int64_t nchunks = (Vpad + vc - 1) / vc;
  const GemmArgs none{};
  for (int64_t ci = 0; ci < nchunks; ++ci) {
    const int64_t vc0 = ci * vc, vcw = (Vpad - vc0) < vc ? (Vpad - vc0) : vc;
    const SoftCeDzArgs z{Wp, (int)ld_weight, w.S, (int)H, (int)V, w.counts + 1, rcp_temperature, w.lse_student,
                         w.lse_teacher, w.dloss, (int)vc0, (int)(vcw / 256), (int)(2 * Tp / BN), tail, w.D, (int)(vcw + kLdPad),
                         ncu};
    {
      Timed timed(kSoftCeDz, s);
      const TileShapes shapes = tile_shapes_of_any_count(H, z.tiles_m, z.tiles_m * z.tiles_n, z.ncu);
      auto kernel = flagged_kernel([](auto, auto even, auto others) { return &softce_dz_tiles<even.value, others.value>; }, true,
                                   even_ktiles(H), shapes.used);
      hipLaunchKernelGGL(kernel, dim3((unsigned)(z.tiles_m * z.tiles_n + shapes.split)), dim3(NTHREADS), 0, s, z);
    }
    if ((e = hipGetLastError()) != hipSuccess) return (int)e;
    // d student hidden [t, h] (+)= sum_v D[t, v] . weight[vc0 + v, h]: the dHidden GEMM of the log-probability backward,
    // partial sums carried from chunk to chunk in accumulator order, bf16 rows written by the last chunk.
    const bool first = ci == 0, last = ci == nchunks - 1;
    GemmArgs gh = dhidden_gemm(w.D, vcw + kLdPad, Tp, Wp, ld_weight, w_in_place ? nullptr : w.Wt, Vpad + kLdPad, vc0, vcw, V, T, H,
                               (uint16_t*)d_student_hidden, w.dHacc, first, last, w.counts + 1);
    gh.splits_dev = w_in_place ? w.counts + 2 : nullptr, gh.row_map = w.idx;
    e = launch_bwd_gemm(s, gh, none, split);
    if (e == hipSuccess && last) e = launch_dh_reduce(s, gh, split);
    if (e != hipSuccess) return (int)e;
  }
  return SKYRL_LMHEAD_OK;
}


size_t skyrl_lmhead_topk_workspace_bytes(int64_t T, int64_t H, int64_t V, int64_t k) {
  if (T < 1 || V < 1 || H < 1 || k < 1 || k > V || k > topk::kMaxK) return 0;
  if (T > kMaxExtent || V > kMaxExtent || H > kMaxExtent) return 0;
  return carve_topk(nullptr, T, V, k, SIZE_MAX).bytes;
}

int skyrl_lmhead_topk_logits(const void* hidden, int64_t ld_hidden, const void* weight, int64_t ld_weight, int64_t T, int64_t H,
                             int64_t V, int64_t k, float rcp_temperature, float* values, int32_t* columns, void* workspace,
                             size_t workspace_bytes, void* stream) {
  int st = check_operands(hidden, ld_hidden, weight, ld_weight, T, H, V, rcp_temperature, true);
  if (st) return st;
  if (!values || !columns) return SKYRL_LMHEAD_ERR_NULL;
  if (k < 1 || k > V || k > topk::kMaxK) return SKYRL_LMHEAD_ERR_ARG;
  const TopkWorkspace w = carve_topk(workspace, T, V, k, workspace_bytes);
  if (!workspace || workspace_bytes < w.bytes) return SKYRL_LMHEAD_ERR_WORKSPACE;
  if ((uintptr_t)workspace & 255u) return SKYRL_LMHEAD_ERR_ALIGN;

  hipStream_t s = (hipStream_t)stream;
  const int64_t block_tokens = fwd_block_tokens(w.block_tokens, ld_hidden);
  const uint16_t* Wp = (const uint16_t*)weight;
  const size_t select_lds = (size_t)topk::kSelectWaves * (size_t)(k + topk::kSelectStage) * sizeof(topk::key_t);
  hipError_t e;
  for (int64_t t0 = 0; t0 < T; t0 += block_tokens) {
    const int64_t Tb = (T - t0) < block_tokens ? (T - t0) : block_tokens;
    const int tiles_n = (int)((Tb + BN - 1) / BN);
    const uint16_t* Hp = (const uint16_t*)hidden + (size_t)t0 * (size_t)ld_hidden;
    auto chunk_shapes = [&](int64_t vrows) { return tile_shapes(Tb, H, (int)((vrows + BM - 1) / BM), compute_units()); };
    auto chunk_args = [&](int64_t v0, int64_t vrows) {
      return topk::FilterArgs{Wp + (size_t)v0 * (size_t)ld_weight, (int)ld_weight, Hp, (int)ld_hidden, (int)Tb, (int)H, (int)vrows,
                              (int)v0, rcp_temperature, (int)((vrows + BM - 1) / BM), tiles_n, kGroupM,
                              chunk_shapes(vrows).split, w.thr, w.cnt, w.cand, (int)w.cap, (float*)w.cand};
    };
    auto launch_tiles = [&](bool first, const topk::FilterArgs& a) {
      auto kernel = flagged_kernel(
          [](auto first, auto even, auto shapes) {
            if constexpr (first.value) return &topk::topk_first_tiles<even.value, shapes.value>;
            else return &topk::topk_filter_tiles<even.value, shapes.value>;
          },
          first, even_ktiles(H), chunk_shapes(a.vrows).used);
      Timed timed(kTopkFilter, s);
      hipLaunchKernelGGL(kernel, dim3((unsigned)(a.tiles_m * a.tiles_n + a.split)), dim3(NTHREADS), 0, s, a);
      return hipGetLastError();
    };
    // First chunk: one tile per CU where the stored logits allow it.
    int64_t dense = round_up(BM * ((256 + tiles_n - 1) / tiles_n), 256);
    dense = dense < kTopkDenseMin ? kTopkDenseMin : (dense > kTopkDenseMax ? kTopkDenseMax : dense);
    if (dense > w.cap) dense = w.cap;
    if (dense > V) dense = V;
    {
      const topk::FilterArgs a = chunk_args(0, dense);
      if ((e = launch_tiles(true, a)) != hipSuccess) return (int)e;
      Timed timed(kTopkSelect, s);
      auto init = dense <= 256 * topk::kInitLogits ? topk::topk_init<256> : topk::topk_init<1024>;
      hipLaunchKernelGGL(init, dim3((unsigned)Tb), dim3(dense <= 256 * topk::kInitLogits ? 256 : 1024), 0, s, (int)k,
                         (const float*)w.cand, a.tiles_m * BM, (int)dense, w.best, w.have, w.thr, w.cnt);
      if ((e = hipGetLastError()) != hipSuccess) return (int)e;
    }
    const int64_t round_columns = tiles_n < 256 ? BM * (256 / tiles_n) : BM;  // columns of a chunk whose tiles fill the CUs once
    for (int64_t v0 = dense;;) {
      int64_t width = 512 / k > 1 ? v0 * (512 / k) : v0;
      width = width < w.cap ? width : w.cap;
      width = width > round_columns ? width / round_columns * round_columns : width / BM * BM;
      if (width < BM) width = BM;
      const int64_t vrows = (V - v0) < width ? (V - v0) : width;
      const bool last = v0 + vrows >= V;
      if (vrows > 0 && (e = launch_tiles(false, chunk_args(v0, vrows))) != hipSuccess)
        return (int)e;
      {
        Timed timed(kTopkSelect, s);
        hipLaunchKernelGGL(topk::topk_select, dim3((unsigned)((Tb + topk::kSelectWaves - 1) / topk::kSelectWaves)),
                           dim3(64 * topk::kSelectWaves), select_lds, s, (int)Tb, (int)k, w.best, w.have, w.thr, w.cnt, w.cand,
                           (int)w.cap, last ? values + (size_t)t0 * (size_t)k : (float*)nullptr,
                           last ? columns + (size_t)t0 * (size_t)k : (int32_t*)nullptr);
      }
      if ((e = hipGetLastError()) != hipSuccess) return (int)e;
      v0 += vrows;
      if (last) break;
    }
  }
  return SKYRL_LMHEAD_OK;
}

namespace {
int check_topk_rows(const void* weight, int64_t ld_weight, int64_t T, int64_t H, int64_t V, int64_t k, float rcp_temperature) {
  if (!weight) return SKYRL_LMHEAD_ERR_NULL;
  if (T < 1 || V < 1 || H < 8 || H % 8 != 0 || ld_weight < H || k < 1 || k > V || k > topk::kMaxK) return SKYRL_LMHEAD_ERR_SHAPE;
  if (T > kMaxExtent || V > kMaxExtent || H > kMaxExtent || ld_weight > kMaxExtent) return SKYRL_LMHEAD_ERR_SHAPE;
  if (!aligned16(weight) || ld_weight % 8 != 0) return SKYRL_LMHEAD_ERR_ALIGN;
  if (!(rcp_temperature > 0.f) || !isfinite(rcp_temperature)) return SKYRL_LMHEAD_ERR_ARG;
  return SKYRL_LMHEAD_OK;
}
}  // namespace

int skyrl_softce_topk_fwd(const void* student_hidden, int64_t ld_student, const void* weight, int64_t ld_weight,
                          const float* teacher_values, const int32_t* teacher_columns, int64_t T, int64_t seq_len, int64_t shift,
                          int64_t H, int64_t V, int64_t k, float rcp_temperature, float* loss, float* coef, int32_t* columns,
                          void* stream) {
  int st = check_topk_rows(weight, ld_weight, T, H, V, k, rcp_temperature);
  if (st) return st;
  if (!student_hidden || !teacher_values || !teacher_columns || !loss || !coef || !columns) return SKYRL_LMHEAD_ERR_NULL;
  if (ld_student < H || ld_student > kMaxExtent || seq_len < 1 || T % seq_len != 0 || shift < 0) return SKYRL_LMHEAD_ERR_SHAPE;
  if (!aligned16(student_hidden) || ld_student % 8 != 0) return SKYRL_LMHEAD_ERR_ALIGN;
  hipStream_t s = (hipStream_t)stream;
  Timed timed(kTopkRows, s);
  hipLaunchKernelGGL(topk::topk_softce_rows, dim3((unsigned)T), dim3(topk::kRowThreads), (size_t)(2 * k + 4) * sizeof(float), s,
                     (const uint16_t*)student_hidden, (int)ld_student, (const uint16_t*)weight, (int)ld_weight, teacher_values,
                     teacher_columns, (int)T, (int)seq_len, (int)(shift % seq_len), (int)H, (int)V, (int)k, rcp_temperature, loss,
                     coef, columns);
  const hipError_t e = hipGetLastError();
  return e == hipSuccess ? SKYRL_LMHEAD_OK : (int)e;
}

int skyrl_softce_topk_bwd(const void* weight, int64_t ld_weight, const float* coef, const int32_t* columns, const float* dloss,
                          int64_t T, int64_t H, int64_t V, int64_t k, float rcp_temperature, void* d_student_hidden,
                          int64_t ld_d_student, void* stream) {
  int st = check_topk_rows(weight, ld_weight, T, H, V, k, rcp_temperature);
  if (st) return st;
  if (!coef || !columns || !dloss || !d_student_hidden) return SKYRL_LMHEAD_ERR_NULL;
  if (ld_d_student < H || ld_d_student > kMaxExtent) return SKYRL_LMHEAD_ERR_SHAPE;
  if (!aligned16(d_student_hidden) || ld_d_student % 8 != 0) return SKYRL_LMHEAD_ERR_ALIGN;
  hipStream_t s = (hipStream_t)stream;
  Timed timed(kTopkBwdRows, s);
  hipLaunchKernelGGL(topk::topk_softce_bwd_rows, dim3((unsigned)T), dim3(topk::kRowThreads), (size_t)(2 * k) * sizeof(float), s,
                     (const uint16_t*)weight, (int)ld_weight, coef, columns, dloss, (int)H, (int)V, (int)k, rcp_temperature,
                     (uint16_t*)d_student_hidden, (int)ld_d_student);
  const hipError_t e = hipGetLastError();
  return e == hipSuccess ? SKYRL_LMHEAD_OK : (int)e;
}

int skyrl_lmhead_mfma_probe(const void* operands, int workgroups, int iters, float* sink, void* stream) {
  if (!operands || !sink) return SKYRL_LMHEAD_ERR_NULL;
  if (workgroups < 1 || workgroups > 65536 || iters < 1) return SKYRL_LMHEAD_ERR_ARG;
  if (!aligned16(operands)) return SKYRL_LMHEAD_ERR_ALIGN;
  hipLaunchKernelGGL(mfma_probe, dim3((unsigned)workgroups), dim3(NTHREADS), 0, (hipStream_t)stream, (const bf16x8*)operands, iters,
                     sink);
  return (int)hipGetLastError();
}

int skyrl_lmhead_atomic_floor_probe(float* d_weight, float* d_hidden, int64_t T, int64_t H, int64_t V, void* stream) {
  if (!d_weight || !d_hidden) return SKYRL_LMHEAD_ERR_NULL;
  if (T < BN || V < BM || T % BN != 0 || V % BM != 0 || H < 1 || T > kMaxExtent || V > kMaxExtent) return SKYRL_LMHEAD_ERR_SHAPE;
  const int64_t tiles = (T / BN) * (V / BM);
  if (tiles > ((int64_t)1 << 30)) return SKYRL_LMHEAD_ERR_SHAPE;
  hipLaunchKernelGGL(atomic_floor_probe, dim3((unsigned)tiles), dim3(NTHREADS), 0, (hipStream_t)stream, d_weight, d_hidden,
                     (int)(V / BM), (int)H);
  return (int)hipGetLastError();
}

int skyrl_lmhead_device_info(int* compute_units_out, int* max_clock_khz) {
  if (!compute_units_out || !max_clock_khz) return SKYRL_LMHEAD_ERR_NULL;
  int dev = 0;
  hipError_t e = hipGetDevice(&dev);
  if (e == hipSuccess) e = hipDeviceGetAttribute(compute_units_out, hipDeviceAttributeMultiprocessorCount, dev);
  if (e == hipSuccess) e = hipDeviceGetAttribute(max_clock_khz, hipDeviceAttributeClockRate, dev);
  return e == hipSuccess ? SKYRL_LMHEAD_OK : (int)e;
}

int skyrl_lmhead_num_kernel_kinds(void) { return kNumKernelKinds; }

const char* skyrl_lmhead_kernel_name(int kind) {
  return (kind >= 0 && kind < kNumKernelKinds) ? kKernelNames[kind] : "";
}

void* skyrl_lmhead_profile_begin(void) {
  if (tl_profile) return nullptr;
  tl_profile = new Profile();
  return tl_profile;
}

int skyrl_lmhead_profile_end(void* handle, double* total_ms, int64_t* launches) {
  if (!handle || handle != (void*)tl_profile || !total_ms || !launches) return SKYRL_LMHEAD_ERR_NULL;
  Profile* p = tl_profile;
  tl_profile = nullptr;
  for (int k = 0; k < kNumKernelKinds; ++k) total_ms[k] = 0.0, launches[k] = 0;
  int status = SKYRL_LMHEAD_OK;
  for (auto& r : p->recs) {
    hipError_t e = hipEventSynchronize(r.b);
    float ms = 0.f;
    if (e == hipSuccess) e = hipEventElapsedTime(&ms, r.a, r.b);
    if (e == hipSuccess) {
      total_ms[r.kind] += ms;
      launches[r.kind] += 1;
    } else if (status == SKYRL_LMHEAD_OK) {
      status = (int)e;
    }
    (void)hipEventDestroy(r.a);
    (void)hipEventDestroy(r.b);
  }
  delete p;
  return status;
}

}  // extern "C"

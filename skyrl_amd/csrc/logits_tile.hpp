// What the square tiles (gemm_core.hpp) and the half tiles (half_tile.hpp) of logits have in common behind their products: the forward
// statistics of a tile and their layout in the scratch, and the dz values of a tile and their way into the panel.
#pragma once
#include <math.h>

#include "gemm_core.hpp"

namespace lmhead {

typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

constexpr float kLog2e = 1.4426950408889634f;
constexpr float kLn2 = 0.6931471805599453f;
constexpr float kLowestMax = -3.0e38f;
#ifndef LMHEAD_GROUP_M
#define LMHEAD_GROUP_M 4  // measured best of 2, 4, 6, 8, 16, 32 on both passes
#endif
constexpr int kGroupM = LMHEAD_GROUP_M;

// Partial statistics live in blocks of 64 tokens: [token block][part][64 tokens].  A wave of the tile kernel writes 64
// contiguous bytes (16 tokens) of one part; the merge kernel reads a token block's parts as one contiguous stream, 256 bytes
// per wave instruction.  The arrays hold nparts * round_up(T, 64) floats.
constexpr int kPartTokens = 64;
__host__ __device__ inline size_t part_index(int part, int t, int nparts) {
  return ((size_t)(t / kPartTokens) * (size_t)nparts + (size_t)part) * kPartTokens + (size_t)(t % kPartTokens);
}
__host__ __device__ inline size_t part_elems(size_t nparts, int64_t T) {
  return nparts * (size_t)((T + kPartTokens - 1) / kPartTokens * kPartTokens);
}

// N: token blocks per wave, 8 on square tiles, 4 on half tiles (half_tile.hpp).
// PAIRED (the soft cross-entropy, below): odd token blocks hold teacher rows, and their third statistic weighs the
// *student's* logit -- the same lane's accumulator one block earlier -- with the teacher's exp: sum z_student e^(z_teacher - m).
template <bool ENTROPY, bool MASKED, bool PAIRED, int N>
__device__ __forceinline__ void fwd_tile_stats(const f32x4 (&acc)[TM][N], int j, int vbase, int V, float scale2, int kq, float& m_out,
                                               float& s_out, float& e_out) {
  const int jy = (PAIRED && j % 2) ? j - 1 : j;  // j is a constant of the caller's unrolled loop
  // Two read-only passes over the accumulators (they live in AGPRs; writing scaled values back would cost a move each
  // way).  scale2 > 0, so the maximum commutes with the scaling.  The third statistic of an ordinary row is taken relative
  // to the tile's maximum, sum (z - m) e^(z - m): the exponent is at hand, and the entropy ln s - e / s then comes out of two
  // small numbers when the row is nearly deterministic, where lse - sum p z would cancel two large ones.  (The paired
  // statistic of the soft cross-entropy stays sum z_student e^(z_teacher - m): it is an expectation of another row's logit.)
  float mx = -INFINITY;
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      float x = acc[i][j][r];
      if (MASKED) {
        const int v = vbase + i * MT + kq * 4 + r;
        if (v >= V) x = -INFINITY;
      }
      mx = fmaxf(mx, x);
    }
  // Logits that are all -inf or NaN have a maximum of -inf (fmaxf passes NaN over).  Relative to a finite floor instead, the former
  // sum to 0, which the merge passes over, and a NaN among them to NaN, which it keeps.
  const float m2 = fmaxf(col_max(mx) * scale2, kLowestMax);
  float s = 0.f, e = 0.f;
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const float x = acc[i][j][r];
      const float t2 = fmaf(x, scale2, -m2);
      float p = __builtin_amdgcn_exp2f(t2);
      if (MASKED) {
        const int v = vbase + i * MT + kq * 4 + r;
        if (v >= V) p = 0.f;
      }
      s += p;
      if (ENTROPY) e = fmaf(PAIRED ? acc[i][jy][r] : t2, p, e);
    }
  s = col_sum(s);
  if (ENTROPY) e = col_sum(e);
  if (ENTROPY && s == 0.f) e = 0.f;  // the logits are all -inf: e holds 0 * -inf
  m_out = m2 * kLn2;
  s_out = s;
  e_out = PAIRED ? e * scale2 * kLn2 : e * kLn2;
}

// The shape of token tile tn of 256, by how many of a call's T tokens it holds.
__device__ __forceinline__ int shape_of_tile(int tn, int T) {
  const int rest = __builtin_amdgcn_readfirstlane(T - tn * BN);
  return rest <= BN / 2 ? kNarrow : rest <= BN * 3 / 4 ? kMedium : kSquare;
}

// Statistics of a wave's accumulators, those of part `part` (vocabulary rows 128 * part .. + 127, of nparts parts) and of the N token blocks
// from token t0 on, into the partials.
template <bool ENTROPY, bool PAIRED, int N>
__device__ __forceinline__ void fwd_epilogue(const f32x4 (&acc)[TM][N], int part, int nparts, int t0, int T, int V, float rcp_temp,
                                             float* __restrict__ part_max, float* __restrict__ part_sum,
                                             float* __restrict__ part_pz) {
  const int lane = threadIdx.x & 63;
  const int lrow = lane & 15, kq = lane >> 4;
  const int vbase = part * WM;
  const float scale2 = rcp_temp * kLog2e;
  // Whether the wave's 128 vocab rows all exist (0), partly (1: the last vocab tile) or not at all (2) is the same for the
  // whole wave: decided once, outside the unrolled loop over the token blocks.
  const int rows_kind = __builtin_amdgcn_readfirstlane(vbase + WM <= V ? 0 : (vbase < V ? 1 : 2));
  auto token_blocks = [&](auto kind) {
    constexpr int KIND = decltype(kind)::value;
#pragma unroll
    for (int j = 0; j < N; ++j) {
      const int t = t0 + j * MT + lrow;
      float m = -INFINITY, s = 0.f, e = 0.f;
      if (KIND < 2) fwd_tile_stats<ENTROPY, KIND == 1, PAIRED>(acc, j, vbase, V, scale2, kq, m, s, e);
      if (kq == 0 && t < T) {
        const size_t idx = part_index(part, t, nparts);
        part_max[idx] = m;
        part_sum[idx] = s;
        if (ENTROPY) part_pz[idx] = e;
      }
    }
  };
  if (rows_kind == 0) token_blocks(std::integral_constant<int, 0>{});
  else if (rows_kind == 1) token_blocks(std::integral_constant<int, 1>{});
  else token_blocks(std::integral_constant<int, 2>{});
}

// ------------------------------------------------------------------------------------------------------------
// Backward dz producer.  Same tile as the forward; the epilogue is purely element-wise because the row
// statistics come from the forward pass.  Formula of efficient_entropy_backward_kernel_general_d_logits_split_N
// (fused_linear_logprob_triton.py:1402-1538, the arithmetic is at :947-957 of the fused variant):
//     p  = exp(z - lse);   dz = ( g*(onehot - p) - q*p*(z - pz) ) / temperature
// written as  p * (c0 + c1*x) + onehot*g/temperature  with x the raw dot product.
// Out-of-range labels get no one-hot term but keep -p*g (model_utils.py:405-411).
// ------------------------------------------------------------------------------------------------------------
struct DzArgs {
  const uint16_t* W;
  int ldw;
  const uint16_t* Hd;
  int ldh;
  int T, H, V;
  float rcp_temp;
  const int64_t* labels;
  const float* row_lse;
  const float* row_pz;
  const float* dlogprobs;
  const float* dentropy;
  int vc0, tiles_m, tiles_n;  // first vocab row of the chunk; tiles of the chunk panel along vocab and tokens
  VocabTail tail;
  uint16_t* D;                // [T rounded up to 256, ldd]  dz, token-major; behind the tokens zeros up to the next kTokenGroup
  int ldd;
  // When not NULL: the number of tokens, <= T, as a value in device memory (what a compaction kernel counted).  T then
  // only sizes the grid: token tiles at or beyond the device-side count return at once.
  const int* T_dev;
  // When not NULL (fp32 weights): for every token whose label lies in the vocabulary, its label's dz value before the
  // rounding to bf16, fp32 [T].  That one value per token, g (1 - p) / temperature, is of order 1 where every other dz value
  // of the row is of order p; the caller adds what the bf16 product dropped of it (label_residual_update) so that the label
  // rows of dW keep fp32 accuracy.
  float* label_resid;
  // 0, or 126 - n: softmax probabilities below 2^-n are treated as zero (SKYRL_BWD_FLUSH_TINY_DZ).
  float p_shift;
  int ncu;  // CUs of the device
};

// Which vocabulary rows the 128 panel columns of a wave (columns panel0 .. panel0 + 127 in the full numbering) stand for:
// column vl is vocabulary row v0 + vl for lo <= vl < hi and carries zeros elsewhere.
struct WaveRows {
  int v0, lo, hi;
};
__device__ __forceinline__ WaveRows wave_vocab_rows(int panel0, int V, const VocabTail& tail) {
  const bool moved = tail.back > 0 && panel0 == tail.from;
  const int v0 = panel0 - (moved ? tail.back : 0);
  const int left = (tail.back > 0 && panel0 > tail.from) ? 0 : V - v0;  // no rows at all behind the moved group
  return WaveRows{v0, moved ? tail.back : 0, left < 0 ? 0 : (left < WM ? left : WM)};
}

// The A operand of a dz tile: weight rows of panel columns panel0 .. panel0 + 255, the moved group included.
__device__ __forceinline__ Operand dz_weight_rows(const uint16_t* W, int ldw, int panel0, int V, const VocabTail& tail) {
  Operand a{W, ldw, panel0, V};
  if (tail.back > 0 && panel0 == tail.from) a.row0 -= tail.back;
  if (tail.back > 0 && panel0 + WM == tail.from) a.upper_back = tail.back;
  return a;
}

// Which tile of `tile_n` tokens workgroup `id` makes, of the tokens in force (T, as dz_tile takes it); false: none.
// With a device-side count the tiles that hold tokens are numbered 0 .. tiles_m * ceil(T / tile_n) - 1, so that the hardware's
// round-robin of workgroup ids over the XCDs spreads exactly those; the other workgroups of the (static) grid return at once.
// The last tiles first: the forward ended with their weight rows, and the last-level cache still holds some of them.  Few tokens, whole
// training pass, first to last -> last to first: 778 -> 755 us at T=200, H=2048, V=151936, 469 -> 461 at T=40, H=1536; many: the same.
// SPLIT: the last round may be made of short tiles.
template <bool SPLIT>
__device__ __forceinline__ bool dz_tile_of(const DzArgs& z, int id, int tile_n, int& T, Tile& tile) {
  T = z.T_dev ? __builtin_amdgcn_readfirstlane(*z.T_dev) : z.T;
  const int tiles_n = z.T_dev ? (T + tile_n - 1) / tile_n : z.tiles_n;
  const int split = SPLIT ? split_last_round(z.tiles_m * tiles_n, z.ncu) : 0;
  if (id >= z.tiles_m * tiles_n + split) return false;
  tile = tile_of<true, SPLIT>(id, z.tiles_m, tiles_n, kGroupM, split);
  return true;
}

// Tokens that the products behind the panel contract at once, two k-tiles.  A tile of whatever width writes its tokens' rows up to the next
// multiple (dz_tile's end); what lies behind that in the panel is whatever the scratch held.
constexpr int kTokenGroup = 2 * BK;
static_assert(BN % kTokenGroup == 0, "tiles begin at whole groups");

// One tile: panel columns col0 .. + 255 of the tokens t0 .. t0 + 32 * NB - 1, of T.  NB: token blocks of 16 per wave.  SHORT: the four
// waves side by side along the tokens, panel columns col0 .. + 127 and twice the tokens.  product(a, b, acc) leaves the tile's products in
// acc, with LDS free and at least NWAVES * NB * 16 * (kDzTokRow + kDzTokBytes) bytes of it, or returns false, which ends the tile; store(v, p)
// writes one piece.
constexpr int kDzTokRow = WM * 2 + 16, kDzTokBytes = 24;
template <bool ENTGRAD, int NB, bool SHORT, class Product, class Store>
__device__ __forceinline__ void dz_tile(const DzArgs& z, int T, int col0, int t0, char* lds, Product product, Store store) {
  constexpr int WAVE_N = NB * MT;  // tokens per wave
  const uint16_t* __restrict__ W = z.W;
  const uint16_t* __restrict__ Hd = z.Hd;
  const int ldw = z.ldw, ldh = z.ldh, V = z.V, vc0 = z.vc0, ldd = z.ldd;
  const float rcp_temp = z.rcp_temp;
  const int64_t* __restrict__ labels = z.labels;
  const float* __restrict__ row_lse = z.row_lse;
  const float* __restrict__ row_pz = z.row_pz;
  const float* __restrict__ dlogprobs = z.dlogprobs;
  const float* __restrict__ dentropy = z.dentropy;
  uint16_t* __restrict__ D = z.D;

  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int wm = SHORT ? 0 : wave / WAVES_N, wn = SHORT ? wave : wave % WAVES_N;
  const int lrow = lane & 15, kq = lane >> 4;
  const int vloc_base = col0 + wm * WM;       // first column of this wave inside the chunk panel
  const WaveRows rows = wave_vocab_rows(vc0 + vloc_base, V, z.tail);
  const int vbase = rows.v0;                  // the vocabulary row of its first column
  const int tbase = t0 + wn * WAVE_N;  // first token of this wave (always inside the padded panels)
  const bool full = rows.lo == 0 && rows.hi == WM;
  const float scale2 = rcp_temp * kLog2e;

  // Per-token inputs of the epilogue.  The loads are issued here, before the mainloop, and their values are first touched
  // behind it, so the mainloop hides their latency; they are unconditional loads from a clamped token index (a load under
  // `t < T` becomes a branch with its own wait: one memory round trip per token block before the first copy is issued).  Lane
  // l loads tokens l and (square tiles) 64 + l of the wave's -- twelve registers to carry through the mainloop -- and the values reach
  // the lanes that need them (token j * 16 + lrow for every token block j) through LDS afterwards.
  constexpr int NU = (WAVE_N + 63) / 64;
  float g_[NU], q_[NU], lse_[NU], pz_[NU];
  int64_t y_[NU];
#pragma unroll
  for (int u = 0; u < NU; ++u) {
    const int t = tbase + u * 64 + lane;
    const int tc = t < T ? t : T - 1;  // T >= 1 here: a tile without a token has returned above
    g_[u] = dlogprobs[tc];
    q_[u] = ENTGRAD ? dentropy[tc] : 0.f;
    lse_[u] = row_lse[tc];
    pz_[u] = ENTGRAD ? row_pz[tc] : 0.f;
    y_[u] = labels[tc];
  }

  Operand a = dz_weight_rows(W, ldw, vc0 + col0, V, z.tail);
  if (SHORT && a.row0 >= V) a.row0 = V - 1;  // the upper half of the last 256 columns may lie behind the vocabulary: zeros, from any row
  const Operand b{Hd, ldh, t0, T};
  f32x4 acc[TM][NB];
  if (!product(a, b, acc)) return;

  constexpr int kTokRow = kDzTokRow;  // dz staging (below): the wave's token rows x (128 vocab x 2 B + pad)
  constexpr int kStage = WAVE_N * kTokRow;
  // The wave's per-token values, through a private region of LDS behind the four staging regions (LDS operations of one wave
  // execute in order, so no barrier).
  constexpr int kTokBytes = WAVE_N * kDzTokBytes;
  char* tokv = lds + NWAVES * kStage + wave * kTokBytes;  // float4 {g, q, lse, pz} per token, then the int64 labels
#pragma unroll
  for (int u = 0; u < NU; ++u) {
    if (u * 64 + lane >= WAVE_N) break;
    const f32x4 v = {g_[u], q_[u], lse_[u], pz_[u]};
    *(f32x4*)(tokv + (u * 64 + lane) * 16) = v;
    *(int64_t*)(tokv + WAVE_N * 16 + (u * 64 + lane) * 8) = y_[u];
  }
  float gs_[NB], c0_[NB], c1_[NB], lse2_[NB];
  int yrel_[NB];
#pragma unroll
  for (int j = 0; j < NB; ++j) {
    const bool valid = tbase + j * MT + lrow < T;
    const f32x4 v = *(const f32x4*)(tokv + (j * MT + lrow) * 16);
    const float g = valid ? v[0] : 0.f;
    const float q = (ENTGRAD && valid) ? v[1] : 0.f;
    lse2_[j] = valid ? v[2] * kLog2e : INFINITY;
    const float pz = (ENTGRAD && valid) ? v[3] : 0.f;
    const int64_t y = valid ? *(const int64_t*)(tokv + WAVE_N * 16 + (j * MT + lrow) * 8) : (int64_t)-1;
    const int64_t yrel64 = y - (int64_t)vbase;
    yrel_[j] = (y >= 0 && y < (int64_t)V && yrel64 >= rows.lo && yrel64 < rows.hi) ? (int)yrel64 : -1;
    gs_[j] = g * rcp_temp;
    c0_[j] = -(g - q * pz) * rcp_temp;
    c1_[j] = -q * rcp_temp * rcp_temp;
    // Optional (DzArgs::p_shift > 0): probabilities below 2^(p_shift - 126) count as zero.  The exponent is moved down by
    // p_shift so that v_exp_f32 -- which returns 0 where the result would be a denormal, below 2^-126 -- does the flush,
    // and the two coefficients carry the power of two back (exact).  Not for coefficients so large that the scaled ones
    // could overflow.
    if (z.p_shift > 0.f && fabsf(c0_[j]) < 0x1p30f && fabsf(c1_[j]) < 0x1p20f) {
      const float up = __builtin_amdgcn_exp2f(z.p_shift);
      lse2_[j] += z.p_shift;
      c0_[j] *= up;
      c1_[j] *= up;
    }
  }

  // The wave's 128 x WAVE_N dz block leaves through LDS so that the panel is written with 16-byte stores: a lane holds four
  // consecutive vocab rows of one token, an 8-byte piece of a D row.  mainloop() left LDS free and every wave uses a
  // private region, so no barrier is needed (LDS operations of one wave execute in order).  The stores are marked
  // non-temporal: the panel is a gigabyte that is read back only by the next launch, and letting it displace the operand
  // panels from L2 costs the mainloops of the neighbouring tiles more than the stores themselves.
  char* stage = lds + wave * kStage;
  // Every staging address is one per-lane base plus a compile-time constant (an immediate of the LDS instruction), and the
  // panel rows are walked with one running pointer: written as (j * 16 + row) * pitch the compiler keeps eight row indices
  // alive across the whole epilogue and spills them, and a spill reload waits for vmcnt(0) -- i.e. for every panel store in flight.
  char* const st_w = stage + lrow * kTokRow + kq * 8;                      // + (j * MT) * kTokRow + i * MT * 2
  const char* const st_r = stage + (lane >> 4) * kTokRow + (lane & 15) * 16;  // + (j * MT + it * 4) * kTokRow
  uint16_t* d_row = D + (size_t)(tbase + (lane >> 4)) * (size_t)ldd + vloc_base + (lane & 15) * 8;  // four rows further per store
  const size_t d_step = (size_t)4 * (size_t)ldd;

  // A token block j (16 token rows x 128 vocab, 4 KiB of the staging region) is complete after its eight i-steps; its 256
  // 16-byte pieces (4 per lane; 16 lanes cover one token row of 256 bytes) go out in the middle of block j + 1, so that the
  // read-back and the store issue hide behind that block's arithmetic instead of forming a tail of their own.  Blocks are
  // flushed in order, j = 0 .. NB - 1.
  auto flush_block = [&](int j) {
#pragma unroll
    for (int it = 0; it < 4; ++it) {
      const u32x4 v = *(const u32x4*)(st_r + (j * MT + it * 4) * kTokRow);
      store(v, (u32x4*)d_row);
      d_row += d_step;
    }
  };
  // One token block: eight i-steps of four values per lane.  What is the same for the whole wave -- rows past the
  // vocabulary's end (RAGGED: only the last vocab tile), a label of some token inside the wave's rows (LABEL, decided per
  // token block by a ballot), the fp32 residual of the label's value (fp32 operands only) -- is decided once outside the
  // unrolled loops: as tests inside them they cost three branches per i-step, a third of the epilogue's time.
  auto token_block = [&](int j, auto ragged, auto label) {
    constexpr bool RAGGED = decltype(ragged)::value, LABEL = decltype(label)::value;
    const float gs = gs_[j], c0 = c0_[j], c1 = c1_[j], lse2 = lse2_[j];
    const int yrel = yrel_[j];
#pragma unroll
    for (int i = 0; i < TM; ++i) {
      float d[4];
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const float x = acc[i][j][r];
        const float p = __builtin_amdgcn_exp2f(fmaf(x, scale2, -lse2));
        d[r] = ENTGRAD ? p * fmaf(c1, x, c0) : p * c0;
      }
      const int vl = i * MT + kq * 4;  // vocab row inside the wave block; this lane holds vl .. vl+3
      if (LABEL) {
#pragma unroll
        for (int r = 0; r < 4; ++r)
          if (yrel == vl + r) d[r] += gs;
      }
      if (RAGGED) {
#pragma unroll
        for (int r = 0; r < 4; ++r)
          if (vl + r < rows.lo || vl + r >= rows.hi) d[r] = 0.f;
      }
      f32x4 v4 = {d[0], d[1], d[2], d[3]};
      const bf16x4 b4 = __builtin_convertvector(v4, bf16x4);
      *(uint2*)(st_w + (j * MT) * kTokRow + i * (MT * 2)) = *(const uint2*)&b4;
      if (LABEL && z.label_resid) {
#pragma unroll
        for (int r = 0; r < 4; ++r)
          if (yrel == vl + r) z.label_resid[tbase + j * MT + lrow] = d[r];
      }
      if (i == TM / 2 - 1 && j > 0) flush_block(j - 1);
    }
  };
  std::true_type yes;
  std::false_type no;
  if (__builtin_amdgcn_readfirstlane((int)full)) {
#pragma unroll
    for (int j = 0; j < NB; ++j) {
      if (__any(yrel_[j] >= 0)) token_block(j, no, yes);  // some token of this block has its label inside the wave's rows
      else token_block(j, no, no);
    }
  } else {
#pragma unroll
    for (int j = 0; j < NB; ++j) token_block(j, yes, yes);
  }
  flush_block(NB - 1);
  // The products behind the panel run over whole groups of tokens: a medium tile, whose tokens end in its second group, leaves zeros in
  // what remains of that.
  constexpr int kTokens = WAVE_N * (SHORT ? NWAVES : WAVES_N), kRest = (kTokens + kTokenGroup - 1) / kTokenGroup * kTokenGroup - kTokens;
  static_assert(!SHORT || kRest == 0, "the rows below are those of two waves side by side");
  if constexpr (kRest > 0) {
    uint16_t* zero_row = D + (size_t)(t0 + WAVES_N * WAVE_N + wn * (kRest / WAVES_N) + (lane >> 4)) * (size_t)ldd + vloc_base + (lane & 15) * 8;
#pragma unroll
    for (int it = 0; it < kRest / WAVES_N / 4; ++it) {
      store(u32x4{0u, 0u, 0u, 0u}, (u32x4*)zero_row);
      zero_row += d_step;
    }
  }
}

}  // namespace lmhead

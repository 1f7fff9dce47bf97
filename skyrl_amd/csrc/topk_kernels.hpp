// Device code of the top-k draft loss of multi-token prediction (skyrl/backends/skyrl_train/mtp/soft_ce.py:243-341,
// _VocabParallelTopkSoftCE on one vocabulary shard): the k largest teacher logits of every token straight from the teacher's
// hidden states -- no [T, V] logits tensor -- and the soft cross-entropy of the student over those k columns.
//
//   topk_first_tiles    one 256(vocab) x 256(token) logits tile of the first vocabulary chunk, the forward's GEMM; the logits
//                       themselves are stored, [T, chunk] fp32.
//   topk_filter_tiles   the same of a later chunk; the epilogue compares every logit with the token's threshold (the k-th
//                       largest logit among the columns of earlier chunks, a lower bound of the final one) and appends the few
//                       that pass to the token's candidate list.
//   topk_init           one workgroup per token: the k best of the first chunk's logits and the first threshold.
//   topk_select         one wave per token: merges the chunk's candidates into the token's running k best, raises its
//                       threshold, empties the candidate list.  After the last chunk it also writes the k logits and their
//                       columns, best first.
//   topk_softce_rows    one workgroup per token: the student's logits at the (rolled) teacher's k columns, k dot products with
//                       gathered weight rows; softmax of both over the k columns; loss and d loss / d student logits.
//   topk_softce_bwd_rows  one workgroup per token: d student hidden = upstream * sum_j coef[j] * weight[column j] / temperature.
//
// Order of logits: higher value first, lower column first among equal values; -0.0 sorts below +0.0.  That order is total,
// so the k best of a row are a unique set whatever order the candidates arrive in, and the results are reproducible although
// the candidate lists are filled with atomic counters.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "gemm_core.hpp"
#include "logits_tile.hpp"

namespace topk {
using namespace lmhead;

typedef unsigned long long key_t;

// Bits of a float such that unsigned comparison orders them as the floats order (negative values below positive ones).
__device__ __forceinline__ uint32_t ordered_bits(float z) {
  const uint32_t b = __float_as_uint(z);
  return b ^ ((b >> 31) ? 0xffffffffu : 0x80000000u);
}
__device__ __forceinline__ float value_of_bits(uint32_t o) {
  return __uint_as_float(o ^ ((o >> 31) ? 0x80000000u : 0xffffffffu));
}
// A logit and its column as one key: a larger key is a better candidate.
__device__ __forceinline__ key_t make_key(float z, int column) { return ((key_t)ordered_bits(z) << 32) | (key_t)(uint32_t)(~column); }
__device__ __forceinline__ float key_value(key_t k) { return value_of_bits((uint32_t)(k >> 32)); }
__device__ __forceinline__ int key_column(key_t k) { return (int)(~(uint32_t)k); }

struct FilterArgs {
  const uint16_t* W;   // first weight row of the chunk
  int ldw;
  const uint16_t* Hd;  // hidden rows of the token block
  int ldh;
  int T, H;
  int vrows;           // weight rows of the chunk that exist (the last tile may overhang them)
  int v0;              // column number of the chunk's first row
  float rcp_temp;
  int tiles_m, tiles_n, group_m;
  int split;           // how many of the tiles are made as short ones (tile_shapes)
  const float* thr;    // [T] threshold per token, -inf while fewer than k columns have been seen
  unsigned* cnt;       // [T] candidates appended in this launch
  key_t* cand;         // [T, cap]
  int cap;             // >= columns of a chunk, so that a list cannot overflow
  float* dense;        // first chunk: its logits [T, tiles_m * 256]
};

// The tile of SHAPE whose first row and token are vtile and ttile.
template <bool DENSE, bool EVEN, int SHAPE>
__device__ __forceinline__ void topk_tile(const FilterArgs& a, int vtile, int ttile, char* lds) {
  constexpr int N = wave_cols(SHAPE);
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int wm = wave / waves_n(SHAPE), wn = wave % waves_n(SHAPE);
  const int lrow = lane & 15, kq = lane >> 4;
  // The tokens' thresholds (fixed for the launch): unconditional loads from a clamped index, issued before the mainloop and
  // first touched behind it -- a load under `t < T` is a branch with its own wait, eight memory round trips in a row.
  const int tbase = ttile + wn * (N * MT) + lrow;  // this lane's token of block j: 16 j further
  float th[N];
#pragma unroll
  for (int j = 0; j < N; ++j) {
    const int t = tbase + j * MT;
    th[j] = DENSE ? 0.f : a.thr[t < a.T ? t : a.T - 1];
  }

  // The upper half of the last tile may lie behind the chunk's rows: multiplied from any row, and dropped below.
  Operand oa{a.W, a.ldw, SHAPE == kShort && vtile >= a.vrows ? a.vrows - 1 : vtile, a.vrows};
  Operand ob{a.Hd, a.ldh, ttile, a.T};
  f32x4 acc[TM][N];
  tile_product<SHAPE, EVEN>(oa, ob, a.H / BK, lds, acc);

  const int vbase = vtile + wm * WM;  // first row of this wave inside the chunk
  if (vbase >= a.vrows) return;
  const float s = a.rcp_temp;
  if (DENSE) {  // columns past vrows are stored as they come (copies of the last row) and not read
    const size_t pitch = (size_t)a.tiles_m * BM;
#pragma unroll
    for (int j = 0; j < N; ++j) {
      const int t = tbase + j * MT;
      if (t >= a.T) continue;
      float* row = a.dense + (size_t)t * pitch + vbase + kq * 4;
#pragma unroll
      for (int i = 0; i < TM; ++i) *(f32x4*)(row + i * MT) = acc[i][j] * s;
    }
    return;
  }
#pragma unroll
  for (int j = 0; j < N; ++j) {
    const int t = tbase + j * MT;
    if (t >= a.T) th[j] = NAN;  // rows past the last token never pass: every comparison with NaN is false
  }
  // A lane holds 32 logits of each of its eight tokens.  First sweep: the largest of the 32 against the threshold (rounding is
  // monotone and s > 0, so the scaled maximum is the maximum of the scaled values); a wave-wide vote skips the tokens of which nothing
  // passes, and for the others every logit that passes becomes a bit of a word.  Then one atomic add per lane and token reserves
  // as many slots of the token's list -- eight independent atomics in flight, one round trip per tile -- and a second sweep stores the
  // keys.  A lane has about one passing logit of its 256 while thresholds are young: it finds them by their bits, and the values,
  // which cannot be indexed in registers, through its own 128 bytes of LDS (free behind the mainloop; no other lane reads them).
  // At T=1800, H=2048, k=32, tests and branches block of four by block of four -> bits: 59 -> 48 us for a tile of the chunk behind the
  // first 8192 columns, 48 -> 46 for one of the chunk behind that.
  uint32_t exists = 0xffffffffu;  // which of the lane's logits do, as the bits below: the chunk's last rows may end inside the tile
  if (vbase + WM > a.vrows) {
#pragma unroll
    for (int x = 0; x < TM * 4; ++x)
      if (vbase + (x / 4) * MT + kq * 4 + x % 4 >= a.vrows) exists &= ~(0x80000000u >> x);
  }
  uint32_t hit[N];  // bit 31 - (i * 4 + r)
#pragma unroll
  for (int j = 0; j < N; ++j) {
    float m = acc[0][j][0];
#pragma unroll
    for (int x = 1; x < TM * 4; ++x) m = fmaxf(m, acc[x / 4][j][x % 4]);
    hit[j] = 0;
    if (!__any(m * s >= th[j])) continue;
#pragma unroll
    for (int i = 0; i < TM; ++i) {
      const f32x4 z = acc[i][j] * s;
      // A comparison's result is a carry two wait states later at the earliest, which the compiler cannot keep inside an assembly
      // statement: four comparisons, then four additions, so that three instructions lie between the two of a pair.
      uint64_t p0, p1, p2, p3;
      asm("v_cmp_ge_f32_e64 %1, %5, %9\n\tv_cmp_ge_f32_e64 %2, %6, %9\n\tv_cmp_ge_f32_e64 %3, %7, %9\n\tv_cmp_ge_f32_e64 %4, %8, %9\n\t"
          "v_addc_co_u32_e64 %0, vcc, %0, %0, %1\n\tv_addc_co_u32_e64 %0, vcc, %0, %0, %2\n\t"
          "v_addc_co_u32_e64 %0, vcc, %0, %0, %3\n\tv_addc_co_u32_e64 %0, vcc, %0, %0, %4"
          : "+v"(hit[j]), "=&s"(p0), "=&s"(p1), "=&s"(p2), "=&s"(p3)
          : "v"(z[0]), "v"(z[1]), "v"(z[2]), "v"(z[3]), "v"(th[j])
          : "vcc");
    }
    hit[j] &= exists;
  }
  unsigned base[N];
#pragma unroll
  for (int j = 0; j < N; ++j) {
    const int t = tbase + j * MT;
    base[j] = hit[j] ? atomicAdd(a.cnt + t, (unsigned)__popc(hit[j])) : 0u;
  }
  char* const mine = lds + wave * (TM * 4 * 64 * 4) + lane * 16;  // [i][lane] pieces of four values
#pragma unroll
  for (int j = 0; j < N; ++j) {
    if (hit[j] == 0) continue;
    key_t* list = a.cand + (size_t)(tbase + j * MT) * (size_t)a.cap;
#pragma unroll
    for (int i = 0; i < TM; ++i) *(f32x4*)(mine + i * 1024) = acc[i][j];
    unsigned slot = base[j];
    for (uint32_t left = hit[j]; left; ++slot) {
      const int x = __clz((int)left);
      left &= ~(0x80000000u >> x);
      const float z = *(const float*)(mine + (x >> 2) * 1024 + (x & 3) * 4) * s;
      if (slot < (unsigned)a.cap) list[slot] = make_key(z, a.v0 + vbase + (x >> 2) * MT + kq * 4 + (x & 3));
    }
  }
}

template <bool DENSE, bool EVEN, bool SHAPES>
__device__ __forceinline__ void topk_tile_of_workgroup(const FilterArgs& a, char* lds) {
  const Tile t = tile_of<false, SHAPES>(blockIdx.x, a.tiles_m, a.tiles_n, a.group_m, a.split);
  const int v = t.tm * BM, n = t.tn * BN;
  if constexpr (SHAPES) {
    const int shape = shape_of_tile(t.tn, a.T);
    if (shape == kNarrow) {  // of the two workgroups of a split tile the first makes it
      if (t.half < 1) topk_tile<DENSE, EVEN, kNarrow>(a, v, n, lds);
      return;
    }
    if (t.half >= 0) return topk_tile<DENSE, EVEN, kShort>(a, v + t.half * WM, n, lds);
    if (shape == kMedium) return topk_tile<DENSE, EVEN, kMedium>(a, v, n, lds);
  }
  topk_tile<DENSE, EVEN, kSquare>(a, v, n, lds);
}

template <bool EVEN, bool SHAPES>
__global__ __launch_bounds__(NTHREADS) void topk_first_tiles(const FilterArgs a) {
  __shared__ __attribute__((aligned(1024))) char lds[LDS_BYTES];
  topk_tile_of_workgroup<true, EVEN, SHAPES>(a, lds);
}

template <bool EVEN, bool SHAPES>
__global__ __launch_bounds__(NTHREADS) void topk_filter_tiles(const FilterArgs a) {
  __shared__ __attribute__((aligned(1024))) char lds[LDS_BYTES];
  topk_tile_of_workgroup<false, EVEN, SHAPES>(a, lds);
}

// Smallest key of the wave's values, in every lane.
__device__ __forceinline__ key_t wave_min_key(key_t v) {
#pragma unroll
  for (int o = 32; o >= 1; o >>= 1) {
    const key_t w = __shfl_xor(v, o, 64);
    v = w < v ? w : v;
  }
  return v;
}

constexpr int kSelectWaves = 4;
constexpr int kMaxK = 1024;

// LDS operations of one wave execute in order; the fences only keep the compiler from caching entries that another lane has
// rewritten.
__device__ __forceinline__ void wave_lds_fence() { __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront"); }

constexpr int kInRegisters = 512;  // keys that keep_largest() takes into registers

// The k largest of the M > k keys in `list` (LDS, unique keys), moved to its front by the calling wave: a bisection over the key
// bits finds a threshold that exactly k keys reach (a count of the keys per bit, usually 20 to 30 bits until it is exact).  BATCHES: M <= 64 BATCHES,
// and a lane holds its keys in registers, so that a count is a few comparisons and votes; 0: any M, from LDS, with a sum over the lanes per bit.  What
// bounds it is that chain, a wave per token.  From LDS -> registers, T=1800, k=32: topk_init (33 keys a token) 28 -> 22 us,
// topk_select (300) 20 -> 10; pass 1032 -> 1013, at k=128, T=600, H=1024, V=128000 421 -> 405.
template <int BATCHES>
__device__ __forceinline__ void keep_largest_of(key_t* list, int M, int k, int lane) {
  if constexpr (BATCHES == 0) {
    key_t reach = 0;  // grows bit by bit while at least k keys reach it; done when exactly k do
    for (int b = 63; b >= 0; --b) {
      const key_t trial = reach | ((key_t)1 << b);
      int c = 0;
      for (int e = lane; e < M; e += 64) c += list[e] >= trial ? 1 : 0;
#pragma unroll
      for (int o = 32; o >= 1; o >>= 1) c += __shfl_xor(c, o, 64);
      if (c >= k) {
        reach = trial;
        if (c == k) break;
      }
    }
    int w = 0;  // in-place compaction: a step reads 64 entries and writes at or below where it read
    for (int base = 0; base < M; base += 64) {
      const int e = base + lane;
      const key_t x = e < M ? list[e] : 0;
      const bool keep = e < M && x >= reach;
      const unsigned long long mask = __ballot(keep);
      wave_lds_fence();
      if (keep) list[w + __popcll(mask & (((key_t)1 << lane) - 1))] = x;
      w += (int)__popcll(mask);
      wave_lds_fence();
    }
  } else {
    key_t x[BATCHES];
#pragma unroll
    for (int u = 0; u < BATCHES; ++u) x[u] = u * 64 + lane < M ? list[u * 64 + lane] : 0;  // 0 reaches no trial
    key_t reach = 0;
    for (int b = 63; b >= 0; --b) {
      const key_t trial = reach | ((key_t)1 << b);
      int c = 0;
#pragma unroll
      for (int u = 0; u < BATCHES; ++u) c += (int)__popcll(__ballot(x[u] >= trial));
      if (c >= k) {
        reach = trial;
        if (c == k) break;
      }
    }
    wave_lds_fence();
    int w = 0;
#pragma unroll
    for (int u = 0; u < BATCHES; ++u) {
      const bool keep = u * 64 + lane < M && x[u] >= reach;
      const unsigned long long mask = __ballot(keep);
      if (keep) list[w + __popcll(mask & (((key_t)1 << lane) - 1))] = x[u];
      w += (int)__popcll(mask);
    }
    wave_lds_fence();
  }
}
__device__ __forceinline__ void keep_largest(key_t* list, int M, int k, int lane) {
  if (M <= 64) keep_largest_of<1>(list, M, k, lane);
  else if (M <= 256) keep_largest_of<4>(list, M, k, lane);
  else if (M <= kInRegisters) keep_largest_of<8>(list, M, k, lane);
  else keep_largest_of<0>(list, M, k, lane);
}

constexpr int kSelectStage = 1024;   // candidates one bulk round takes into LDS, behind the list
// Fewer candidates than this are inserted one by one, each of which costs a search for the worst entry: where a bulk round works in registers
// (keep_largest) it is the cheaper from four on (topk_select with 27 candidates, k=32, T=1800: 22.9 -> 7.0 us; pass 969 -> 953, at k=128 392 -> 372), else from 96.
constexpr int kSelectBulkMin = 96, kSelectBulkMinInRegisters = 4;

// best: [T, k] running lists (unordered), have: [T] entries of the list that are filled.  One wave per token; the list lives
// in LDS while the wave works on it.  Many candidates (the first chunks, a large k, adversarial data) are merged in bulk: up to
// kSelectStage of them are put behind the list and keep_largest() brings the best to the front.  A few candidates are inserted one by one, each replacing the worst
// entry.  With `final_vals` the finished list is written out best first.
__global__ __launch_bounds__(64 * kSelectWaves) void topk_select(int T, int k, key_t* __restrict__ best, unsigned* __restrict__ have,
                                                                 float* __restrict__ thr, unsigned* __restrict__ cnt,
                                                                 const key_t* __restrict__ cand, int cap,
                                                                 float* __restrict__ final_vals, int* __restrict__ final_idx) {
  extern __shared__ key_t sm_list[];  // kSelectWaves * (k + kSelectStage) keys
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int t = blockIdx.x * kSelectWaves + wave;
  if (t >= T) return;  // whole waves leave; no barrier below
  key_t* list = sm_list + (size_t)wave * (size_t)(k + kSelectStage);
  key_t* gl = best + (size_t)t * (size_t)k;
  int n_have = (int)have[t];
  for (int e = lane; e < n_have; e += 64) list[e] = gl[e];
  auto lds_fence = []() { wave_lds_fence(); };
  lds_fence();
  const unsigned n_raw = cnt[t];
  const int n = (int)(n_raw < (unsigned)cap ? n_raw : (unsigned)cap);

  // the worst entry of a full list: its key and position
  key_t worst = 0;
  int worst_pos = 0;
  auto find_worst = [&]() {
    key_t mine = ~(key_t)0;
    for (int e = lane; e < k; e += 64) mine = list[e] < mine ? list[e] : mine;
    worst = wave_min_key(mine);
    int pos = -1;
    for (int e = lane; e < k; e += 64)
      if (list[e] == worst) pos = e;  // keys are unique (columns are)
    const unsigned long long owner = __ballot(pos >= 0);
    worst_pos = __shfl(pos, (int)__ffsll((long long)owner) - 1, 64);
  };
  const key_t* cl = cand + (size_t)t * (size_t)cap;
  int done = 0;
  const int bulk_min = n_have + n <= kInRegisters ? kSelectBulkMinInRegisters : kSelectBulkMin;
  while (n - done >= bulk_min) {
    const int take = (n - done) < kSelectStage ? (n - done) : kSelectStage;
    for (int e = lane; e < take; e += 64) list[n_have + e] = cl[done + e];
    lds_fence();
    const int M = n_have + take;
    done += take;
    if (M <= k) {
      n_have = M;
      continue;
    }
    keep_largest(list, M, k, lane);
    n_have = k;
  }
  if (n_have == k) find_worst();

  for (int c0 = done; c0 < n; c0 += 64) {
    const bool in = c0 + lane < n;
    const key_t c = in ? cl[c0 + lane] : 0;
    unsigned long long pending = __ballot(in && (n_have < k || c > worst));
    while (pending) {
      const int src = (int)__ffsll((long long)pending) - 1;
      pending &= pending - 1;
      const key_t x = __shfl(c, src, 64);
      if (n_have < k) {
        if (lane == 0) list[n_have] = x;
        lds_fence();
        ++n_have;
        if (n_have == k) {
          find_worst();
          pending &= __ballot(c > worst);
        }
      } else if (x > worst) {
        if (lane == 0) list[worst_pos] = x;
        lds_fence();
        find_worst();
        pending &= __ballot(c > worst);
      }
    }
  }

  if (!final_vals) {
    for (int e = lane; e < n_have; e += 64) gl[e] = list[e];
    if (lane == 0) {
      have[t] = (unsigned)n_have;
      thr[t] = n_have == k ? key_value(worst) : -INFINITY;
      cnt[t] = 0u;
    }
    return;
  }
  // Final pass: rank every entry among the k (number of better keys) and write value and column at that rank.
  for (int e = lane; e < k; e += 64) {
    if (e < n_have) {
      const key_t mine = list[e];
      int rank = 0;
      for (int o = 0; o < n_have; ++o) rank += list[o] > mine ? 1 : 0;
      final_vals[(size_t)t * (size_t)k + rank] = key_value(mine);
      final_idx[(size_t)t * (size_t)k + rank] = key_column(mine);
    } else {
      // Fewer than k comparable logits: the row holds NaNs (a NaN never passes the filter's comparison).  torch.topk ranks
      // NaN first and the loss built on it is NaN (mtp/soft_ce.py:258-305); the ranks nobody filled say the same.
      final_vals[(size_t)t * (size_t)k + e] = NAN;
      final_idx[(size_t)t * (size_t)k + e] = 0;
    }
  }
  if (lane == 0) cnt[t] = 0u;
}

// The first chunk's logits [T, pitch] of one token per workgroup -> its k best (unordered) and the first threshold.  A thread
// keeps 32 logits in registers.
//   k <= 128: the k-th largest of the threads' maxima is a lower bound of the k-th largest logit that few others reach (about 33
//     for k = 32, 180 for k = 128); one wave finds it with ballots, the logits that reach it are listed in LDS and keep_largest()
//     takes the k best of them.
//   larger k, or so many equal logits that the list overflows: a bisection over the bits of the values (all threads count, one
//     barrier per bit, fewer when the count comes out exact), and among equal values one over the columns.
// Bound by the read of the logits.  Filling the lists through the candidate path instead (every logit passes while there is no
// threshold) took 93 us for 32 tiles of 1024 columns at T=1800; first tiles of 8192 columns and this kernel take 61 + 22 us (the bisection alone: 61 + 45).
constexpr int kInitLogits = 32;  // per thread
constexpr int kInitList = 1024;
constexpr int kInitListK = 128;

template <int THREADS>
__global__ __launch_bounds__(THREADS) void topk_init(int k, const float* __restrict__ dense, int pitch, int columns,
                                                     key_t* __restrict__ best, unsigned* __restrict__ have,
                                                     float* __restrict__ thr, unsigned* __restrict__ cnt) {
  __shared__ int red[2][THREADS / 64];
  __shared__ unsigned filled;
  __shared__ uint32_t smallest[THREADS / 64];
  __shared__ uint32_t maxima[THREADS];
  __shared__ key_t listed[kInitList];
  const int t = blockIdx.x, tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const float* row = dense + (size_t)t * (size_t)pitch;
  uint32_t o[kInitLogits];  // ordered bits; 0 is below every number and stands for "no logit here" (a NaN, or past the columns)
#pragma unroll
  for (int u = 0; u < kInitLogits / 4; ++u) {
    const int c = (u * THREADS + tid) * 4;
    f32x4 z = {NAN, NAN, NAN, NAN};
    if (c < columns) z = *(const f32x4*)(row + c);  // the pitch is a multiple of four
#pragma unroll
    for (int e = 0; e < 4; ++e) o[u * 4 + e] = (c + e < columns && z[e] == z[e]) ? ordered_bits(z[e]) : 0u;
  }
  if (tid == 0) filled = 0;
  if (k <= kInitListK) {
    uint32_t mx = 0;
#pragma unroll
    for (int e = 0; e < kInitLogits; ++e) mx = o[e] > mx ? o[e] : mx;
    maxima[tid] = mx;
    __syncthreads();
    if (wave == 0) {
      uint32_t m[THREADS / 64], bound = 0;
#pragma unroll
      for (int w = 0; w < THREADS / 64; ++w) m[w] = maxima[w * 64 + lane];
      for (int b = 31; b >= 0; --b) {
        const uint32_t trial = bound | (1u << b);
        int c = 0;
#pragma unroll
        for (int w = 0; w < THREADS / 64; ++w) c += __popcll(__ballot(m[w] >= trial));
        if (c >= k) {
          bound = trial;
          if (c == k) break;
        }
      }
      if (lane == 0) smallest[0] = bound > 0 ? bound : 1u;  // fewer than k threads hold a logit: everything is listed
    }
    __syncthreads();
    const uint32_t bound = smallest[0];
#pragma unroll
    for (int e = 0; e < kInitLogits; ++e) {
      if (o[e] >= bound) {
        const unsigned pos = atomicAdd(&filled, 1u);
        if (pos < (unsigned)kInitList) listed[pos] = ((key_t)o[e] << 32) | (key_t)(uint32_t)(~(((e / 4) * THREADS + tid) * 4 + e % 4));
      }
    }
    __syncthreads();
    const int M = (int)filled;
    if (M <= kInitList) {
      if (wave != 0) return;
      if (M > k) keep_largest(listed, M, k, lane);
      const int kept = M < k ? M : k;
      key_t worst = ~(key_t)0;
      for (int e = lane; e < kept; e += 64) {
        const key_t x = listed[e];
        best[(size_t)t * (size_t)k + e] = x;
        worst = x < worst ? x : worst;
      }
      worst = wave_min_key(worst);
      if (lane == 0) have[t] = (unsigned)kept, thr[t] = kept == k ? key_value(worst) : -INFINITY, cnt[t] = 0u;
      return;
    }
    __syncthreads();  // everybody has read `filled`
    if (tid == 0) filled = 0;
  }
  int parity = 0;
  auto total = [&](int mine) {  // sum over the workgroup, in every thread
#pragma unroll
    for (int x = 32; x >= 1; x >>= 1) mine += __shfl_xor(mine, x, 64);
    if (lane == 0) red[parity][wave] = mine;
    __syncthreads();
    int sum = 0;
    for (int w = 0; w < THREADS / 64; ++w) sum += red[parity][w];
    parity ^= 1;
    return sum;
  };
  auto reaching = [&](uint32_t limit) {
    int c = 0;
#pragma unroll
    for (int e = 0; e < kInitLogits; ++e) c += o[e] >= limit ? 1 : 0;
    return total(c);
  };
  uint32_t reach = 1;
  int count = reaching(1);
  const int n = count;
  if (count > k) {
    reach = 0;
    for (int b = 31; b >= 0 && count != k; --b) {
      const uint32_t trial = reach | (1u << b);
      const int c = reaching(trial);
      if (c >= k) reach = trial, count = c;
    }
  }
  int column_limit = 0x7fffffff;
  if (count > k) {  // several logits equal the k-th largest: the lower columns win
    const int wanted = k - reaching(reach + 1);
    int lo = 0, hi = columns;  // smallest limit below which at least `wanted` of them lie
    while (lo < hi) {
      const int mid = (lo + hi) >> 1;
      int c = 0;
#pragma unroll
      for (int e = 0; e < kInitLogits; ++e) c += (o[e] == reach && ((e / 4) * THREADS + tid) * 4 + e % 4 < mid) ? 1 : 0;
      if (total(c) >= wanted) hi = mid; else lo = mid + 1;
    }
    column_limit = lo;
  }
  uint32_t low = 0xffffffffu;
#pragma unroll
  for (int e = 0; e < kInitLogits; ++e) {
    const int c = ((e / 4) * THREADS + tid) * 4 + e % 4;
    if (o[e] > reach || (o[e] == reach && c < column_limit)) {
      low = o[e] < low ? o[e] : low;
      const unsigned pos = atomicAdd(&filled, 1u);
      best[(size_t)t * (size_t)k + pos] = ((key_t)o[e] << 32) | (key_t)(uint32_t)(~c);
    }
  }
#pragma unroll
  for (int x = 32; x >= 1; x >>= 1) {
    const uint32_t w = __shfl_xor(low, x, 64);
    low = w < low ? w : low;
  }
  if (lane == 0) smallest[wave] = low;
  __syncthreads();
  if (tid == 0) {
    for (int w = 1; w < THREADS / 64; ++w) low = smallest[w] < low ? smallest[w] : low;
    have[t] = (unsigned)(n < k ? n : k);
    thr[t] = n >= k ? value_of_bits(low) : -INFINITY;
    cnt[t] = 0u;
  }
}

// fp32 dot product of two bf16 rows, the wave's lanes taking 16-byte pieces; the sum in every lane.
__device__ __forceinline__ float wave_dot_bf16(const uint16_t* __restrict__ x, const uint16_t* __restrict__ y, int H, int lane) {
  float dot = 0.f;
  for (int c = lane * 8; c < H; c += 64 * 8) {
    const uint4 xv = *(const uint4*)(x + c);
    const uint4 yv = *(const uint4*)(y + c);
    const uint32_t xx[4] = {xv.x, xv.y, xv.z, xv.w};
    const uint32_t yy[4] = {yv.x, yv.y, yv.z, yv.w};
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      dot = fmaf(__uint_as_float(xx[q] << 16), __uint_as_float(yy[q] << 16), dot);
      dot = fmaf(__uint_as_float(xx[q] & 0xffff0000u), __uint_as_float(yy[q] & 0xffff0000u), dot);
    }
  }
#pragma unroll
  for (int o = 32; o >= 1; o >>= 1) dot += __shfl_xor(dot, o, 64);
  return dot;
}

constexpr int kRowThreads = 256;

__device__ __forceinline__ float block_reduce(float v, bool take_max, float* sm) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
#pragma unroll
  for (int o = 32; o >= 1; o >>= 1) {
    const float w = __shfl_xor(v, o, 64);
    v = take_max ? fmaxf(v, w) : v + w;
  }
  __syncthreads();  // sm may still be read from the previous reduction
  if (lane == 0) sm[wave] = v;
  __syncthreads();
  float r = sm[0];
  for (int w = 1; w < kRowThreads / 64; ++w) r = take_max ? fmaxf(r, sm[w]) : r + sm[w];
  return r;
}

// Token b * seq_len + s is scored against the teacher's list of token b * seq_len + (s + shift) mod seq_len
// (torch.roll of the [B, S, k] top-k result by -shift, soft_ce.py:277-279).
//   t_p = softmax(teacher values), q_s = softmax(student values) over the k columns,
//   loss = -sum_j t_p[j] log q_s[j]   (soft_ce.py:282-300),   coef[j] = q_s[j] - t_p[j]   (:309)
__global__ __launch_bounds__(kRowThreads) void topk_softce_rows(const uint16_t* __restrict__ student, int lds_,
                                                                const uint16_t* __restrict__ W, int ldw,
                                                                const float* __restrict__ t_vals, const int* __restrict__ t_idx,
                                                                int T, int seq_len, int shift, int H, int V, int k, float rcp_temp,
                                                                float* __restrict__ loss, float* __restrict__ coef,
                                                                int* __restrict__ columns) {
  extern __shared__ float sm_rows[];  // k student values, k teacher values, 4 reduction slots
  float* sv = sm_rows;
  float* tv = sm_rows + k;
  float* red = sm_rows + 2 * k;
  const int t = blockIdx.x;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int row = t / seq_len, pos = t - row * seq_len;
  const size_t tt = (size_t)row * (size_t)seq_len + (size_t)((pos + shift) % seq_len);
  const uint16_t* hs = student + (size_t)t * (size_t)lds_;
  for (int j = wave; j < k; j += kRowThreads / 64) {
    int col = t_idx[tt * (size_t)k + j];
    col = col < 0 ? 0 : (col >= V ? V - 1 : col);  // a caller's own column list cannot make the gather leave the weight
    const float dot = wave_dot_bf16(hs, W + (size_t)col * (size_t)ldw, H, lane);
    if (lane == 0) {
      sv[j] = dot * rcp_temp;
      tv[j] = t_vals[tt * (size_t)k + j];
      columns[(size_t)t * (size_t)k + j] = col;
    }
  }
  __syncthreads();
  float ms = -INFINITY, mt = -INFINITY;
  for (int j = threadIdx.x; j < k; j += kRowThreads) ms = fmaxf(ms, sv[j]), mt = fmaxf(mt, tv[j]);
  ms = block_reduce(ms, true, red);
  mt = block_reduce(mt, true, red);
  float ss = 0.f, st = 0.f;
  for (int j = threadIdx.x; j < k; j += kRowThreads) ss += expf(sv[j] - ms), st += expf(tv[j] - mt);
  ss = block_reduce(ss, false, red);
  st = block_reduce(st, false, red);
  const float log_ss = logf(ss);
  float l = 0.f;
  for (int j = threadIdx.x; j < k; j += kRowThreads) {
    const float tp = expf(tv[j] - mt) / st;
    const float qs = expf(sv[j] - ms) / ss;
    l -= tp * ((sv[j] - ms) - log_ss);
    coef[(size_t)t * (size_t)k + j] = qs - tp;
  }
  l = block_reduce(l, false, red);
  if (threadIdx.x == 0) loss[t] = l;
}

// d student hidden[t, :] = dloss[t] / temperature * sum_j coef[t, j] * weight[columns[t, j], :]   (the scatter of
// soft_ce.py:309-312 followed by the output layer's backward), fp32 sums, bf16 result.
__global__ __launch_bounds__(kRowThreads) void topk_softce_bwd_rows(const uint16_t* __restrict__ W, int ldw,
                                                                    const float* __restrict__ coef, const int* __restrict__ columns,
                                                                    const float* __restrict__ dloss, int H, int V, int k, float rcp_temp,
                                                                    uint16_t* __restrict__ d_student, int ldd) {
  extern __shared__ float sm_bwd[];  // k coefficients, then k columns
  float* cf = sm_bwd;
  int* cl = (int*)(sm_bwd + k);
  const int t = blockIdx.x;
  const float g = dloss[t] * rcp_temp;
  for (int j = threadIdx.x; j < k; j += kRowThreads) {
    cf[j] = coef[(size_t)t * (size_t)k + j] * g;
    const int col = columns[(size_t)t * (size_t)k + j];
    cl[j] = col < 0 ? 0 : (col >= V ? V - 1 : col);
  }
  __syncthreads();
  for (int c = threadIdx.x * 8; c < H; c += kRowThreads * 8) {
    float acc[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
    for (int j = 0; j < k; ++j) {
      const uint4 wv = *(const uint4*)(W + (size_t)cl[j] * (size_t)ldw + c);
      const uint32_t ww[4] = {wv.x, wv.y, wv.z, wv.w};
      const float f = cf[j];
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        acc[2 * q] = fmaf(f, __uint_as_float(ww[q] << 16), acc[2 * q]);
        acc[2 * q + 1] = fmaf(f, __uint_as_float(ww[q] & 0xffff0000u), acc[2 * q + 1]);
      }
    }
    const f32x4 lo4 = {acc[0], acc[1], acc[2], acc[3]}, hi4 = {acc[4], acc[5], acc[6], acc[7]};
    const bf16x4 lo = __builtin_convertvector(lo4, bf16x4), hi = __builtin_convertvector(hi4, bf16x4);
    const uint2 a2 = *(const uint2*)&lo, b2 = *(const uint2*)&hi;
    *(uint4*)(d_student + (size_t)t * (size_t)ldd + c) = make_uint4(a2.x, a2.y, b2.x, b2.y);
  }
}

}  // namespace topk

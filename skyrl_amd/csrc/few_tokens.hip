// Kernels for calls of few tokens.  A 256 x 256 tile fills a CU by itself (gemm_core.hpp), so what it does once per tile -- the
// latency of its first copies, its epilogue -- overlaps nothing.  With few tokens that, and not the contraction, is most of the
// tile's time; the tiles here are half as large and two workgroups share a CU.
#include "few_tokens.hpp"

#include "gemm_core.hpp"
#include "half_tile.hpp"

#include <type_traits>
#include <utility>

namespace lmhead {
namespace {

// ------------------------------------------------------------------------------------------------------------
// Weight gradient of a chunk for few tokens: dW[v, h] = sum_t D[t, v] . hidden[t, h], a contraction of a few 32-token steps that
// writes V x H values.  What bounds it is the writing (8 bytes per clock and CU at 5 TB/s), and what a 256 x 256 tile does once per
// tile -- the first copies' latency, 256 accumulators through LDS, the stores -- does not overlap anything when one workgroup
// fills the CU.  So: 256 (vocab) x 128 (hidden) tiles, eight waves of 64 x 64, two workgroups per CU, one's loads and MFMAs under
// the other's stores.  Both operands are read K-major where they are (no hidden^T): a ring of three slots of 32 tokens, LDS rows
// of 128 columns whose 32-byte windows are permuted by (row & 3) | (row bit 3) << 2, so that the eight row pieces of half a
// transposing read fall into different banks.  Tiles along the hidden size first: neighbours share the dz columns in L2.
// The stores are non-temporal: with ordinary ones the kernels behind this one write dW's dirty lines back while they read the weight
// (V=151936, H=1536: dHidden 150 -> 106 us, forward 141 -> 128 at T=137, this kernel the same).  At every size, although results
// below 256 MiB would be found in the last-level cache: backward, and forward + backward + the sum of dW into another tensor, ordinary ->
// non-temporal, 98 MiB (bf16, V=32000, H=1600, T=64; the least that comes here) 102 -> 101 and 202 -> 199 us, 141 MiB (V=128256, H=576)
// 152 -> 136 and 270 -> 258, 195 MiB (fp32) 122 -> 117 and 281 -> 275, 282 MiB 203 -> 159 and 390 -> 358, 890 MiB (V=151936, H=1536) 469 ->
// 416 and 1089 -> 1035.  A norm of dW behind it gains too, but for 98 MiB at T=64 (187 -> 192).
// H=1536, V=151936: 88 us at T=17 (5.3 TB/s), 123 at T=64, 144 at T=96.
// ------------------------------------------------------------------------------------------------------------
constexpr int kDwK = 32;                          // tokens per step
constexpr int kDwThreads = 512, kDwSlots = 3;
constexpr int kDwBlockBytes = kDwK * 128 * 2;     // 32 tokens x 128 columns
constexpr int kDwSlotBytes = 3 * kDwBlockBytes;   // hidden, dz columns 0 .. 127 and 128 .. 255
static_assert(kDwThreads / 64 * 1024 == kDwBlockBytes, "one copy per wave fills a block");

__device__ __forceinline__ void copy_to_lds(const uint16_t* g, uint32_t lds_addr) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, off" : : "s"(lds_addr), "v"(g) : "memory", "m0");
}

template <bool F32>
__device__ __forceinline__ void dw_few_tile(const DwFewArgs& a, int n, int logical, char* lds) {
  const int tiles_h = (a.H + kDwH - 1) / kDwH;
  const int tv = logical / tiles_h;
  const int h0 = __builtin_amdgcn_readfirstlane((logical - tv * tiles_h) * kDwH), v0 = __builtin_amdgcn_readfirstlane(tv * kDwV);
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wh = wave >> 2, wv = wave & 3;  // the wave's 64 hidden columns and 64 vocabulary rows
  const int lrow = lane & 15, kq = lane >> 4;
  const int steps = (n + kDwK - 1) / kDwK;

  // Copies: wave w brings rows 4w .. 4w + 3 of every block, 16 lanes a row.  Token rows behind the last one exist in the panel (zeros)
  // and repeat the last one of the hidden states.
  const int krow = wave * 4 + kq;
  const int ckey = kq | (((wave >> 1) & 1) << 2);
  const int col = (((lrow >> 1) ^ ckey) * 2 + (lrow & 1)) * 8;
  const uint16_t* h_src = a.Hd + (h0 + col < a.H - 8 ? h0 + col : a.H - 8);
  const uint16_t* d_src = a.D + (size_t)krow * (size_t)a.ldd + v0 + col;
  const uint32_t base = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) char*)lds;
  auto issue = [&](int step, uint32_t slot) {
    const int k = step * kDwK + krow;
    const uint16_t* d = d_src + (size_t)(step * kDwK) * (size_t)a.ldd;
    copy_to_lds(h_src + (size_t)(k < n ? k : n - 1) * (size_t)a.ldh, slot + wave * 1024);
    copy_to_lds(d, slot + wave * 1024 + kDwBlockBytes);
    copy_to_lds(d + 128, slot + wave * 1024 + 2 * kDwBlockBytes);
  };

  // Fragments (as for the K-major operand of gemm_core.hpp): lane (kq, s) supplies row kq * 8 + half * 4 + (s >> 2), columns (s & 3) * 4
  // .. + 3 of the 16, and receives column s of the eight rows kq * 8 .. + 7.
  typedef __attribute__((address_space(3))) i16x4* half_ptr;
  typedef __attribute__((ext_vector_type(8))) short i16x8;
  const int fkey = (lrow >> 2) | ((kq & 1) << 2);
  const uint32_t frow = (uint32_t)((kq * 8 + (lrow >> 2)) * 256 + (lrow & 3) * 8);
  uint32_t h_off[4], v_off[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    h_off[i] = frow + (uint32_t)(((wh * 4 + i) ^ fkey) << 5);
    v_off[i] = frow + (uint32_t)((((wv & 1) * 4 + i) ^ fkey) << 5) + (uint32_t)(1 + (wv >> 1)) * kDwBlockBytes;
  }
  auto fragment = [&](uint32_t addr) -> bf16x8 {
    const i16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((half_ptr)(uintptr_t)addr);
    const i16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((half_ptr)(uintptr_t)(addr + 4 * 256));
    const i16x8 v = __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
    return __builtin_bit_cast(bf16x8, v);
  };

  uint32_t s0 = base, s1 = base + kDwSlotBytes, s2 = base + 2 * kDwSlotBytes;  // slots of this step, the next, the one after
  if (steps > 0) issue(0, s0);
  if (steps > 1) issue(1, s1);
  f32x4 acc[4][4];
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
  asm volatile("s_nop 7" ::: "memory");  // as in zero_acc()
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j) asm volatile("" : "+a"(acc[i][j]));
  for (int step = 0; step < steps; ++step) {
    // This step's copies have landed (the next one's three may be in flight), and every wave has left the slot that is filled next.
    if (step + 1 < steps) wait_copies_and_barrier<3>();
    else wait_copies_and_barrier<0>();
    if (step + 2 < steps) issue(step + 2, s2);
    bf16x8 hf[4], vf[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) hf[i] = fragment(s0 + h_off[i]);
#pragma unroll
    for (int j = 0; j < 4; ++j) vf[j] = fragment(s0 + v_off[j]);
#pragma unroll
    for (int j = 0; j < 4; ++j)
#pragma unroll
      for (int i = 0; i < 4; ++i) mfma_16x16x32(acc[i][j], hf[i], vf[j]);
    const uint32_t t = s0;
    s0 = s1, s1 = s2, s2 = t;
  }
  wait_copies_and_barrier<0>();  // no wave reads the ring any more: it becomes the staging room, an eighth of it per wave, all of it
  asm volatile("s_nop 15\n\ts_nop 15" ::: "memory");  // as behind the other mainloops
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j) asm volatile("" : "+a"(acc[i][j]));

  if (h0 + wh * 64 >= a.H) return;
  constexpr int kStageBytes = 64 * (64 * 2 + 16);
  static_assert(kStageBytes * (kDwThreads / 64) <= kDwSlots * kDwSlotBytes && 32 * (64 * 4 + 16) <= kStageBytes, "staging room");
  char* const stage = lds + wave * kStageBytes;
  const size_t c0 = (size_t)(h0 + wh * 64);
  auto out_row = [&](int row) {  // the row of C that row `row` of this wave is, or -1
    int r = v0 + wv * 64 + row;
    if (r >= a.N) return -1;
    if (r >= a.n_tail) {
      r -= a.n_back;
      if (r < a.n_tail) return -1;
    }
    return r;
  };
  if constexpr (F32) {  // 32 rows at a time: a store instruction writes 256 contiguous bytes of four rows
    constexpr int kPitch = 64 * 4 + 16;
#pragma unroll
    for (int half = 0; half < 2; ++half) {
#pragma unroll
      for (int j = 0; j < 2; ++j)
#pragma unroll
        for (int i = 0; i < 4; ++i) *(f32x4*)(stage + (j * 16 + lrow) * kPitch + (i * 16 + kq * 4) * 4) = acc[i][half * 2 + j];
#pragma unroll
      for (int it = 0; it < 8; ++it) {
        const f32x4 v = *(const f32x4*)(stage + (it * 4 + kq) * kPitch + lrow * 16);
        const int r = out_row(half * 32 + it * 4 + kq);
        if (r >= 0) __builtin_nontemporal_store(v, (f32x4*)(a.Cf + (size_t)r * (size_t)a.H + c0 + lrow * 4));
      }
    }
  } else {  // a store instruction writes 128 contiguous bytes of eight rows
    constexpr int kPitch = 64 * 2 + 16;
#pragma unroll
    for (int j = 0; j < 4; ++j)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const bf16x4 b4 = __builtin_convertvector(acc[i][j], bf16x4);
        *(uint2*)(stage + (j * 16 + lrow) * kPitch + (i * 16 + kq * 4) * 2) = *(const uint2*)&b4;
      }
#pragma unroll
    for (int it = 0; it < 8; ++it) {
      const u32x4 v = *(const u32x4*)(stage + (it * 8 + (lane >> 3)) * kPitch + (lane & 7) * 16);
      const int r = out_row(it * 8 + (lane >> 3));
      if (r >= 0) __builtin_nontemporal_store(v, (u32x4*)(a.Cb + (size_t)r * (size_t)a.H + c0 + (lane & 7) * 8));
    }
  }
}

// A tile per workgroup.
template <bool F32>
__global__ __launch_bounds__(kDwThreads, 4) void lmhead_bwd_dw_few(const DwFewArgs a) {
  __shared__ __attribute__((aligned(1024))) char lds[kDwSlots * kDwSlotBytes];
  const int n = a.T_dev ? __builtin_amdgcn_readfirstlane(*a.T_dev) : a.T;
  dw_few_tile<F32>(a, n, xcd_contiguous(blockIdx.x, gridDim.x), lds);
}

// The tiles of a call for more tokens, of which up to kDwTileActive turn out to have a gradient.  Two workgroups per CU make all of them, because
// those of a launch that finds more have to end before the next one begins (a workgroup per tile: 7128 at H=1536, V=151936, training pass with 137 of 137
// tokens 505 -> 507 us, with 428 of 611 865 -> 870).  A tile begins when the stores of the one before have left, which costs 6 us of a pass with 20 tokens;
// with its copies in front of those stores it is no faster (459 -> 456 us with 20 tokens, 469 -> 476 with 40), and neither are four workgroups per CU.
// Tokens of one step: the workgroups go through the tiles side by side, 512 at a time; of two: each has neighbours, which read the same dz columns.  dW in
// us, 24 and 40 tokens, side by side / neighbours: H=1536, V=151936 101 / 106 and 111 / 112; H=2048, V=100000 80 / 95 and 112 / 97; H=4096, V=128256 196 / 226 and
// 254 / 226 (dz in registers 244 and 243, a workgroup per tile 222 and 260 with no launch beside it).
template <bool F32>
__global__ __launch_bounds__(kDwThreads, 4) void lmhead_bwd_dw_few_active(const DwFewArgs a, int tiles) {
  __shared__ __attribute__((aligned(1024))) char lds[kDwSlots * kDwSlotBytes];
  const int n = __builtin_amdgcn_readfirstlane(*a.T_dev);
  if (n > kDwTileActive) return;
  const bool neighbours = n > kDwK;
  const int groups = gridDim.x, group = neighbours ? xcd_contiguous(blockIdx.x, groups) : (int)blockIdx.x;
  const int first = neighbours ? (int)((int64_t)tiles * group / groups) : group, end = neighbours ? (int)((int64_t)tiles * (group + 1) / groups) : tiles;
  for (int id = first; id < end; id += neighbours ? 1 : groups) {
    if (id != first) asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");  // every wave has taken its rows of the tile before from LDS
    dw_few_tile<F32>(a, n, neighbours ? id : xcd_contiguous(id, tiles), lds);
  }
}

// ------------------------------------------------------------------------------------------------------------
// Weight gradient of a chunk for few tokens: dW[v, h] = sum_t D[t, v] . hidden[t, h], a contraction of up to 24 32-token steps that
// writes V x H values, with the dz values of 256 vocabulary rows resident in registers.
//
// What bounds the tiles above behind a hundred tokens or so is the copies and the LDS: per 256 x 128 values they copy dz and hidden, 768 bytes a
// token, and each of their eight waves reads both operands from LDS.  Here each of four waves keeps 64 vocabulary rows of dz, of all tokens, in
// registers (64 x 448 values are 224 of its 512), and the hidden states pass by, 32 columns of all tokens at a time, through LDS: what is copied
// per value falls to a third, what is read from LDS to half, and an MFMA needs a quarter of a fragment.  One workgroup per CU takes its equal share
// of the units of 256 rows x 64 columns, tile by tile; a new tile costs 6 us in which its dz comes through LDS and is transposed there.
// A half of a unit is 8 MFMAs a step; meanwhile the next but one slot of hidden columns is copied (the next one where three slots do not fit), and
// the values of the half before it leave: converted, turned through the wave's own LDS and stored in 128-byte pieces of rows, past the cache as
// above.  Two barriers a half, none that waits for what has just been asked for.
// H=1536, V=151936, tiles above -> this: 166 -> 122 us at T=137, 255 -> 201 at 428 (1.0 PFLOP/s), 359 -> 306 at 768; fp32 result, H=1024, V=64000,
// T=400 102 -> 76.  Of the 201 us the MFMAs alone would take 103, with their fragment reads 130; dz, the stores and the copies add 28, 26 and 16 (timed
// with each of them left out).  No faster: up to seven slots, stores spread over two halves, whole units stored as one piece of memory, the next
// tile's first dz pieces copied ahead, two to twelve times as many workgroups.
// ------------------------------------------------------------------------------------------------------------
constexpr int kDwResidentThreads = 256;
constexpr int kDwHalf = 32;                             // hidden columns of a slot of the ring
constexpr int kDwStepBytes = 32 * kDwHalf * 2;          // 32 tokens of a slot
constexpr int kDwStageBytes = 64 * 128;                 // per wave: 64 vocabulary rows of 128 bytes
constexpr int kDwAgprSteps = 16;                        // steps whose dz fragments are in AGPRs; the others' are in VGPRs

// f(0), f(1), ... f(N - 1), the arguments as compile-time constants (the compiler leaves loops of this size rolled).
template <class F, int... I>
__device__ __forceinline__ void unrolled(std::integer_sequence<int, I...>, F f) {
  (f(std::integral_constant<int, I>{}), ...);
}
template <int N, class F>
__device__ __forceinline__ void unrolled(F f) {
  unrolled(std::make_integer_sequence<int, N>{}, f);
}

// One wave-wide copy: 1 KiB at lds_addr, from the uniform address g and the lanes' 32-bit offsets.
__device__ __forceinline__ void dw_copy(const char* g, uint32_t off, uint32_t lds_addr) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2" : : "s"(lds_addr), "v"(off), "s"(g) : "memory", "m0");
}

// acc (+)= a . b, the accumulator in VGPRs, b (dz) in AGPRs or VGPRs.
template <bool FIRST, bool B_AGPR>
__device__ __forceinline__ void dw_mfma(f32x4& c, const bf16x8& a, const bf16x8& b) {
  if constexpr (FIRST) {
    if constexpr (B_AGPR) asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, 0" : "=&v"(c) : "v"(a), "a"(b));
    else asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, 0" : "=&v"(c) : "v"(a), "v"(b));
  } else {
    if constexpr (B_AGPR) asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, %0" : "+v"(c) : "v"(a), "a"(b));
    else asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, %0" : "+v"(c) : "v"(a), "v"(b));
  }
}

// A dz fragment is in the registers that dw_mfma() takes it from.
template <bool AGPR>
__device__ __forceinline__ void dw_keep(bf16x8& b) {
  if constexpr (AGPR) asm volatile("" : "+a"(b));
  else asm volatile("" : "+v"(b));
}

// Where the 64 x 64 values of a wave's unit go: rows lo .. of the 64, as many as `bytes` holds.
struct DwOut {
  uint32_t base_lo, base_hi, bytes;
  int lo;
};

// How many of `count` events at first, first + step, ... come before `at`.
constexpr int dw_before(int at, int first, int step, int count) {
  const int n = at <= first ? 0 : (at - first + step - 1) / step;
  return n < count ? n : count;
}

template <bool F32, int KT>
__device__ __forceinline__ void dw_resident_units(const DwFewArgs& a, int n, char* lds) {
  static_assert(KT % 2 == 0 && KT >= 4, "pairs of steps");
  constexpr int PT = KT / 2;                            // pairs of steps; also copies per wave and slot
  constexpr int kSlotBytes = KT * kDwStepBytes;
  // Slots of the ring: while one is read, the one behind the last that has been filled is filled.
  constexpr int kSlots = KT <= 20 ? 3 : 2;
  constexpr bool kDeep = kSlots > 2;
  constexpr int kRing = kSlots * kSlotBytes;
  // Room for dz on its way into registers: what the ring and the stages leave, and the slot that is filled next.
  constexpr int kDzRoom = LDS_BYTES - kRing - 4 * kDwStageBytes, kPieceBytes = 2 * kDwStepBytes;
  constexpr int kOwnPieces = kDzRoom / (4 * kPieceBytes), kSlotPieces = kDeep ? kSlotBytes / (4 * kPieceBytes) : 0;
  constexpr int kPieces = kOwnPieces + kSlotPieces < KT ? kOwnPieces + kSlotPieces : KT;
  static_assert(kPieces >= 2, "room for the dz pieces");
  constexpr int ES = F32 ? 4 : 2;
  // The two steps of a pair back to back on an accumulator (mainloop_pairs() in gemm_core.hpp); one step behind the other where the dz
  // fragments leave no registers for those of two steps ahead.
  constexpr bool kStepOrder = KT > 22;
  constexpr int kMfmas = 16 * PT;                       // of a half
  constexpr int kAhead = KT >= 6 && KT <= 20 ? 6 : kStepOrder ? 2 : 4;  // fragments read ahead; one is read every four MFMAs
  constexpr int kNextLanded = kMfmas - 4 * kAhead;      // from here on the fragments are those of the next slot
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int lrow = lane & 15, kq = lane >> 4;
  const uint32_t base = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) char*)lds;
  typedef __attribute__((address_space(3))) i16x4* half_ptr;
  typedef __attribute__((ext_vector_type(8))) short i16x8;

  const int per_tile = a.H / kDwUnitH, units = (a.N + kDwV - 1) / kDwV * per_tile;
  const int id = xcd_contiguous(blockIdx.x, gridDim.x);
  const int share = __builtin_amdgcn_readfirstlane(units / (int)gridDim.x), more = units - share * (int)gridDim.x;
  const int u0 = id * share + (id < more ? id : more), u1 = u0 + share + (id < more ? 1 : 0);  // at least one: the grid has no more workgroups

  // Copies of a slot: copy j of wave w brings tokens 16 (4 j + w) .. + 15, four lanes a token.  Tokens behind the last one repeat it, in the
  // last copy.
  const uint32_t c_row = (uint32_t)(lane >> 2);
  const uint32_t c_col = (uint32_t)((((lane & 3) ^ (((lane >> 5) & 1) << 1))) * 16);
  const uint32_t h_pitch = (uint32_t)a.ldh * 2u, d_pitch = (uint32_t)a.ldd * 2u;
  auto first_token = [&](int j) {
    const int t = 16 * (4 * j + wave);
    return t < n ? t : n - 1;
  };
  const uint32_t behind = (uint32_t)(n - 1 - first_token(PT - 1));
  const uint32_t h_off[2] = {c_row * h_pitch + c_col, (c_row < behind ? c_row : behind) * h_pitch + c_col};
  auto copy_hidden = [&](int j, int h, uint32_t slot) {
    dw_copy((const char*)(a.Hd + (size_t)first_token(j) * (size_t)a.ldh + h), h_off[j == PT - 1], slot + (uint32_t)((4 * j + wave) * 1024));
  };
  // Fragments: lane (kq, s) supplies row kq * 8 + half * 4 + (s >> 2), columns (s & 3) * 4 .. + 3 of the 16, and receives column s of
  // the eight rows kq * 8 .. + 7.
  const uint32_t f_lane = (uint32_t)((kq * 8 + (lrow >> 2)) * 64 + (lrow & 3) * 8 + (kq & 1) * 32);
  auto fragment = [&](uint32_t addr) -> bf16x8 {
    const i16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((half_ptr)(uintptr_t)addr);
    const i16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((half_ptr)(uintptr_t)(addr + 4 * 64));
    const i16x8 v = __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
    return __builtin_bit_cast(bf16x8, v);
  };

  // dz of the wave's 64 vocabulary rows: step ks, rows 16 j .. + 15.
  bf16x8 dz[KT][4];
  const uint32_t dz_room = base + (uint32_t)(kRing + 4 * kDwStageBytes + wave * kOwnPieces * kPieceBytes);
  auto load_dz = [&](int v0, uint32_t free_slot) {
    const char* src = (const char*)(a.D + v0 + wave * 64);
    auto room = [&](int ks) {
      const int x = ks % kPieces;
      return x < kOwnPieces ? dz_room + (uint32_t)(x * kPieceBytes) : free_slot + (uint32_t)((wave * kSlotPieces + x - kOwnPieces) * kPieceBytes);
    };
    auto issue = [&](int ks) {
#pragma unroll
      for (int c = 0; c < 4; ++c)
        dw_copy(src + (size_t)(ks * 32 + (c & 1) * 16) * (size_t)d_pitch + (c >> 1) * 64, c_row * d_pitch + c_col, room(ks) + (uint32_t)(c * 1024));
    };
#pragma unroll
    for (int ks = 0; ks < kPieces; ++ks) issue(ks);
    unrolled<KT>([&](auto ks_const) {
      constexpr int ks = decltype(ks_const)::value;
      asm volatile("s_waitcnt vmcnt(%0)" ::"n"(4 * (KT - 1 - ks < kPieces - 1 ? KT - 1 - ks : kPieces - 1)) : "memory");
#pragma unroll
      for (int j = 0; j < 4; ++j) dz[ks][j] = fragment(room(ks) + (f_lane ^ (uint32_t)((j & 1) * 32)) + (uint32_t)((j >> 1) * kDwStepBytes));
      if (ks + kPieces < KT) {
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        issue(ks + kPieces);
      }
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        if constexpr (ks > 0) dw_keep<(ks <= kDwAgprSteps)>(dz[ks - 1][j]);
        if constexpr (ks == KT - 1) dw_keep<(ks < kDwAgprSteps)>(dz[ks][j]);
      }
    });
    asm volatile("s_nop 7" ::: "memory");
  };

  char* const stage = lds + kRing + wave * kDwStageBytes;
  const int st_w = lrow * 128 + (kq & 1) * 8, st_key = (lrow >> 1) & 7;  // rows 16 j further: the same key
  const int st_r = lane * 16 ^ (((lane >> 4) & 3) << 4);  // row lane >> 3 of eight; rows 8 it further: the key's third bit is that of it
  f32x4 acc[2][2][4] = {};
  auto stage_block = [&](int set, int i, int j) {  // 16 columns x 16 rows of a half
    char* row = stage + j * (16 * 128) + st_w;
    asm volatile("" : "+v"(acc[set][i][j]));
    if constexpr (F32) {
      *(f32x4*)(stage + j * (16 * 128) + lrow * 128 + (((i * 4 + kq) ^ st_key) << 4)) = acc[set][i][j];
    } else {
      const bf16x4 b4 = __builtin_convertvector(acc[set][i][j], bf16x4);
      *(uint2*)(row + (((set * 4 + i * 2 + (kq >> 1)) ^ st_key) << 4)) = *(const uint2*)&b4;
    }
  };
  auto staged = [&](int it) { return *(const u32x4*)(stage + it * 1024 + (st_r ^ ((it & 1) << 6))); };
  const uint32_t o_pitch = (uint32_t)a.H * ES, o_lane = (uint32_t)(lane >> 3) * o_pitch + (uint32_t)(lane & 7) * 16u;
  auto store = [&](const DwOut& o, int col_bytes, int it, const u32x4& v) {
    uint32_t row = (uint32_t)lane >> 3, first = o_lane;
    // Eight rows and offsets formed once would be sixteen registers, which the largest cases do not have.
    if constexpr (KT > 20) asm volatile("" : "+v"(row), "+v"(first));
    const uint32_t off = it * 8 + (int)row < o.lo ? 0x80000000u : first + (uint32_t)(it * 8) * o_pitch;
    const auto rsrc = __builtin_amdgcn_make_buffer_rsrc((void*)(uintptr_t)(((uint64_t)o.base_hi << 32 | o.base_lo) + (uint64_t)col_bytes), 0, (int)o.bytes,
                                                        0x00020000);
    __builtin_amdgcn_raw_buffer_store_b128(v, rsrc, (int)off, 0, 2);
  };

  uint32_t cur = base;
  auto slot_behind = [&](uint32_t slot) { return slot == base + (uint32_t)(kRing - kSlotBytes) ? base : slot + (uint32_t)kSlotBytes; };
  auto slot_before = [&](uint32_t slot) { return slot == base ? base + (uint32_t)(kRing - kSlotBytes) : slot - (uint32_t)kSlotBytes; };
  bf16x8 ahead[kAhead];  // the first fragments of the slot that is read next
  auto hidden_fragment = [&](uint32_t slot_lane0, uint32_t slot_lane1, int g) {  // in the order of their use
    const int ks = g / 4 * 2 + (kStepOrder ? (g / 2) % 2 : g % 2), i = kStepOrder ? g % 2 : (g / 2) % 2;
    return fragment((i ? slot_lane1 : slot_lane0) + (uint32_t)(ks * kDwStepBytes));
  };

  // A half of a unit: 32 columns, accumulators S.  Meanwhile a slot is filled with columns fill_h and the accumulators of the half before it
  // are staged; what is staged leaves, to `out`.
  auto half = [&](auto s_const, int fill_h, const DwOut& out) {
    constexpr int S = decltype(s_const)::value;
    constexpr int kSpread = kNextLanded / 2 / PT < 2 ? 2 : kNextLanded / 2 / PT > 6 ? 6 : kNextLanded / 2 / PT;
    constexpr int kLastCopy = 3 + (PT - 1) * kSpread;
    constexpr int kFirstStore = 18, kStores = F32 || S == 0 ? 8 : 0;
    constexpr int kStoreStep = kStores == 0 ? 1 : (kMfmas - kFirstStore - 2) / kStores;
    static_assert(kLastCopy < kNextLanded && kStoreStep >= 1, "the copies come before the wait");
    // What is issued behind the next slot's copies and may be under way when it is waited for: three slots, the stores of the half before this
    // one from its last copy on, this half's copies and its stores up to the wait; two, this half's stores between its last copy and the wait.
    constexpr int kBefore = F32 || S == 1 ? 8 : 0;  // stores of the half before this one
    constexpr int kBeforeStep = kBefore == 0 ? 1 : (kMfmas - kFirstStore - 2) / kBefore;
    constexpr int kUpToWait = dw_before(kNextLanded, kFirstStore, kStoreStep, kStores);
    constexpr int kBehind = kDeep ? kBefore - dw_before(kLastCopy, kFirstStore, kBeforeStep, kBefore) + PT + kUpToWait
                                  : kUpToWait - dw_before(kLastCopy, kFirstStore, kStoreStep, kStores);
    static_assert(kBehind >= 0 && kBehind < 64, "vmcnt is a 6-bit counter");
    const uint32_t next = slot_behind(cur), fill = slot_before(cur);
    const uint32_t c0 = cur + f_lane, c1 = cur + (f_lane ^ 32u);
    bf16x8 fr[4 * PT + kAhead];
    u32x4 held[8];
#pragma unroll
    for (int g = 0; g < kAhead; ++g) fr[g] = ahead[g];
    unrolled<kMfmas>([&](auto x_const) {
      constexpr int at = decltype(x_const)::value, x = at % 16;
      constexpr int b = kStepOrder ? x % 8 : x / 2, ks = kStepOrder ? x / 8 : x % 2, i = b / 4, j = i ? 7 - b : b;
      constexpr int step = at / 16 * 2 + ks, g = at / 16 * 4 + (kStepOrder ? ks * 2 + i : i * 2 + ks);
      if constexpr (at == kNextLanded) asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" ::"n"(kBehind) : "memory");
      dw_mfma<step == 0, (step < kDwAgprSteps)>(acc[S][i][j], fr[g], dz[step][j]);
      __builtin_amdgcn_sched_barrier(0);
      if constexpr (at % 4 == 0) {
        constexpr int r = at / 4 + kAhead;
        if constexpr (r < 4 * PT) fr[r] = hidden_fragment(c0, c1, r);
        else fr[r] = hidden_fragment(next + f_lane, next + (f_lane ^ 32u), r - 4 * PT);
      }
      if constexpr (at == 2) asm volatile("s_barrier" ::: "memory");  // every wave has left the slot that is filled
      if constexpr (at >= 6 && at < 14) stage_block(1 - S, (at - 6) / 4, (at - 6) % 4);
      if constexpr (at >= 3 && (at - 3) % kSpread == 0 && (at - 3) / kSpread < PT) copy_hidden((at - 3) / kSpread, fill_h, fill);
      if constexpr (at + 2 >= kFirstStore && (at + 2 - kFirstStore) % kStoreStep == 0 && (at + 2 - kFirstStore) / kStoreStep < kStores) {
        held[(at + 2 - kFirstStore) / kStoreStep] = staged((at + 2 - kFirstStore) / kStoreStep);
      }
      if constexpr (at >= kFirstStore && (at - kFirstStore) % kStoreStep == 0 && (at - kFirstStore) / kStoreStep < kStores) {
        constexpr int it = (at - kFirstStore) / kStoreStep;
        store(out, (F32 && S == 0) ? 128 : 0, it, held[it]);
      }
      __builtin_amdgcn_sched_barrier(0);
    });
#pragma unroll
    for (int g = 0; g < kAhead; ++g) ahead[g] = fr[4 * PT + g];
    cur = next;
  };

  int tile = __builtin_amdgcn_readfirstlane(u0 / per_tile), hb = u0 - tile * per_tile;
  auto column_ahead = [&](int n_units) {  // of the unit that many behind hb (those behind the last one are not used)
    int x = hb + n_units;
    while (x >= per_tile) x -= per_tile;
    return x * 64;
  };
#pragma unroll
  for (int s = 0; s < kSlots - 1; ++s) {  // the first slots
    const int h = column_ahead(s / 2) + s % 2 * kDwHalf;
#pragma unroll
    for (int j = 0; j < PT; ++j) copy_hidden(j, h, base + (uint32_t)(s * kSlotBytes));
  }
  asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");
#pragma unroll
  for (int g = 0; g < kAhead; ++g) ahead[g] = hidden_fragment(cur + f_lane, cur + (f_lane ^ 32u), g);
  DwOut out{0u, 0u, 0u, 0};  // nothing has been made yet: no store passes the range check
  for (int left_units = u1 - u0; left_units > 0; ++tile, hb = 0) {
    if constexpr (kSlotPieces > 0) asm volatile("s_barrier" ::: "memory");  // every wave has left the slot that is filled next
    load_dz(tile * kDwV, slot_before(cur));
    const int v = tile * kDwV + wave * 64;
    const bool moved = v >= a.n_tail;
    const int rows = a.N - v < 0 ? 0 : a.N - v < 64 ? a.N - v : 64, lo = moved ? a.n_tail + a.n_back - v : 0;
    const uint64_t row0 = (uint64_t)(uintptr_t)(F32 ? (char*)a.Cf : (char*)a.Cb) + (uint64_t)((int64_t)(v - (moved ? a.n_back : 0)) * (int64_t)a.H) * ES;
    const int last = hb + left_units < per_tile ? hb + left_units : per_tile;
    left_units -= last - hb;
    for (; hb < last; ++hb) {
      const int h = hb * 64, ahead_h = column_ahead(1);
      // scalar registers: a buffer descriptor in vector registers would be a loop over the lanes
      const uint64_t at = row0 + (uint64_t)(h * ES);
      const DwOut here{(uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)at), (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)(at >> 32)),
                       (uint32_t)__builtin_amdgcn_readfirstlane(rows * a.H * ES), lo > 0 ? lo : 0};
      half(std::integral_constant<int, 0>{}, kDeep ? ahead_h : h + kDwHalf, out);
      half(std::integral_constant<int, 1>{}, kDeep ? ahead_h + kDwHalf : ahead_h, here);
      out = here;
    }
  }
  asm volatile("s_waitcnt vmcnt(0)\n\ts_nop 15\n\ts_nop 15" ::: "memory");  // no copy is in flight when the workgroup ends
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j) stage_block(1, i, j);
#pragma unroll
  for (int it = 0; it < 8; ++it) store(out, F32 ? 128 : 0, it, staged(it));
}

template <bool F32>
__global__ __launch_bounds__(kDwResidentThreads, 1) void lmhead_bwd_dw_resident(const DwFewArgs a) {
  __shared__ __attribute__((aligned(1024))) char lds[LDS_BYTES];
  const int n = a.T_dev ? __builtin_amdgcn_readfirstlane(*a.T_dev) : a.T;
  static_assert(kDwTileActive == 64 && kDwTileTokens >= 64, "below 65 tokens there is no code here");
  if (n <= kDwTileActive) return;  // made in tiles, by the launch before
  switch ((n + 63) / 64) {
    case 2: return dw_resident_units<F32, 4>(a, n, lds);
    case 3: return dw_resident_units<F32, 6>(a, n, lds);
    case 4: return dw_resident_units<F32, 8>(a, n, lds);
    case 5: return dw_resident_units<F32, 10>(a, n, lds);
    case 6: return dw_resident_units<F32, 12>(a, n, lds);
    case 7: return dw_resident_units<F32, 14>(a, n, lds);
    case 8: return dw_resident_units<F32, 16>(a, n, lds);
    case 9: return dw_resident_units<F32, 18>(a, n, lds);
    case 10: return dw_resident_units<F32, 20>(a, n, lds);
    case 11: return dw_resident_units<F32, 22>(a, n, lds);
    default: return dw_resident_units<F32, 24>(a, n, lds);
  }
}

// ------------------------------------------------------------------------------------------------------------
// Logits of few tokens on half tiles (half_tile.hpp): the forward's statistics and the backward's dz values.  Same bits as on
// the square tiles.
// ------------------------------------------------------------------------------------------------------------
template <bool ENTROPY>
__global__ __launch_bounds__(NTHREADS, 2) void lmhead_fwd_half_tiles(const uint16_t* __restrict__ W, int ldw,
                                                                     const uint16_t* __restrict__ Hd, int ldh, int T, int H, int V,
                                                                     float rcp_temp, float* __restrict__ part_max,
                                                                     float* __restrict__ part_sum, float* __restrict__ part_pz) {
  __shared__ __attribute__((aligned(1024))) char lds[kHalfLdsBytes];
  const int tiles_m = (V + BM - 1) / BM, tiles_n = (T + kHalfBN - 1) / kHalfBN;
  int tm, tn;
  tile_coords(blockIdx.x, tiles_m, tiles_n, kGroupM, tm, tn);
  half_acc_t acc;
  half_tile_product(Operand{W, ldw, tm * BM, V}, Operand{Hd, ldh, tn * kHalfBN, T}, H / kHalfBK, lds, acc);
  const int wave = threadIdx.x >> 6, wm = wave / WAVES_N, wn = wave % WAVES_N;
  fwd_epilogue<ENTROPY, false>(acc, tm * WAVES_M + wm, tiles_m * WAVES_M, tn * kHalfBN + wn * kHalfWN, T, V, rcp_temp, part_max, part_sum,
                               part_pz);
}

constexpr int kHalfDzLdsBytes = NWAVES * kHalfWN * (kDzTokRow + kDzTokBytes);  // 74 KiB: the epilogue's staging, before it the ring
static_assert(kHalfDzLdsBytes >= kHalfLdsBytes && 2 * kHalfDzLdsBytes <= LDS_BYTES, "two workgroups per CU");
template <bool ENTGRAD>
__global__ __launch_bounds__(NTHREADS, 2) void lmhead_bwd_half_dz(const DzArgs z) {
  __shared__ __attribute__((aligned(1024))) char lds[kHalfDzLdsBytes];
  int T;
  Tile tile;
  if (!dz_tile_of<false>(z, blockIdx.x, kHalfBN, T, tile)) return;
  dz_tile<ENTGRAD, kHalfTN, false>(
      z, T, tile.tm * BM, tile.tn * kHalfBN, lds,
      [&](const Operand& a, const Operand& b, half_acc_t& acc) {
        half_tile_product(a, b, z.H / kHalfBK, lds, acc);
        return true;
      },
      [](u32x4 v, u32x4* p) { __builtin_nontemporal_store(v, p); });
}

}  // namespace

hipError_t launch_bwd_dw_few(hipStream_t s, const DwFewArgs& a) {
  if (dw_resident(a.T, a.H)) {
    if (a.T_dev) {  // either kernel returns at once where the other one makes dW
      const int64_t tiles = dw_few_tiles(a.H, a.N), most = 2 * (int64_t)a.ncu;
      hipLaunchKernelGGL(a.Cf ? lmhead_bwd_dw_few_active<true> : lmhead_bwd_dw_few_active<false>, dim3((unsigned)(tiles < most ? tiles : most)),
                         dim3(kDwThreads), 0, s, a, (int)tiles);
      const hipError_t e = hipGetLastError();
      if (e != hipSuccess) return e;
    }
    const int64_t units = (a.N + kDwV - 1) / kDwV * (a.H / kDwUnitH);
    hipLaunchKernelGGL(a.Cf ? lmhead_bwd_dw_resident<true> : lmhead_bwd_dw_resident<false>, dim3((unsigned)(units < a.ncu ? units : a.ncu)),
                       dim3(kDwResidentThreads), 0, s, a);
    return hipGetLastError();
  }
  hipLaunchKernelGGL(a.Cf ? lmhead_bwd_dw_few<true> : lmhead_bwd_dw_few<false>, dim3((unsigned)dw_few_tiles(a.H, a.N)),
                     dim3(kDwThreads), 0, s, a);
  return hipGetLastError();
}

void launch_fwd_half_tiles(hipStream_t s, bool entropy, const uint16_t* W, int ldw, const uint16_t* Hd, int ldh, int T, int H, int V,
                           float rcp_temp, float* part_max, float* part_sum, float* part_pz) {
  const int tiles = (V + BM - 1) / BM * ((T + kHalfBN - 1) / kHalfBN);
  hipLaunchKernelGGL(entropy ? lmhead_fwd_half_tiles<true> : lmhead_fwd_half_tiles<false>, dim3((unsigned)tiles), dim3(NTHREADS), 0, s, W,
                     ldw, Hd, ldh, T, H, V, rcp_temp, part_max, part_sum, part_pz);
}

hipError_t launch_bwd_half_dz(hipStream_t s, bool entgrad, const DzArgs& z) {
  hipLaunchKernelGGL(entgrad ? lmhead_bwd_half_dz<true> : lmhead_bwd_half_dz<false>, dim3((unsigned)(z.tiles_m * z.tiles_n)),
                     dim3(NTHREADS), 0, s, z);
  return hipGetLastError();
}

}  // namespace lmhead

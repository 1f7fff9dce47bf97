// Kernels for calls of few tokens.  A 256 x 256 tile fills a CU by itself (gemm_core.hpp), so what it does once per tile -- the
// latency of its first copies, its epilogue -- overlaps nothing.  With few tokens that, and not the contraction, is most of the
// tile's time; the tiles here are half as large and two workgroups share a CU.
#include "few_tokens.hpp"

#include "gemm_core.hpp"
#include "half_tile.hpp"

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
// 416 and 1089 -> 1035; T=400 and 768 likewise.  A norm of dW behind it gains too, but for 98 MiB at T=64 (187 -> 192).
// H=1536, V=151936: 88 us at T=17 (5.3 TB/s), 162 at T=137, 250 at T=400, 419 at T=768.
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
__global__ __launch_bounds__(kDwThreads, 4) void lmhead_bwd_dw_few(const DwFewArgs a) {
  __shared__ __attribute__((aligned(1024))) char lds[kDwSlots * kDwSlotBytes];
  const int n = a.T_dev ? __builtin_amdgcn_readfirstlane(*a.T_dev) : a.T;
  const int tiles_h = (a.H + kDwH - 1) / kDwH;
  const int logical = xcd_contiguous(blockIdx.x, gridDim.x);
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

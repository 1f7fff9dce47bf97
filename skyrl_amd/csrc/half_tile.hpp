// 256 x 128 tiles for calls of few tokens: C[M,N] = A[M,K] * B[N,K]^T as in gemm_core.hpp, half as wide along the tokens, with two
// workgroups per CU.
//
// What bounds such a call is the weight coming from HBM.  On a 256 x 256 tile that stream stops once per tile -- one workgroup
// fills the CU, so nothing overlaps its first copies' latency and its epilogue -- and the copies and MFMAs of up to 128 of
// its 256 tokens are for nothing.  Here one workgroup's epilogue runs under the other's loop.  Per 32 k a tile copies 24 KiB (768 clk
// at the 32 B/clk that a CU takes from L2) for 512 clk of MFMAs per SIMD, half again as many bytes per product as the square
// tile, which therefore is the better one as soon as there are products enough to bind (kHalfTileTokens).  Forward with its merge
// at T=16, V=151936: 84 -> 62 us at H=896 (4.4 TB/s of weight), 144 -> 121 at H=1536.  A copy behind every fourth MFMA instead of all six
// of a step at once: the same (60 and 121 us at T=17).
//
// Four waves of 128 x 64 (8 x 4 accumulators, 128 AGPRs).  A ring of three slots of 32 k: while one is consumed the next has landed
// or is landing and the copies of the one after it are issued; one barrier per step.  Slots hold rows of 64 bytes, four 16-byte
// chunks; chunk c of row r sits at c ^ half_swz(r).  That key puts the 16 chunks of sixteen rows at one k, and those of rows 0-3 and
// 12-15 at one k with rows 4-11 at its neighbour, into 16 different bank groups.
#pragma once
#include "gemm_core.hpp"

namespace lmhead {

constexpr int kHalfBN = 128, kHalfBK = 32, kHalfSlots = 3;
constexpr int kHalfWN = kHalfBN / WAVES_N;  // 64 tokens per wave
constexpr int kHalfTN = kHalfWN / MT;
constexpr int kHalfRowBytes = kHalfBK * 2;
constexpr int kHalfABytes = BM * kHalfRowBytes, kHalfBBytes = kHalfBN * kHalfRowBytes;
constexpr int kHalfSlotBytes = kHalfABytes + kHalfBBytes;  // 24 KiB
constexpr int kHalfLdsBytes = kHalfSlots * kHalfSlotBytes;
constexpr int kHalfACopies = kHalfABytes / 1024 / NWAVES, kHalfBCopies = kHalfBBytes / 1024 / NWAVES;
typedef f32x4 half_acc_t[TM][kHalfTN];

__device__ __forceinline__ int half_swz(int row) {
  const int b0 = (row >> 2) & 1, b1 = (row >> 3) & 1;
  return ((b0 ^ b1) << 1) | b1;
}

// One wave-wide copy: 16 rows of 64 bytes at the 32-bit offsets `src` from the uniform address g, 1 KiB at `slot_wave_addr` + OFS.
template <int OFS>
__device__ __forceinline__ void half_copy(const char* g, uint32_t src, uint32_t slot_wave_addr) {
  asm volatile("s_add_u32 m0, %0, %1\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %2, %3"
               :
               : "s"(slot_wave_addr), "n"(OFS), "v"(src), "s"(g)
               : "memory", "m0", "scc");
}

// acc = A[a.row0 : +256, 0 : 32 * steps] * B[b.row0 : +128, same k]^T.  steps >= 2.  Every thread of the workgroup calls this with the
// same arguments; on return no copy is in flight, every wave has left the ring, and the accumulators may be read.
__device__ __forceinline__ void half_tile_product(const Operand& a, const Operand& b, int steps, char* lds, half_acc_t& acc) {
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wm = wave / WAVES_N, wn = wave % WAVES_N;
  uint32_t a_src[kHalfACopies], b_src[kHalfBCopies];
  const int in_copy = lane >> 2, chunk = ((lane & 3) ^ half_swz(in_copy)) * 16;
#pragma unroll
  for (int j = 0; j < kHalfACopies; ++j) {
    const int row = (j * NWAVES + wave) * 16 + in_copy;
    int r = row >= BM / 2 ? row - a.upper_back : row;
    r = a.row0 + r < a.rows ? r : a.rows - 1 - a.row0;
    a_src[j] = (uint32_t)r * (uint32_t)a.ld * 2u + (uint32_t)chunk;
  }
#pragma unroll
  for (int j = 0; j < kHalfBCopies; ++j) {
    const int row = (j * NWAVES + wave) * 16 + in_copy;
    const int r = b.row0 + row < b.rows ? row : b.rows - 1 - b.row0;
    b_src[j] = (uint32_t)r * (uint32_t)b.ld * 2u + (uint32_t)chunk;
  }
  const char* ga = (const char*)(a.ptr + (size_t)__builtin_amdgcn_readfirstlane(a.row0) * (size_t)a.ld);
  const char* gb = (const char*)(b.ptr + (size_t)__builtin_amdgcn_readfirstlane(b.row0) * (size_t)b.ld);
  const uint32_t w0 = wave_copy_base(lds);
  constexpr int kCopies = kHalfACopies + kHalfBCopies;
  static_assert(kHalfACopies == 4 && kHalfBCopies == 2, "issue() is written for these");
  auto issue = [&](uint32_t slot) {  // the next 32 k of both operands
    half_copy<0 * NWAVES * 1024>(ga, a_src[0], slot);
    half_copy<1 * NWAVES * 1024>(ga, a_src[1], slot);
    half_copy<2 * NWAVES * 1024>(ga, a_src[2], slot);
    half_copy<3 * NWAVES * 1024>(ga, a_src[3], slot);
    half_copy<kHalfABytes + 0 * NWAVES * 1024>(gb, b_src[0], slot);
    half_copy<kHalfABytes + 1 * NWAVES * 1024>(gb, b_src[1], slot);
    ga += kHalfRowBytes, gb += kHalfRowBytes;
  };

  const int lrow = lane & 15;
  const uint32_t frag = (uint32_t)(lrow * kHalfRowBytes + (((lane >> 4) ^ half_swz(lrow)) << 4)) - (uint32_t)wave * 1024u;
  const uint32_t a_off = frag + (uint32_t)(wm * WM * kHalfRowBytes);
  const uint32_t b_off = frag + (uint32_t)(kHalfABytes + wn * kHalfWN * kHalfRowBytes);
  typedef const __attribute__((address_space(3))) bf16x8* frag_ptr;

  uint32_t s0 = w0, s1 = w0 + kHalfSlotBytes, s2 = w0 + 2 * kHalfSlotBytes;  // slots of this step, the next, the one after
  issue(s0);
  issue(s1);
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < kHalfTN; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
  asm volatile("s_nop 7" ::: "memory");  // as in zero_acc()
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < kHalfTN; ++j) asm volatile("" : "+a"(acc[i][j]));
  for (int step = 0; step < steps; ++step) {
    // This step's copies have landed (the next one's may be in flight), and every wave has left the slot that is filled next.
    if (step + 1 < steps) wait_copies_and_barrier<kCopies>();
    else wait_copies_and_barrier<0>();
    if (step + 2 < steps) issue(s2);
    bf16x8 af[TM], bfr[kHalfTN];
#pragma unroll
    for (int j = 0; j < kHalfTN; ++j) bfr[j] = *(frag_ptr)(uintptr_t)(s0 + b_off + (uint32_t)(j * MT * kHalfRowBytes));
#pragma unroll
    for (int i = 0; i < TM; ++i) af[i] = *(frag_ptr)(uintptr_t)(s0 + a_off + (uint32_t)(i * MT * kHalfRowBytes));
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
      for (int j = 0; j < kHalfTN; ++j) {
        const int jj = (i & 1) ? kHalfTN - 1 - j : j;  // consecutive MFMAs share one operand
        mfma_16x16x32(acc[i][jj], af[i], bfr[jj]);
      }
    const uint32_t t = s0;
    s0 = s1, s1 = s2, s2 = t;
  }
  wait_copies_and_barrier<0>();
  asm volatile("s_nop 15\n\ts_nop 15" ::: "memory");  // as behind the other mainloops
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < kHalfTN; ++j) asm volatile("" : "+a"(acc[i][j]));
}

}  // namespace lmhead

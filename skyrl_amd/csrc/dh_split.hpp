// How the contraction of the dHidden tiles over the vocabulary is cut: the rating that the host and the device make alike, and what the
// launches take from it.  Plain arithmetic on sizes, for any C++ compiler.
#pragma once

#include <stdint.h>

#ifdef __HIPCC__
#define LMHEAD_HD __host__ __device__
#else
#define LMHEAD_HD
#endif

namespace lmhead {

constexpr int kSplitTile = 256;  // edge of a C tile
constexpr int kSplitPair = 128;  // vocabulary rows of a pair of k-tiles

// How many workgroups share the vocabulary of one dHidden tile.  There are tokens/256 x H/256 such tiles with a contraction of a
// whole chunk of the vocabulary: 18 tiles of 2374 k-tiles at T=611, H=1536, V=151936, which one workgroup each leaves on 18
// of 256 CUs for 2.5 ms.  Rated in k-tiles of mainloop: the dHidden tiles alone in whole rounds of the CUs, or everything the
// launch carries spread evenly plus half a dW tile of tail, plus what the slabs cost to write, read and add (a 256 KiB slab
// tile about a seventeenth of a k-tile of the whole chip).  At least 1024 vocabulary rows per split.  Integer arithmetic: the
// host and compact_active_rows, which rates one candidate per lane for the token count it found, must agree.
// Measured, GEMM launches of the backward, one workgroup per tile -> split: 2750 -> 560 us at T=428 (active), H=1536, V=151936
// (12 tiles x 8 splits beside the dW tiles; alone in the launch, as now, 12 x 21 in 180); 544 -> 168 us at T=1050, H=1024, V=32000,
// fp32 weight; 2714 -> 1509 us at T=4096, H=2048, V=151936 and 2304 -> 1317 us at T=1592, H=4096, V=128261, both without dW; 3030 ->
// 2700 us at T=4096, H=1536, V=151936.  What the slabs have room for (slab_slots) bounds the choice.
constexpr int kMinSplitPairs = 8;
constexpr int kMaxSplits = 64;
struct SplitProblem {
  int tiles_h;    // dHidden tiles per 256 tokens
  int pairs;      // k-tile pairs of a chunk's vocabulary
  int dw_tiles;   // dW tiles of the same launch (0: frozen weight)
  int slots;      // slab tiles there is room for
  int shares;     // whether the launch may go in Shares
  int ncu;
};
LMHEAD_HD inline int64_t split_cost(const SplitProblem& p, int tokens, int splits) {
  const int tiles = (tokens + kSplitTile - 1) / kSplitTile * p.tiles_h;
  if (splits > 1 && ((int64_t)tiles * splits > p.slots || p.pairs / splits < kMinSplitPairs)) return INT64_MAX;
  const int64_t len = 2 * ((p.pairs + splits - 1) / splits) + (splits > 1 ? 10 : 8);
  const int64_t items = (int64_t)tiles * splits, dw_len = (tokens + kSplitPair - 1) / kSplitPair * 2 + 6;
  const int64_t alone = (int64_t)(((int)items + p.ncu - 1) / p.ncu) * len * p.ncu;
  const int64_t spread = items * len + p.dw_tiles * dw_len + (p.dw_tiles ? dw_len * p.ncu / 2 : 0);
  return (alone > spread ? alone : spread) + (splits > 1 ? items * 15 + 4 * p.ncu : 0);
}

// Shares.  Where dHidden is alone in its launch, a whole number of workgroups per tile leaves CUs idle: 96 tiles go in two splits on 192 of 256.  So
// the tiles may also be taken in groups of b, u workgroups each, and every workgroup takes an equal share of its group's k-tile pairs, laid end to
// end: the end of one tile, whole tiles, the beginning of another.  Splits are groups of one tile.  Group g holds tiles g, g + G, g + 2 G, ... of the
// launch's order, G groups in all: the workgroups at one place j of their groups read the same range of the vocabulary for G neighbouring tiles
// and come one behind the other, on one XCD.  Splits -> shares, the GEMM launch: 1437 -> 1251 us at 96 tiles (draft loss of 2868 tokens, H=2048,
// V=151936), one round and a part -> shares 2457 -> 1582 at 288 tiles (draft loss of 8192, H=2304, V=64000; pass 9135 -> 8282) and 2580 -> 2311 at
// 400 (5120 tokens, H=5120, V=64000), three quarters of a round 1877 -> 1578 at 192 (2868 of 4096 tokens, H=4096, V=100000).  112 tiles in two splits, 224
// CUs, draw the power that 256 do: 1261 and 1290, hence the term for it in share_cost().
struct Shares {
  int b, u, groups;
  LMHEAD_HD int workgroups() const { return groups * u; }
  LMHEAD_HD int slots() const { return groups * (u + b - 1); }
  // Group g: its tiles, and the first and last of them that workgroup j shares in, the first and last workgroup of its i-th tile.
  LMHEAD_HD int tiles_of(int g, int tiles) const { return (tiles - g + groups - 1) / groups; }
  LMHEAD_HD int first_tile(int j, int bg) const { return j * bg / u; }
  LMHEAD_HD int last_tile(int j, int bg) const { return ((j + 1) * bg + u - 1) / u - 1; }
  LMHEAD_HD int first_workgroup(int i, int bg) const { return i * u / bg; }
  LMHEAD_HD int last_workgroup(int i, int bg) const { return ((i + 1) * u + bg - 1) / bg - 1; }
  // Where workgroup j's share of the group's bg * pairs k-tile pairs begins, and the one before it ends.  Below 2^26: chunks have fewer than 2^15 pairs.
  LMHEAD_HD int begin(int j, int bg, int pairs) const { return bg * pairs * j / u; }
  // The slab of workgroup j's sums for the i-th tile: j + i differs along a group, because each step goes on to the next of either.
  LMHEAD_HD int slot(int g, int i, int j) const { return (j + i) * groups + g; }
};
constexpr int kMaxGroup = 32;
// Blocks that may have this many tiles and more.  Below it splits leave little: from 64000 columns on shares are rated at most 2.7 % shorter (52 tiles, whose
// four splits keep 208 of 256 CUs busy), with narrower chunks up to 4 % of launches of some 30 us.  And calls of few tokens notice what finding a
// share takes: draft loss of 20 tokens, H=896, V=246016, four tiles in 64 splits, GEMM 109 -> 111 us, their sum 8.6 -> 11.4.
constexpr int64_t kSharesFromTiles = 65;
// code: u, and b above its lowest eight bits where it is not 1.
LMHEAD_HD inline Shares shares_of(int code, int tiles) {
  const int b = code < 256 ? 1 : code >> 8;
  return Shares{b, code & 255, b == 1 ? tiles : (tiles + b - 1) / b};
}
// Groups of b >= 2 tiles, as many workgroups each as the CUs hold at once, rated as above.  A workgroup's further tiles cost it an epilogue and
// another beginning each.  `code` is set where the answer is below INT64_MAX.
// Behind six sevenths of the CUs the power is what limits, so that a workgroup more makes the others slower.  Draft loss, V=151936, rated
// without that -> with it: 6 tiles x 23 workgroups -> 2 x 7 at 66 tiles, GEMM 951 -> 897 us, pass 4.91 -> 4.77 ms; 9 x 32 -> three splits at 72, 977 -> 989 and
// 5.12 -> 4.99; 5 x 16 -> three splits at 80, 1014 -> 1017 and 5.56 -> 5.49; no difference at 120.  split_cost() has no such term, which
// prefers splits that keep six sevenths busy to shares of the same length.
LMHEAD_HD inline int64_t share_cost(const SplitProblem& p, int tokens, int b, int& code) {
  const int tiles = (tokens + kSplitTile - 1) / kSplitTile * p.tiles_h;
  if (!p.shares || b > tiles) return INT64_MAX;
  const int groups = (tiles + b - 1) / b;
  int u = p.ncu / groups;
  u = u < kMaxSplits ? u : kMaxSplits;
  if (u < 1) return INT64_MAX;
  const Shares s{b, u, groups};
  const int pairs = (p.pairs * b + u - 1) / u;  // chunks have fewer than 2^15 pairs
  if (s.slots() > p.slots || pairs < kMinSplitPairs) return INT64_MAX;
  code = b << 8 | u;
  const int64_t len = 2 * pairs + 10 * ((b + u - 1) / u + (b % u && u % b ? 1 : 0));
  const int64_t busy = s.workgroups() * 7 / 6;
  return len * (busy > p.ncu ? busy : p.ncu) + (int64_t)s.slots() * 15 + 4 * p.ncu;
}

// dHidden tiles of T tokens.
inline int64_t dh_tiles(int64_t T, int64_t H) { return (T + kSplitTile - 1) / kSplitTile * ((H + kSplitTile - 1) / kSplitTile); }
inline SplitProblem split_problem(int64_t T, int64_t H, int64_t vc, bool want_dw, int64_t slots, int ncu) {
  const int64_t tiles_h = (H + kSplitTile - 1) / kSplitTile;
  return SplitProblem{(int)tiles_h, (int)(vc / kSplitPair), want_dw ? (int)(tiles_h * (vc / kSplitTile)) : 0, (int)slots,
                      !want_dw && dh_tiles(T, H) >= kSharesFromTiles, ncu};
}

// Slab tiles of dHidden partial sums for at most T tokens and chunks of vc columns: room for one tile per CU, at least two per dHidden
// tile; none beyond one per dHidden tile from 192 tiles on, where dW tiles in the same launch fill the CUs that dHidden leaves idle.
// The line is drawn for launches with dW.  Without (a frozen weight, the draft loss, a dW launch of its own) shares would go further where there is
// room for them: the draft loss always has it, a frozen weight from the room that row compaction brings (carve_bwd).
constexpr int64_t kSplitBelowTiles = 192;
inline int64_t slab_slots(int64_t T, int64_t H, int64_t vc) {
  const int64_t tiles = dh_tiles(T, H), most = vc / kSplitPair / kMinSplitPairs;
  if (tiles >= kSplitBelowTiles || most < 2) return tiles;
  const int64_t room = 2 * tiles > 256 ? 2 * tiles : 256;
  const int64_t used = tiles * (most < kMaxSplits ? most : kMaxSplits);
  return room < used ? room : used;
}

inline int best_splits(const SplitProblem& p, int64_t tokens) {
  int best = 1;
  int64_t best_cost = split_cost(p, (int)tokens, 1);
  for (int k = 2; k <= kMaxSplits; ++k) {
    const int64_t c = split_cost(p, (int)tokens, k);
    if (c < best_cost) best = k, best_cost = c;
  }
  for (int b = 2; b <= kMaxGroup; ++b) {
    int code = 0;
    const int64_t c = share_cost(p, (int)tokens, b, code);
    if (c < best_cost) best = code, best_cost = c;
  }
  return best;
}

// The launch of a block of at most `tiles` dHidden tiles: whether it goes to lmhead_bwd_dh_shares, which alone understands codes of Shares, and the
// workgroups for dHidden.  p is what rates the block, here or on the device (the code is then not known yet): with row compaction that is one
// problem for all blocks of a call, and the last of them may have far fewer tiles than it was made for.
struct DhLaunch {
  bool shares;
  int workgroups;
};
inline DhLaunch dh_launch(const SplitProblem& p, int tiles, int code, bool code_on_device) {
  int n = shares_of(code, tiles).workgroups();
  if (code_on_device && n < p.slots) n = p.slots;             // splits: a slab each
  if (code_on_device && p.shares && n < p.ncu) n = p.ncu;  // shares: at most a workgroup per CU
  return DhLaunch{(bool)p.shares, n};
}

}  // namespace lmhead

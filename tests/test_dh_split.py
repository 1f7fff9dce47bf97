"""How the dHidden contraction is cut (``csrc/dh_split.hpp``), compiled for the CPU and walked through: for every block of a call and every number
of tokens with a gradient that the device may find in it, the kernel that the host launches has to understand what the rating chose, in the
grid and in the slabs that there are.

The driver below takes each launch apart as the kernels do (``lmhead_bwd_gemm``, ``lmhead_bwd_dh_shares``, ``lmhead_dh_reduce``): every k-tile pair of
every tile is multiplied once, every sum that leaves as a slab has one of its own, and the reduction reads exactly those.
"""

from __future__ import annotations

import os
import shutil
import subprocess

import pytest

from skyrl_amd import _lib
from skyrl_amd.csrc import build as B

pytestmark = pytest.mark.skipif(not shutil.which("g++"), reason="needs a C++ compiler")

DRIVER = r"""
#include <stdio.h>
#include <stdlib.h>
#include <string.h>
#include <algorithm>
#include <vector>
#include "dh_split.hpp"
using namespace lmhead;
static long checked = 0, in_shares = 0;
static int fail(const char* what, const SplitProblem& p, int64_t tokens, int code) {
  printf("%s: tiles_h %d pairs %d dw %d slots %d shares %d ncu %d, %ld tokens, code %d = %d x %d\n", what, p.tiles_h, p.pairs, p.dw_tiles, p.slots,
         (int)p.shares, p.ncu, (long)tokens, code, code < 256 ? 1 : code >> 8, code & 255);
  exit(1);
}
// One launch with `pairs` k-tile pairs, as few as a narrow last chunk has.
static void walk(const SplitProblem& p, const DhLaunch& l, int64_t tokens, int code, int pairs) {
  const int tiles = (int)((tokens + kSplitTile - 1) / kSplitTile) * p.tiles_h;
  if (code >= 256 && !l.shares) fail("shares in a kernel of splits", p, tokens, code);
  const Shares s = shares_of(code, tiles);
  if (s.workgroups() > l.workgroups) fail("more workgroups than the grid has", p, tokens, code);
  if (tiles == 0) return;
  std::vector<int> next(tiles, 0), slabs(tiles, 0);  // pairs multiplied, and sums made so far
  std::vector<char> used(p.slots, 0);
  for (int j = 0; j < s.u; ++j)
    for (int g = 0; g < s.groups; ++g) {
      const int bg = s.b == 1 ? 1 : s.tiles_of(g, tiles), first = s.first_tile(j, bg), last = s.last_tile(j, bg);
      const int from = s.begin(j, bg, pairs), to = s.begin(j + 1, bg, pairs);
      int done = from;
      for (int i = first; i <= last; ++i) {
        const int tile = i * s.groups + g, k0 = std::max(from - i * pairs, 0), k1 = std::min(to - i * pairs, pairs);
        if (i >= bg || tile >= tiles) fail("no such tile", p, tokens, code);
        if (k0 != next[tile] || k1 < k0) fail("pairs left out or taken twice", p, tokens, code);
        next[tile] = k1, done += k1 - k0;
        const bool alone = s.first_workgroup(i, bg) == s.last_workgroup(i, bg);
        if (j < s.first_workgroup(i, bg) || j > s.last_workgroup(i, bg)) fail("a workgroup that the reduction does not know", p, tokens, code);
        const int slot = s.b > 1 ? s.slot(g, i, j) : j * tiles + g;
        if (slot < 0 || slot >= p.slots) fail("no such slab", p, tokens, code);
        if (used[slot]++) fail("two sums in one slab", p, tokens, code);
        if (!alone && slot != (s.b > 1 ? s.slot(g, i, s.first_workgroup(i, bg)) + slabs[tile] * s.groups : tile + slabs[tile] * tiles))
          fail("the reduction reads another slab", p, tokens, code);
        ++slabs[tile];
      }
      if (done != to) fail("a share that its tiles do not hold", p, tokens, code);
    }
  for (int g = 0; g < s.groups; ++g)
    for (int i = 0; i < (s.b == 1 ? 1 : s.tiles_of(g, tiles)); ++i) {
      const int tile = i * s.groups + g, bg = s.b == 1 ? 1 : s.tiles_of(g, tiles);
      if (next[tile] != pairs || slabs[tile] != s.last_workgroup(i, bg) - s.first_workgroup(i, bg) + 1) fail("an unfinished tile", p, tokens, code);
    }
  ++checked, in_shares += code >= 256;
}
int main(int argc, char** argv) {
  if (argc > 1) {  // T H vc compact tokens: what is chosen where dHidden is alone, with the scratch of the query
    const int64_t T = atoll(argv[1]), Tb = std::min<int64_t>(T, 32768), H = atoll(argv[2]), vc = atoll(argv[3]), more = atoi(argv[4]) ? T * H / 2 / 65536 : 0;
    printf("%d\n", best_splits(split_problem(Tb, H, vc, false, slab_slots(Tb, H, vc) + more, 256), atoll(argv[5])));
    return 0;
  }
  const int64_t block = 32768;
  for (const int ncu : {256, 80})
    for (const int64_t T : {1, 300, 1400, 2100, 4500, 8192, 32768, 32769, 33024, 33792, 35000, 41000, 49152, 65536, 65537, 65792, 70000, 98304, 99000})
      for (const int64_t H : {64, 256, 512, 768, 896, 1024, 1536, 2048, 2304, 3072, 3584, 4096, 4160, 5120})
        for (const int64_t vc : {256, 1024, 2048, 4096, 7680, 15104, 16128, 20480, 32000, 49152, 100096, 152064})
          for (const bool want_dw : {false, true})
            for (int room = 0; room < 3; ++room) {
              const int64_t Tb = std::min(T, block), least = dh_tiles(Tb, H), more = T * H / 2 / (256 * 256);
              const int64_t slots = room == 0 ? least : room == 1 ? least + more : slab_slots(Tb, H, vc) + more;
              const SplitProblem rated = split_problem(Tb, H, vc, want_dw, slots, ncu);  // compact_active_rows rates all blocks with it
              for (int64_t t0 = 0; t0 < T; t0 += block) {
                if (t0 && T - t0 >= block) continue;
                const int64_t Tcur = std::min(T - t0, block);
                const int tiles = (int)dh_tiles(Tcur, H), most = (int)((Tcur + 255) / 256);
                for (int m = 0; m <= most; m += m < 24 || Tcur < block ? 1 : 13) {
                  const int64_t tokens = std::min((int64_t)m * 256, Tcur);
                  const int code = best_splits(rated, tokens);
                  const DhLaunch l = dh_launch(rated, tiles, 1, true);
                  for (const int pairs : {rated.pairs, rated.pairs / 2, 1})
                    if (pairs) walk(rated, l, tokens, code, pairs);
                }
                // without row compaction the host rates the block that it launches
                const SplitProblem own = split_problem(Tcur, H, vc, want_dw, slots, ncu);
                const int code = best_splits(own, Tcur);
                walk(own, dh_launch(own, tiles, code, false), Tcur, code, own.pairs);
              }
            }
  printf("%ld launches, %ld in shares\n", checked, in_shares);
  return in_shares > 1000 ? 0 : 1;
}
"""


@pytest.fixture(scope="module")
def driver(tmp_path_factory):
    out = tmp_path_factory.mktemp("dh_split")
    (out / "driver.cpp").write_text(DRIVER)
    proc = subprocess.run(["g++", "-std=c++17", "-O2", "-I", B.HERE, "-o", str(out / "driver"), str(out / "driver.cpp")], capture_output=True, text=True)
    assert proc.returncode == 0, proc.stderr[-2000:]
    return str(out / "driver")


def test_every_launch_understands_what_the_rating_chose(driver):
    run = subprocess.run([driver], capture_output=True, text=True, timeout=300)
    assert run.returncode == 0, run.stdout[-1000:]


def _library_chunk(T, H, V, compact):
    """The chunk of vocabulary that the library takes by itself: the one whose scratch is as large as that of its own choice."""
    query = _lib.load().skyrl_lmhead_bwd_active_rows_workspace_bytes if compact else _lib.load().skyrl_lmhead_bwd_workspace_bytes
    fits = [vc for vc in range(256, (V + 255) // 256 * 256 + 1, 256) if query(T, H, V, vc) == query(T, H, V, 0)]
    assert len(fits) == 1, fits
    return fits[0]


def _shares(driver, T, H, V, vc, compact, tokens):
    vc = vc or _library_chunk(T, H, V, compact)
    return int(subprocess.run([driver, *map(str, (T, H, vc, int(compact), tokens))], capture_output=True, text=True, check=True).stdout) >= 256


def test_sizes_of_the_gpu_tests_go_in_shares(driver):
    """test_tile_edges_gpu.py compares dHidden in shares with dHidden whole or in splits: its sizes have to be some that go in shares."""
    from tests import test_tile_edges_gpu as G

    for T, H, V, vc in G.SHARES:
        assert _shares(driver, T, H, V, vc, True, T) or _shares(driver, T, H, V, vc, True, int(0.7 * T)), (T, H, V, vc)
    assert not _shares(driver, *G.NO_ROOM_FOR_SHARES, True, G.NO_ROOM_FOR_SHARES[0])
    for T, H, V, vc in G.SHARES_OF_A_SHORT_LAST_BLOCK:
        assert _shares(driver, T, H, V, vc, True, T - 32768), (T, H, V, vc)

"""The host's rules and the maps that kernels evaluate (sa_launch.h, sa_common.h), compiled as they are and run on the CPU: the order in
which a workgroup goes through the tiles of its window, the rows that a workgroup of the one-launch backward keeps values of, and
the order in which workgroups are dispatched."""
import os
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "kernels_amd", "csrc")
HIPCC = os.path.join(os.environ.get("ROCM_PATH", "/opt/rocm"), "bin", "hipcc")
CHUNKS = "1, 7, 8, 10, 16, 24, 32, 50, 64, 96, 100, 128, 192, 256, 300"

HEAD = r"""
#include <cstdio>
#include <cstdlib>
#include <vector>
#include <algorithm>
#include "sa_launch.h"
using namespace sa;
namespace sa { std::atomic<int> g_tune_override[3] = {{-1}, {-1}, {-1}}; }
#define CHECK(x, ...) do { if (!(x)) { printf("line %d: %s: ", __LINE__, #x); printf(__VA_ARGS__); printf("\n"); exit(1); } } while (0)
static FwdParams problem(int B, int H, int T, int C, int R) {
  FwdParams p{};
  p.B = B, p.H = H, p.T = T, p.C = C, p.R = R;
  return p;
}
"""

# Every tile once; a full window starts at a multiple of the period, so that overlapping windows agree in time; with one period a
# smaller workgroup's row goes through its tiles in the order of the largest workgroup's.
TILE_ORDER = HEAD + r"""
struct Window { int t0, t1; };
static Window window(int r0, int rows, int T, int C, int R, int tile) {   // key tiles of query rows [r0, r0 + rows)
  const int last = std::min(r0 + rows, T) - 1;
  return {std::max(r0 / C - R, 0) * C / tile, (std::min((last / C + 1) * C, T) + tile - 1) / tile};
}
static std::vector<int> sequence(Window w, const FwdParams& p) {
  const TileOrder order(w.t0, w.t1, p.period, p.pdiv);
  std::vector<int> s;
  for (int t = order.first, it = 0; it < w.t1 - w.t0; ++it, t = order.next(t)) s.push_back(t);
  return s;
}
int main() {
  int windows = 0;
  const int shapes[][2] = {{128, 64}, {64, 32}, {128, 32}, {256, 32}};
  for (auto& sh : shapes)
    for (int C : {CHUNKS})
      for (int R : {0, 1, 2, 5, 9}) {
        const int rows = sh[0], tile = sh[1], T = 5 * (C * (R + 2) + rows);
        FwdParams p = problem(1, 1, T, C, R);
        set_tile_order(p, rows, tile);
        CHECK(p.period > 0, "C %d R %d", C, R);
        CHECK(tiles_of_window(C * (R + 1), C, R, rows, tile) == 0, "C %d R %d", C, R);
        for (int r0 = 0; r0 < T; r0 += rows) {
          const Window w = window(r0, rows, T, C, R, tile);
          std::vector<int> s = sequence(w, p), sorted = s;
          std::sort(sorted.begin(), sorted.end());
          CHECK((int)s.size() == w.t1 - w.t0 && (int)s.size() <= p.period, "C %d R %d r0 %d", C, R, r0);
          for (int i = 0; i < (int)s.size(); ++i) CHECK(sorted[i] == w.t0 + i, "C %d R %d r0 %d", C, R, r0);
          if ((int)s.size() == p.period) CHECK(s[0] % p.period == 0, "C %d R %d r0 %d", C, R, r0);
          for (int small = 64; small < rows; small *= 2)   // the same rows in smaller workgroups, wave by wave
            for (int r = r0; r < std::min(r0 + rows, T); r += 32) {
              const Window mine = window(r, 32, T, C, R, tile);
              auto of = [&](const std::vector<int>& all) {
                std::vector<int> out;
                for (int t : all) if (t >= mine.t0 && t < mine.t1) out.push_back(t);
                return out;
              };
              CHECK(of(s) == of(sequence(window(r / small * small, small, T, C, R, tile), p)), "C %d R %d r %d in %d", C, R, r, small);
            }
          ++windows;
        }
      }
  printf("ok %d\n", windows);
}
""".replace("CHUNKS", CHUNKS)

# The one-launch backward: no workgroup goes through more query rows, in whole tiles, than it keeps values of.
ROWS_IN_REACH = HEAD + r"""
int main() {
  int windows = 0;
  const int shapes[][2] = {{128, 64}, {64, 32}};
  for (int C = 1; C <= 320; ++C)
    for (int R = 0; C * (R + 1) <= 320; ++R)
      for (auto& sh : shapes) {
        const int rows = sh[0], tile = sh[1], reach = rows_in_reach(C, R, rows, tile);
        int most = 0;
        for (int r0 = 0; r0 < rows * C; r0 += rows) {   // the pattern repeats after at most C workgroups
          const int first = r0 / C * C / tile * tile, end = (((r0 + rows - 1) / C + R + 1) * C + tile - 1) / tile * tile;
          CHECK(end - first <= reach, "C %d R %d rows %d r0 %d", C, R, rows, r0);
          most = std::max(most, end - first);
        }
        CHECK(most == reach, "C %d R %d rows %d", C, R, rows);
        if (fused_backward(64, C, R) && (rows == 64) == fused_backward_in_two_waves(64, C, R)) CHECK(reach <= BWD_FUSED_MAX_ROWS, "C %d R %d", C, R);
        if (fused_backward(32, C, R) && (rows == 64) == fused_backward_in_two_waves(32, C, R)) CHECK(reach <= BWD_FUSED_MAX_ROWS, "C %d R %d", C, R);
        ++windows;
      }
  printf("ok %d\n", windows);
}
"""

# Every tile of every (batch, head) pair is dispatched once, in every order, of query tiles and of key tiles of any lengths.
DISPATCH = HEAD + r"""
int main() {
  int grids = 0;
  int32_t some_lengths = 1;   // head dimension 256: short windows first only where no sequence is shorter than T
  CHECK(backward_tail_256(nullptr) == SHORT_FIRST && backward_tail_256(&some_lengths) == SHORT_LAST, "order at head dimension 256");
  for (int B : {1, 2, 3, 8, 17})
    for (int H : {1, 4, 8})
      for (int T : {1, 127, 128, 129, 1000, 2048, 5000})
        for (int C : {1, 16, 50, 128, 700})
          for (int R : {0, 1, 3, 9})
            for (int rows : {64, 128, 256})
              for (Tail tail : {PLAIN, SHORT_LAST, SHORT_FIRST}) {
                FwdParams p = problem(B, H, T, std::min(C, T), std::min(R, T));
                const int64_t blocks = set_tiles(p, rows, tail);
                const int n = (T + rows - 1) / rows;
                CHECK(blocks == (int64_t)B * H * n && p.tiles.n_tiles == n, "T %d rows %d", T, rows);
                std::vector<int32_t> lens;
                for (int b = 0; b < B; ++b) lens.push_back((b * 7919 + 13) % (T + 3) - 1);
                std::vector<int> query(blocks), key(blocks), key_full(blocks);
                for (int i = 0; i < blocks; ++i) {
                  int bh = -1, t = -1, L = -1;
                  tile_coords(i, (int)blocks, p.tiles, bh, t);
                  CHECK(bh >= 0 && bh < B * H && t >= 0 && t < n, "query tile");
                  ++query[bh * n + t];
                  key_tile_coords(i, (int)blocks, p.tiles, rows, T, nullptr, 0, bh, t, L);
                  CHECK(bh >= 0 && bh < B * H && t >= 0 && t < n && L == T, "key tile");
                  ++key_full[bh * n + t];
                  key_tile_coords(i, (int)blocks, p.tiles, rows, T, lens.data(), 1, bh, t, L);
                  CHECK(bh >= 0 && bh < B * H && t >= 0 && t < n && L == std::min(std::max(lens[bh / H], 0), T), "ragged key tile");
                  ++key[bh * n + t];
                }
                for (int i = 0; i < blocks; ++i)
                  CHECK(query[i] == 1 && key[i] == 1 && key_full[i] == 1, "B %d H %d T %d C %d R %d rows %d", B, H, T, C, R, rows);
                ++grids;
              }
  printf("ok %d\n", grids);
}
"""

# What a dQ wave goes through: a tile is seen where one of its queries sees a key of it, inside where all of them see all of it, and a wave of
# padding sees nothing and has nothing inside.
QUERY_WINDOWS = HEAD + r"""
int main() {
  int waves = 0;
  for (int C : {CHUNKS})
    for (int R : {0, 1, 2, 5})
      for (int L : {1, 31, 32, 33, 127, 128, 129, 300, 700})
        for (int first = 0; first < 896; first += 32) {
          WaveWindow w{};
          bool live = false;
          for (int row = first; row < first + 32; ++row) {
            const WaveWindow mine = query_window(first, row, L, C, R, chunk_div(C));
            if (row == first) w = mine;
            CHECK(mine.lo_max == w.lo_max && mine.hi_min == w.hi_min && mine.lo_min == w.lo_min && mine.hi_max == w.hi_max, "row %d", row);
            live |= row < L;
          }
          for (int tile : {32, 64})
            for (int t = 0; t < L; t += tile) {
              bool seen = false, inside = live;
              for (int row = first; row < std::min(first + 32, L); ++row) {
                const int lo = std::max(row / C - R, 0) * C, hi = std::min((row / C + 1) * C, L);
                CHECK(query_window(first, row, L, C, R, chunk_div(C)).lo == lo && query_window(first, row, L, C, R, chunk_div(C)).hi == hi, "row %d", row);
                seen |= t < hi && t + tile > lo;
                inside &= t >= lo && t + tile <= hi;
              }
              CHECK(w.seen(t, tile) == seen, "C %d R %d L %d first %d t %d", C, R, L, first, t);
              CHECK(w.inside(t, tile) == inside, "C %d R %d L %d first %d t %d", C, R, L, first, t);
            }
          ++waves;
        }
  printf("ok %d\n", waves);
}
""".replace("CHUNKS", CHUNKS)


PROGRAMS = {"tile_order": (TILE_ORDER, 5000), "rows_in_reach": (ROWS_IN_REACH, 3000), "dispatch": (DISPATCH, 10000), "query_windows": (QUERY_WINDOWS, 10000)}


@pytest.mark.skipif(not os.path.exists(HIPCC), reason="no compiler")
@pytest.mark.parametrize("name", PROGRAMS)
def test_as_compiled(name, tmp_path):
    source, least = PROGRAMS[name]
    (tmp_path / f"{name}.hip").write_text(source)
    subprocess.run([HIPCC, "--cuda-host-only", "-O1", "-std=c++17", "-I", CSRC, f"{name}.hip", "-o", name], cwd=tmp_path, check=True)
    r = subprocess.run([str(tmp_path / name)], capture_output=True, text=True)
    assert r.returncode == 0, r.stdout
    assert r.stdout.startswith("ok ") and int(r.stdout.split()[1]) >= least, r.stdout

// The rule for 256 x 128 tiles (csrc/wide_rule.hpp) on shapes that were measured, 256 CUs.
#include <cstdio>

#include "../../kapy-lang_amd/csrc/wide_rule.hpp"

struct Row {
  long m, n, k, k_from;
  bool wide;
};

int main() {
  const Row rows[] = {
      // one round of 256 x 128 against 128 x 128 tiles: from some K on, where those run two to a CU
      {1100, 4096, 128, 512, false}, {1100, 4096, 256, 512, false}, {1100, 4096, 512, 512, true}, {2048, 4096, 128, 512, false}, {2048, 4096, 4096, 512, true},
      {1000, 8192, 1024, 2048, false}, {1000, 8192, 2048, 2048, true}, {1000, 8192, 8192, 2048, true}, {1100, 4096, 128, 0, true},
      // 128 x 128 tiles in one round: never
      {500, 8192, 4096, 0, false}, {128, 8192, 8192, 0, false},
      // against 256 x 256 tiles: three rounds against two at any K, and no longer from three of those on
      {4096, 5120, 128, 512, true}, {4096, 5120, 8192, 512, true}, {2816, 7168, 512, 2048, true}, {6144, 6144, 1024, 512, false}, {6144, 6144, 8192, 2048, false},
      {7168, 8192, 4096, 512, false}, {8192, 9216, 128, 0, false}, {8192, 8192, 8192, 0, false}, {3333, 3328, 2048, 512, false},
  };
  int bad = 0;
  for (const Row &r : rows)
    if (kapy::wide128_wins(r.m, r.n, r.k, r.k_from, 256) != r.wide) {
      std::printf("%ld x %ld, K %ld (from %ld): 256 x 128 tiles should be %s\n", r.m, r.n, r.k, r.k_from, r.wide ? "chosen" : "passed over");
      ++bad;
    }
  // fp8 tiles: 256 x 128 asked for where it does not serve is 256 x 256, as any request of 256 rows is
  using namespace kapy;
  const struct {
    int m, n;
    bool serves, wins;
    F8Tile want;
  } tiles[] = {{256, 128, true, false, kTileWide}, {256, 128, false, false, kTile256}, {256, 128, false, true, kTile256}, {256, 256, true, true, kTile256},
               {256, 0, true, true, kTile256}, {128, 128, true, true, kTile128}, {128, 0, true, true, kTile128}, {0, 0, true, true, kTileWide},
               {0, 128, true, true, kTileWide}, {0, 0, false, true, kTileFree}, {0, 0, true, false, kTileFree}, {64, 64, true, false, kTileFree}};
  for (const auto &t : tiles)
    if (f8_tile(t.m, t.n, t.serves, t.wins) != t.want) {
      std::printf("fp8 tile %d x %d (serves %d, wins %d): %d instead of %d\n", t.m, t.n, t.serves, t.wins, f8_tile(t.m, t.n, t.serves, t.wins), t.want);
      ++bad;
    }
  if (!bad) std::printf("wide rule ok\n");
  return bad != 0;
}

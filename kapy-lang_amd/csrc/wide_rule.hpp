// wide_rule.hpp — when a matrix product goes to 256 x 128 tiles.  Plain C++: the rule can be asked on the host.
#pragma once
#include <cstdint>

namespace kapy {

// 256 x 256 tiles from 0.55 of them per CU on, 128 x 128 below.  (Measured: 144 large tiles on 256 CUs beat 576 small ones -
// 3072^3: 1009 against 899 TFLOP/s - 128 do not.)
constexpr bool enough_256_tiles(int64_t m, int64_t n, int64_t cus) { return ((m + 255) / 256) * ((n + 255) / 256) * 100 >= cus * 55; }

// Rounds of tiles over the CUs decide.  A round of 256 x 128 tiles is priced at 0.62 of a round of 256 x 256 tiles (the larger ones
// read fewer LDS bytes per flop): the narrower tile wins where the wide one's only or second round leaves CUs idle, and not
// from three rounds on.  us, 256 x 256 -> 256 x 128, K = 1024 and 4096:
//   bf16 K-contiguous    4096 x 5120 (2 rounds against 3)   47.7 -> 45.4   152 -> 139      6144 x 6144 (3 : 5)  75.4 -> 76.5   237 -> 241
//                        7168 x 8192 (4 : 7)               103.4 -> 111.7  333 -> 360      8192 x 9216 (5 : 9)  129 -> 140     428 -> 474
//   bf16 row-major rhs   4096 x 5120                        49.6 -> 46.0   156 -> 140      7168 x 8192         107 -> 113     344 -> 360
//   fp8                  2816 x 7168 (2 : 3)                33.9 -> 30.7    83 -> 76       6144 x 6144          49.0 -> 51.1   125 -> 130
// Where the 256 x 256 tiles are too few and the choice is against 128 x 128: not where those fit the CUs in one round (they use
// twice as many CUs: 500 x 8192 x 4096 bf16 36.6 us against 40.9), and not below K = k_from.  At 147 KiB of LDS one workgroup has
// a CU to itself, so nothing hides its prologue and its epilogue, where 128 x 128 tiles of K-contiguous operands run two to a CU.
// us, 128 x 128 -> 256 x 128, one round of the latter:
//   K                                128           256           512          1024          2048
//   bf16 K-contiguous 1100 x 4096    6.9 ->  7.2   8.1 ->  8.1  11.3 -> 10.4  16.3 -> 14.9  25.8 -> 23.5     (k_from 512)
//                     2048 x 4096    8.0 ->  8.4  10.1 -> 10.3  13.5 -> 13.3  19.5 -> 19.1  32.9 -> 30.4
//   fp8               1000 x 8192    7.9 ->  8.7   8.4 ->  9.1  10.5 -> 10.9  13.7 -> 13.8  19.6 -> 19.2     (k_from 2048)
//                     2048 x 4096    7.9 ->  8.7   8.5 ->  9.2  10.5 -> 11.0  13.8 -> 14.0  19.5 -> 19.5
//   bf16 row-major rhs 1100 x 4096   9.3 ->  7.3  10.4 ->  8.2  14.3 -> 10.4  19.2 -> 15.8  31.3 -> 25.1     (k_from 0)
constexpr bool wide128_wins(int64_t m, int64_t n, int64_t k, int64_t k_from, int64_t cus) {
  const int64_t small = ((m + 127) / 128) * ((n + 127) / 128), tall = ((m + 255) / 256) * ((n + 127) / 128), large = ((m + 255) / 256) * ((n + 255) / 256);
  const int64_t tall_rounds = (tall + cus - 1) / cus, large_rounds = (large + cus - 1) / cus;
  if (small <= cus || tall_rounds * 124 >= large_rounds * 200) return false;
  return k >= k_from || enough_256_tiles(m, n, cus);
}

// The tile of an fp8 product: what the caller asked for (kapy_matmul_cfg: 0, 128 or 256 rows; any other request is the library's
// choice), 256 x 128 where that was asked for or wins and the kernel serves the problem.
enum F8Tile { kTileFree, kTile128, kTile256, kTileWide };
constexpr F8Tile f8_tile(int tile_m, int tile_n, bool wide_serves, bool wide_wins) {
  if (tile_m == 256) return tile_n == 128 && wide_serves ? kTileWide : kTile256;
  if (tile_m == 128) return kTile128;
  return wide_serves && wide_wins ? kTileWide : kTileFree;
}

}  // namespace kapy

// Walks the addresses of the tiled matmul kernels' loaders (csrc/operand_pieces.hpp) on the host: every piece of every K-tile of tiles
// that hang over the operand's last rows or columns, in units the kernels use, must lie inside the operand whether or not the
// buffer descriptor's range check counts the scalar part of an address, and existing elements must come from where they are.
#include <cstdio>
#include <cstdlib>
#include <initializer_list>

#include "../../kapy-lang_amd/csrc/operand_pieces.hpp"

static long checked = 0;

template <bool TR, int BK, int EB>
static void walk(int width, int left, int k, int64_t ld) {
  using P = kapy::OperandPieces<TR, BK, EB>;
  const int tiles = (k + BK - 1) / BK, k_left = k - (tiles - 1) * BK, per = 16 / EB;
  const int64_t bytes = P::bytes(k, ld, left);
  auto die = [&](const char *what, int j, int line, int first, int64_t at) {
    std::printf("%s: %s, %d-wide K-tiles of %d-byte elements: tile of %d, %d left, K %d, pitch %lld: K-tile %d line %d position %d at byte %lld of %lld\n", what,
                TR ? "transposed" : "K-contiguous", BK, EB, width, left, k, (long long)ld, j, line, first, (long long)at, (long long)bytes);
    std::exit(1);
  };
  for (int j = 0; j < tiles + 3; ++j) {  // (the kernels issue loads for up to three tiles past the last)
    const bool last = j >= tiles - 1;
    const int64_t scalar = P::tile(j, tiles, (int32_t)ld);
    for (int line = 0; line < (TR ? BK : width); ++line)
      for (int first = 0; first < (TR ? width : BK); first += per) {
        ++checked;
        if (last && k_left < BK && P::beyond_k((uint32_t)line, (uint32_t)first, k_left)) {
          if ((TR ? line : first) < k_left) die("an existing piece is masked", j, line, first, -1);
          if (scalar > bytes) die("the scalar part lies beyond the operand", j, line, first, scalar);
          continue;
        }
        const int64_t lane = P::lane((uint32_t)line * (uint32_t)ld, (uint32_t)first, (int32_t)ld, left), at = scalar + lane;
        if (at < 0 || at + 16 > bytes) die("read outside the operand", j, line, first, at);
        if (lane >= bytes || lane >= bytes - scalar) die("an existing piece fails the range check", j, line, first, at);
        const int jj = last ? tiles - 1 : j;
        const int64_t k_row = (int64_t)jj * BK + (TR ? line : first), other = TR ? first : line;
        if (other < left && at != (TR ? k_row * ld + other : other * ld + k_row) * EB) die("not the element's address", j, line, first, at);
      }
  }
}

// A loader that leaves rows that do not exist to the range check: wherever rows_end_at_descriptor allows it, every piece of such a
// row must be out of range, whether or not the check counts the scalar part.
template <int BK, int EB>
static void walk_rows(int width, int rows, int k, int64_t ld) {
  using P = kapy::OperandPieces<false, BK, EB>;
  if (!kapy::rows_end_at_descriptor(rows, ld, k, width)) return;
  const int left = rows % width ? rows % width : width, tiles = (k + BK - 1) / BK;
  const int64_t bytes = P::bytes(k, ld, left);
  for (int j = 0; j < tiles; ++j)
    for (int line = left; line < width; ++line)
      for (int first = 0; first < BK; first += 16 / EB, ++checked) {
        const int64_t lane = P::lane((uint32_t)line * (uint32_t)ld, (uint32_t)first, (int32_t)ld, width), scalar = P::tile(j, tiles, (int32_t)ld);
        if (lane >= bytes - scalar && lane >= bytes && scalar <= bytes) continue;
        std::printf("a row that does not exist is in range: %d rows in tiles of %d, K %d, pitch %lld: K-tile %d row %d position %d\n", rows, width, k, (long long)ld, j, line, first);
        std::exit(1);
      }
}

template <int BK, int EB>
static void walk_all(int width) {
  const int lefts[] = {1, 2, 7, 8, 9, 31, 32, 33, 40, 96, 104, 120, 127, 128, 129, 136, 232, 248, 255, 256, 300};
  const int ks[] = {BK, 2 * BK, 3 * BK, 2 * BK + 16 / EB, 4 * BK - 16 / EB, BK / 2, 16 / EB};
  const int odd_ks[] = {1, 7, BK + 1, 2 * BK + 33, 3 * BK - 1};
  const int per = 16 / EB;
  for (int left : lefts) {
    for (int k : ks)
      for (int64_t ld : {(int64_t)k, (int64_t)k + per, (int64_t)4 * k, (int64_t)per, (int64_t)0}) walk<false, BK, EB>(width, left, k, ld);  // (rows may overlap, or all be one row)
    for (int k : ks)
      for (int64_t ld : {(int64_t)k, (int64_t)k + per, (int64_t)4 * k, (int64_t)per, (int64_t)k - per, (int64_t)0}) walk_rows<BK, EB>(width, left, k, ld);
    if (EB != 2) continue;
    for (int k : odd_ks)  // (a line that ends inside a piece: the pitch is whole pieces)
      for (int64_t ld : {(int64_t)(k + per - 1) / per * per, (int64_t)(k + 5 * per) / per * per}) walk<false, BK, EB>(width, left, k, ld);
    for (int k : {BK, 3 * BK, 1, 7, BK + 1, 2 * BK + 33, 3 * BK - 1})
      for (int64_t ld : {(int64_t)(left + per - 1) / per * per, (int64_t)1024}) walk<true, BK, EB>(width, left, k, ld);
  }
}

int main() {
  // operands of 2^32 elements and more behind the tile
  for (int rows : {(1 << 19) + 1, (1 << 19) + 40, 1 << 20}) {
    walk<false, 64, 2>(256, rows, 192, 8192);
    walk<true, 64, 2>(256, rows, 192, (1 << 20));
    walk<false, 128, 1>(256, rows, 384, 8192);
  }
  for (int width : {64, 128, 256}) {
    walk_all<64, 2>(width);
    walk_all<32, 2>(width);
    walk_all<128, 1>(width);
  }
  std::printf("operand pieces ok: %ld pieces\n", checked);
  return 0;
}

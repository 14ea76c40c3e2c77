// operand_pieces.hpp — where the loader of a tiled matrix product reads: the per-lane and the scalar part of the address of each
// 16-byte piece of an operand tile.  Plain C++, so that the arithmetic can be walked through on the host.
#pragma once
#include <cstdint>

namespace kapy {

// The address of a piece is: first element of the tile's first line + tile() of the K-tile, a scalar + lane(), kept per lane.
// TR = false: the operand is contiguous along K (a row-major lhs, a column-major rhs).  `line` is a row (column) of the tile, `first`
// the piece's first K position within the K-tile.  TR = true: contiguous along its other extent.  `line` is a k-row of the
// K-tile, `first` the piece's first row (column) within the tile.
//
// A tile may hang over the last rows (columns) of the operand: `left` >= 1 of them exist from the tile's first on.  For one
// that does not exist the last line, or the last piece of the k-row, is read in its place - it only reaches results that are
// not stored.  Nothing is left to the buffer descriptor's range check there: the check need not count the scalar part of an
// address, and a scalar part beyond the end of the operand would turn its remainder negative.  The check is relied on for one
// thing, lanes sent to kNowhere (the pieces at and beyond K of a partial last K-tile, which must arrive as zeros): an offset no
// descriptor covers, whichever way the scalar part is counted, since tile() lies inside the operand.
template <bool TR, int BK, int EB>
struct OperandPieces {
  static constexpr int kPer = 16 / EB;  // elements per piece
  static constexpr int32_t kLines = 256;  // no tile has more rows or columns: the offset of the last existing one inside it fits 32 bits
  static constexpr uint32_t kNowhere = 0x7fffffffu;
  // (`line_at`: line * ld, so that a loader forms it once and steps it from load to load)
  static constexpr uint32_t lane(uint32_t line_at, uint32_t first, int32_t ld, int32_t left) {
    const uint32_t last = (uint32_t)(left < kLines ? left : kLines) - 1u, last_at = last * (uint32_t)ld;
    if (TR) first = first < last ? first : last / kPer * kPer;
    else line_at = line_at < last_at ? line_at : last_at;
    return (line_at + first) * EB;
  }
  // whether the whole piece lies at or beyond K, of which k_left positions are in the last K-tile
  static constexpr bool beyond_k(uint32_t line, uint32_t first, int32_t k_left) { return (int32_t)(TR ? line : first) >= k_left; }
  // scalar offset of K-tile j of `tiles` (loads for tiles past the last repeat it, into LDS nobody reads again)
  static constexpr int32_t tile(int32_t j, int32_t tiles, int32_t ld) { return (j < tiles - 1 ? j : tiles - 1) * BK * (TR ? ld : 1) * EB; }
  // bytes of the operand from the tile's first line on, the last line's last piece whole: what the descriptor covers
  static constexpr int64_t bytes(int32_t k, int64_t ld, int32_t left) {
    const int64_t elems = TR ? (int64_t)(k - 1) * ld + left : (int64_t)(left - 1) * ld + k;
    return (elems * EB + 15) & ~int64_t(15);
  }
};

// A loader that forms the offsets of a tile's rows from the first row's cannot replace single rows: it relies on the range check to
// answer the rows of a K-contiguous operand that do not exist with zeros.  They all start at or behind the operand's end only
// if rows do not overlap - whether that holds for `rows` rows cut into tiles of `tile`.
constexpr bool rows_end_at_descriptor(int64_t rows, int64_t pitch, int64_t k, int tile) { return rows % tile == 0 || pitch >= k; }

}  // namespace kapy

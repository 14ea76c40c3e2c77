// matmul_tn_f8.hip — the tiled kernel on fp8 operands.
#include "matmul_tn.hpp"
#include "wide_rule.hpp"

namespace kapy {
namespace {

template <template <int, int> class P, int BM, int BN, int BK, int WM, int WN, int S>
int launch_f8(const GemmParams &p, int lhs_fmt, int rhs_fmt, hipStream_t s) {
  // the kernel issues mfma(rhs fragment, lhs fragment): the first format selector is the rhs's
  switch (rhs_fmt * 2 + lhs_fmt) {
  case 0: return launch_tn<P<0, 0>, BM, BN, BK, WM, WN, S>(p, s);
  case 1: return launch_tn<P<0, 1>, BM, BN, BK, WM, WN, S>(p, s);
  case 2: return launch_tn<P<1, 0>, BM, BN, BK, WM, WN, S>(p, s);
  default: return launch_tn<P<1, 1>, BM, BN, BK, WM, WN, S>(p, s);
  }
}

}  // namespace

int matmul_f8_tiled(const GemmParams &p, int lhs_fmt, int rhs_fmt, int tile_m, int tile_n, hipStream_t s) {
  if (p.a_sm * 256 + p.K >= (int64_t(1) << 31) || p.b_sn * 256 + p.K >= (int64_t(1) << 31)) return KAPY_ERR_UNSUPPORTED;
  // the ring variants take any M, N >= 128 and any K >= 128 of whole 16-byte chunks (their loads are bounded by the
  // operands' ends); 256x256 tiles when there are at least 0.55 times as many of them as CUs, 128x128 (two workgroups per CU) below
  if (p.K % 16 == 0 && p.K >= 128 && p.M >= 1 && p.N >= 128) {
    // (measured at N = K = 8192: 192 of the large tiles on 256 CUs already beat 768 of the small ones, 128 do not)
    const F8Tile tile = f8_tile(tile_m, tile_n, p.K % 128 == 0 && p.N % 8 == 0 && packed_epilogue(p), p.split_k <= 1 && wide128_wins(p.M, p.N, p.K, 2048, device_cus()));
    if (tile == kTileWide) return launch_wide128_f8(p, lhs_fmt, rhs_fmt, s);
    // Overlapping rows (a pitch below K) in a tile over an edge: the ring builds would read rows that do not exist from behind the
    // operand; the four-stage build replaces them.
    if (!rows_end_at_descriptor(p.M, p.a_sm, p.K, 256) || !rows_end_at_descriptor(p.N, p.b_sn, p.K, 256))
      return p.K % 128 == 0 ? launch_f8<F8, 128, 128, 128, 2, 2, 4>(p, lhs_fmt, rhs_fmt, s) : KAPY_ERR_UNSUPPORTED;
    if (tile == kTile256 || (tile == kTileFree && enough_256_tiles(p.M, p.N, device_cus())))
      return launch_f8<F8M16, 256, 256, 128, 2, 2, kRing25>(p, lhs_fmt, rhs_fmt, s);
    // At most one 128 x 128 tile per CU and K not split: the ring build's 2.5 tiles of loads in flight are sized for two
    // workgroups per CU, and one alone waits for them (N = K = 8192, 161 .. 512 rows: 50 us whatever M is).  The four-stage
    // build has three tiles (96 KiB) in flight per workgroup: 35.6 / 36.4 / 40.0 / 41.6 / 44 us at 161 / 192 / 256 / 384 / 512
    // rows (five stages measured the same).  It fetches the last row again for rows past an operand's end.
    if (tile == kTileFree && p.split_k <= 1 && p.K % 128 == 0 && (int64_t)((p.M + 127) / 128) * ((p.N + 127) / 128) <= device_cus())
      return launch_f8<F8, 128, 128, 128, 2, 2, 4>(p, lhs_fmt, rhs_fmt, s);
    return launch_f8<F8M16, 128, 128, 128, 2, 2, kRing25>(p, lhs_fmt, rhs_fmt, s);
  }
  if (p.M % 256 == 0 && p.N % 256 == 0 && p.K % 128 == 0 && (int64_t)(p.M / 256) * (p.N / 256) * 2 >= device_cus())
    return launch_f8<F8M16, 256, 256, 128, 2, 2, kRing25>(p, lhs_fmt, rhs_fmt, s);
  if (p.M % 128 == 0 && p.N % 128 == 0 && p.K % 128 == 0) return launch_f8<F8, 128, 128, 128, 2, 2, 2>(p, lhs_fmt, rhs_fmt, s);
  return KAPY_ERR_UNSUPPORTED;
}

}  // namespace kapy

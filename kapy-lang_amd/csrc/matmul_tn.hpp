// matmul_tn.hpp — the tiled kernel for two K-contiguous operands and its launchers; instantiated for bf16, f16 and fp8 in
// matmul_tn_bf16.hip, matmul_tn_f16.hip and matmul_tn_f8.hip (one translation unit each: they take minutes to compile).
#pragma once
#include "matmul_tile.hpp"
#include "operand_pieces.hpp"

namespace kapy {
namespace {

// ---------------------------------------------------------------------------------------------
// TN kernel.  BM x BN x BK workgroup tile, WM x WN wavefronts, each owning a (BM/WM) x (BN/WN)
// block of 32x32 accumulators.  STAGES-deep LDS ring filled by LDS-direct loads.
template <typename T, int BM, int BN, int BK, int WM, int WN, int STAGES>
struct TnConfig {
  static constexpr int kWaves = WM * WN, kThreads = 64 * kWaves;
  static constexpr int kWtm = BM / WM, kWtn = BN / WN;       // wave tile
  static constexpr int kTm = kWtm / T::kM, kTn = kWtn / T::kM;  // accumulator blocks per wave
  static constexpr int kRowBytes = BK * T::kBytes;
  static constexpr int kRowsPerLoad = 1024 / kRowBytes;      // rows one LDS-direct wave instruction fills
  static constexpr int kLoadsA = BM / kRowsPerLoad, kLoadsB = BN / kRowsPerLoad;
  static constexpr int kLoadsAPerWave = kLoadsA / kWaves, kLoadsBPerWave = kLoadsB / kWaves;
  static constexpr int kStageBytes = (BM + BN) * kRowBytes;
  // STAGES == kRing25: a ring of ten quarter-tile units (half an operand tile each), i.e. 2.5 tiles
  static constexpr int kUnitBytes = kStageBytes / 4;
  static constexpr int kLdsBytes = STAGES == kRing25 ? 10 * kUnitBytes : STAGES * kStageBytes;
  static_assert(kLoadsA % kWaves == 0 && kLoadsB % kWaves == 0, "loads must divide evenly over the wavefronts");
  static_assert(kWtm % 32 == 0 && kWtn % 32 == 0 && BK % T::kSliceK == 0 && 32 % T::kM == 0, "wave tile must be a multiple of the MFMA tile");
};

template <typename T, int BM, int BN, int BK, int WM, int WN, int STAGES, bool PACKED, bool KTAIL = false, bool TAIL = false>
__global__ __launch_bounds__(64 * WM * WN) void tn_kernel(GemmParams p) {
  using C = TnConfig<T, BM, BN, BK, WM, WN, STAGES>;
  using L = TileLayout<C::kRowBytes, T>;
  constexpr int EB = T::kBytes, CH = T::kChunks;
  // Static, so that the size is a property of the code object (160 KiB, a CU's whole LDS, for the 256 x 256 ring) and no
  // launch depends on the runtime honouring a raised dynamic-LDS limit: LDS-direct loads that land outside the allocation fault.
  __shared__ __attribute__((aligned(1024))) char lds[C::kLdsBytes];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wm = wave % WM, wn = wave / WM;
  int32_t tm, tn;
  tile_of_block(p, tm, tn);
  const int32_t m0 = tm * BM, n0 = tn * BN;
  // (the 128 x 128 builds, which serve the shapes with few tiles, can split K across workgroups)
  constexpr bool kCanSplit = BM == 128 && BN == 128 && STAGES == kRing25;
  int32_t split = 0;
  if constexpr (kCanSplit) split = enter_split(p, EB);

  // Per-lane global byte offsets of the chunks this lane fetches, one per load instruction.
  // Instruction q of an operand fills LDS bytes [q*1024, q*1024+1024); this lane's 16 bytes sit at
  // q*1024 + lane*16, which the (inverse) swizzle maps back to a (row, chunk) of the tile.
  uint32_t a_goff[C::kLoadsAPerWave], b_goff[C::kLoadsBPerWave];
  // (Rows past an operand's end: the last row again, results nobody stores.  Not in the two-pass ring, which keeps the offset of the
  // first load only and leaves such rows to the descriptors; the 256-wide builds outside the ring are only given whole tiles.)
  constexpr bool kRowsReplaced = STAGES == kRing25 ? BK != T::kSliceK : BM <= 128 && BN <= 128;
  using Pieces = OperandPieces<false, BK, EB>;
#pragma unroll
  for (int i = 0; i < C::kLoadsAPerWave; ++i) {
    uint32_t row, chunk;
    L::locate((uint32_t)(wave + i * C::kWaves) * 1024u + lane * 16u, row, chunk);
    a_goff[i] = Pieces::lane(row * (uint32_t)p.a_sm, chunk * Pieces::kPer, (int32_t)p.a_sm, kRowsReplaced ? p.M - m0 : BM);
  }
#pragma unroll
  for (int i = 0; i < C::kLoadsBPerWave; ++i) {
    uint32_t row, chunk;
    L::locate((uint32_t)(wave + i * C::kWaves) * 1024u + lane * 16u, row, chunk);
    b_goff[i] = Pieces::lane(row * (uint32_t)p.b_sn, chunk * Pieces::kPer, (int32_t)p.b_sn, kRowsReplaced ? p.N - n0 : BN);
  }
  const char *a_tile = p.a + (int64_t)m0 * p.a_sm * EB;
  const char *b_tile = p.b + (int64_t)n0 * p.b_sn * EB;

  // Load instruction `idx` (0 .. loads per tile - 1) of this wavefront for K-tile kt into `stage`.
  auto issue_load = [&](int stage, int kt, int idx) {
    char *sa = lds + stage * C::kStageBytes, *sb = sa + BM * C::kRowBytes;
    if (idx < C::kLoadsAPerWave) {
      const char *ga = a_tile + (int64_t)kt * BK * EB;
      __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void *)(ga + a_goff[idx]),
                                       (__attribute__((address_space(3))) void *)(sa + (wave + idx * C::kWaves) * 1024), 16, 0, 0);
    } else {
      const int i = idx - C::kLoadsAPerWave;
      const char *gb = b_tile + (int64_t)kt * BK * EB;
      __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void *)(gb + b_goff[i]),
                                       (__attribute__((address_space(3))) void *)(sb + (wave + i * C::kWaves) * 1024), 16, 0, 0);
    }
  };
  auto issue_loads = [&](int stage, int kt) {
#pragma unroll
    for (int idx = 0; idx < C::kLoadsAPerWave + C::kLoadsBPerWave; ++idx) issue_load(stage, kt, idx);
  };

  // LDS byte offsets of this lane's operand reads, from the operand fragments of the instruction: the lane's
  // row of each KM-row block and, in K slice kk, the 16-byte chunks that hold its kpack consecutive K elements.
  constexpr int KM = T::kM;  // rows per operand block
  static_assert(T::kShape.m == KM && T::kShape.k == T::kSliceK && T::kShape.kpack * EB == 16 * CH, "policy and instruction shape disagree");
  const OperandLane frag_at = operand_lane(T::kShape, lane);
  const uint32_t frag_row = frag_at.row, frag_k0 = frag_at.k0;

  using Acc = typename T::Acc;
  constexpr int kAccRegs = KM * KM / 64;
  Acc acc[C::kTm][C::kTn];
  {
    Acc zero;
#pragma unroll
    for (int v = 0; v < kAccRegs; ++v) zero[v] = 0.f;
#pragma unroll
    for (int i = 0; i < C::kTm; ++i)
#pragma unroll
      for (int j = 0; j < C::kTn; ++j) acc[i][j] = zero;
  }

  const int KT = (p.K + BK - 1) / BK;  // (a partial last tile only in the ring variant)
  constexpr int KK = BK / T::kSliceK;                                   // matrix-instruction K-slices per tile
  constexpr int kLoadsPerTile = C::kLoadsAPerWave + C::kLoadsBPerWave;  // per wavefront
  // A fragment: the CH 16-byte chunks one lane feeds a matrix instruction for one operand block.
  struct Frag {
    u32x4 c[CH];
  };
  // Per-lane LDS offsets of the operand reads of slice kk, relative to the wave's rows of a stage.
  uint32_t frag_off[KK][CH];
#pragma unroll
  for (int kk = 0; kk < KK; ++kk)
#pragma unroll
    for (int c = 0; c < CH; ++c) frag_off[kk][c] = L::offset(frag_row, ((kk * T::kSliceK + frag_k0) * EB) / 16 + c);
  const uint32_t a_rows = (wm * C::kWtm) * C::kRowBytes, b_rows = BM * C::kRowBytes + (wn * C::kWtn) * C::kRowBytes;
  // 32-row blocks are whole multiples of the swizzle period, so block i only adds i*32*rowBytes.
  static_assert((KM * C::kRowBytes) % (256 * L::kLineParam) == 0, "an operand block must span whole swizzle periods");
  // Read `idx` of slice kk (0 .. kReads-1): the first kTm*CH are lhs row blocks, the rest rhs column blocks.
  auto read_frag = [&](int stage, int kk, int idx, Frag *af, Frag *bf) {
    const int blk = idx / CH, c = idx % CH;
    const char *base = lds + stage * C::kStageBytes + frag_off[kk][c];
    if (blk < C::kTm) af[blk].c[c] = *(const u32x4 *)(base + a_rows + blk * KM * C::kRowBytes);
    else bf[blk - C::kTm].c[c] = *(const u32x4 *)(base + b_rows + (blk - C::kTm) * KM * C::kRowBytes);
  };
  auto read_frags = [&](int stage, int kk, Frag *af, Frag *bf) {
#pragma unroll
    for (int idx = 0; idx < (C::kTm + C::kTn) * CH; ++idx) read_frag(stage, kk, idx, af, bf);
  };

  using Yes = std::integral_constant<bool, true>;
  using No = std::integral_constant<bool, false>;
  constexpr int kReads = (C::kTm + C::kTn) * CH, kMfmas = C::kTm * C::kTn;
  constexpr int kReadsPerMfma = (kReads + kMfmas - 1) / kMfmas;  // LDS reads issued behind each matrix instruction

  if constexpr (STAGES == kRing25) {
    // Ring of ten units, a unit being half an operand tile (unit u of tile j: 0/1 = upper/lower half
    // of the lhs rows, 2/3 = left/right half of the rhs columns) at ring position (4j + u) mod 10:
    // all of the 160 KiB of LDS, 2.5 tiles.  A wavefront reads exactly one lhs unit and one rhs unit.
    // There is one barrier per tile, before the tile's last K-slice; it frees the four units of tile
    // kt, and they are refilled in this order: rhs half of tile kt+2 (needed one tile time later),
    // then lhs half of tile kt+3 (needed two tile times later).  That slack lets the loads be spread
    // evenly over the whole tile time - a steady request stream into the L2 instead of every CU
    // bursting at the L1's peak rate right after the barrier - without the last ones running late.
    // Loads for tiles past the end of K are still issued (from the last real tile) into units nobody
    // reads again: every tile step is then identical and the wait counts are constants.
    //
    // The loads are LDS-direct buffer loads: per-lane 32-bit offset (loop invariant) + scalar offset
    // (the K position) + M0 (the LDS destination), so a load costs one scalar and one vector-memory
    // instruction and no vector ALU work.  Ring positions repeat every five tiles; the steady-state
    // loop is unrolled by five so that every LDS address is a constant.
    static_assert(BM == BN && WM == 2 && WN == 2, "the unit ring assumes equal lhs / rhs halves and 2 x 2 wavefronts");
    // A tile step runs in kPhases phases with the barrier before the last one.  Normally a phase is a K-slice (all
    // kTm x kTn blocks with the fragments of that slice, the next slice's fragments fetched meanwhile).  An instruction whose
    // K extent is the whole tile (16x16x128 on 128-byte rows: KK == 1) has 2 x 8 fragment registers per block pair, too many
    // to double-buffer whole; its tile runs as two passes over the halves of the rhs blocks instead: the lhs fragments stay
    // for both passes (double-buffered across tiles), the rhs halves alternate between two buffers.
    constexpr bool kNPass = KK == 1;
    static_assert(kNPass || KK % 2 == 0, "needs an even number of K-slices per tile");
    static_assert(!kNPass || C::kTn % 2 == 0, "two passes over halves of the rhs blocks");
    constexpr int kPhases = kNPass ? 2 : KK, kPhaseMfmas = kNPass ? kMfmas / 2 : kMfmas, kHalfTn = C::kTn / 2;
    constexpr int kUnit = C::kUnitBytes, kHalf = kLoadsPerTile / 2;  // loads per wavefront per operand
    static_assert(C::kLoadsAPerWave == kHalf && C::kLoadsBPerWave == kHalf && kHalf % 2 == 0, "two equal units per operand");
    constexpr int kPerUnit = kHalf / 2;
    constexpr int kEven = (kPhases * kPhaseMfmas) / kLoadsPerTile;
    constexpr int kLoadSpacing = kEven < 1 ? 1 : kEven;
    constexpr int kEarly = kPhaseMfmas / kLoadSpacing < kLoadsPerTile ? kPhaseMfmas / kLoadSpacing : kLoadsPerTile;
    static_assert((kLoadsPerTile - kEarly) * kLoadSpacing <= (kPhases - 1) * kPhaseMfmas, "late loads must go out before the barrier that waits for them");
    // reads and loads in different gaps, where a phase has enough gaps without a load for its reads at one per gap
    constexpr int kFreeGaps = kPhaseMfmas - (kPhaseMfmas + kLoadSpacing - 1) / kLoadSpacing;
    constexpr bool kSpread = kLoadSpacing > 1 && (kNPass ? (kLoadSpacing == kHalfTn && CH <= kHalfTn - 2 && kHalfTn * CH <= kFreeGaps) : kReads <= kFreeGaps);
    // The descriptors must sit in scalar registers (a descriptor in vector registers makes every load
    // a loop over its distinct values): pin the workgroup-uniform tile pointers with readfirstlane.
    auto uniform_ptr = [](const char *ptr) {
      const uint64_t v = (uint64_t)ptr;
      const uint32_t lo = __builtin_amdgcn_readfirstlane((uint32_t)v), hi = __builtin_amdgcn_readfirstlane((uint32_t)(v >> 32));
      return (void *)(((uint64_t)hi << 32) | lo);
    };
    // The descriptors end where the operands end.  In the two-pass ring, a tile that hangs over the last row of the lhs (M not a
    // multiple of BM) or of the rhs leaves the rows that do not exist to them: their row offsets are out of range (rows do
    // not overlap, matmul_tn_f8.hip), which the hardware answers with zeros in LDS instead of a fault.  (An operand with 2 GiB
    // or more behind the tile base has all of the tile's rows.)
    auto bytes_left = [&](int32_t rows, int64_t pitch) {
      const int64_t left = rows <= 0 ? 0 : ((int64_t)(rows - 1) * pitch + p.K) * EB;
      return (int)(left < 0x7fffffff ? left : 0x7fffffff);
    };
    const __amdgpu_buffer_rsrc_t a_rsrc = __builtin_amdgcn_make_buffer_rsrc(uniform_ptr(a_tile), 0, __builtin_amdgcn_readfirstlane(bytes_left(p.M - m0, p.a_sm)), 0x00020000);
    const __amdgpu_buffer_rsrc_t b_rsrc = __builtin_amdgcn_make_buffer_rsrc(uniform_ptr(b_tile), 0, __builtin_amdgcn_readfirstlane(bytes_left(p.N - n0, p.b_sn)), 0x00020000);
    const int wave_lds = wave * 1024;
    auto wrap = [](auto pos) { return pos >= 20 ? pos - 20 : (pos >= 10 ? pos - 10 : pos); };
    // ring position `pos` + D, keeping a compile-time position (an integral_constant) a compile-time position
    auto ring_add = [&](auto pos, auto d) {
      if constexpr (std::is_integral_v<decltype(pos)>) return wrap(pos + decltype(d)::value);
      else return std::integral_constant<int, (decltype(pos)::value + decltype(d)::value) % 10>{};
    };
    using Plus2 = std::integral_constant<int, 2>;
    using Plus4 = std::integral_constant<int, 4>;
    using Plus6 = std::integral_constant<int, 6>;
    // K need not be a multiple of BK (only of the 16 bytes of a chunk): the last tile is then partial, and the lanes
    // whose chunk lies past K ask for an offset beyond any descriptor, which the hardware answers with zeros in LDS.
    // Which chunk of a row a lane fetches is the same for every load it issues (the swizzle only mixes in the bit of
    // the load index that is the wavefront's own), so one mask serves all of them.
    const int k_last = (KT - 1) * BK;
    bool lane_past_k;
    {
      uint32_t row, chunk;
      L::locate((uint32_t)wave * 1024u + lane * 16u, row, chunk);
      lane_past_k = k_last + (int)(chunk * (16 / EB)) >= p.K;
    }
    constexpr int kTailFlag = (int)0x80000000;
    // (only the KTAIL build of the kernel pays the select and the mask: they cost 2 % of the aligned case)
    // Two passes: the per-lane offsets of load idx differ from load 0's by idx x (32 rows) only (the swizzle mixes in no bit of
    // the load index beyond the wavefront's own); they are formed at the load from one register per operand - through an
    // opaque add, or the compiler would keep all of them alive again - which leaves the registers to the fragments.
    auto offset_of = [&](const uint32_t(&goff)[kHalf], int idx, uint32_t row_pitch_bytes) -> uint32_t {
      if constexpr (!kNPass) return goff[idx];
      if (idx == 0) return goff[0];
      uint32_t r;
      const uint32_t delta = (uint32_t)idx * 32u * row_pitch_bytes;
      asm volatile("v_add_u32 %0, %1, %2" : "=v"(r) : "v"(goff[0]), "s"(delta));
      return r;
    };
#define KAPY_VOFF(g) ((KTAIL && soff < 0 && lane_past_k) ? kTailFlag : (int)(g))
#define KAPY_SOFF (KTAIL ? (soff & ~kTailFlag) : soff)
    // scalar byte offset of K-tile j in a row, clamped to the last real tile; the sign bit marks a partial tile
    auto k_off = [&](int j) {
      const int jj = min(j, KT - 1);
      return jj * (BK * EB) | ((KTAIL && jj == KT - 1 && k_last + BK > p.K) ? kTailFlag : 0);
    };
    const uint32_t a_pitch_bytes = (uint32_t)__builtin_amdgcn_readfirstlane((int)(p.a_sm * EB)), b_pitch_bytes = (uint32_t)__builtin_amdgcn_readfirstlane((int)(p.b_sn * EB));
    auto load_a = [&](int idx, int pos_of_unit0, int soff) {  // idx: 0 .. kHalf-1, unit idx / kPerUnit
      const int u = idx / kPerUnit, i = idx % kPerUnit;
      __builtin_amdgcn_raw_ptr_buffer_load_lds(a_rsrc, (__attribute__((address_space(3))) void *)(lds + wrap(pos_of_unit0 + u) * kUnit + i * C::kWaves * 1024 + wave_lds),
                                               16, KAPY_VOFF(offset_of(a_goff, idx, a_pitch_bytes)), KAPY_SOFF, 0, 0);
    };
    auto load_b = [&](int idx, int pos_of_unit2, int soff) {
      const int u = idx / kPerUnit, i = idx % kPerUnit;
      __builtin_amdgcn_raw_ptr_buffer_load_lds(b_rsrc, (__attribute__((address_space(3))) void *)(lds + wrap(pos_of_unit2 + u) * kUnit + i * C::kWaves * 1024 + wave_lds),
                                               16, KAPY_VOFF(offset_of(b_goff, idx, b_pitch_bytes)), KAPY_SOFF, 0, 0);
    };
#undef KAPY_VOFF
#undef KAPY_SOFF
    // Load `slot` (0 .. kLoadsPerTile-1) of the sequence issued after the barrier of the tile at ring
    // position pos0: slots [0, kHalf) = rhs units of the tile two ahead (they take positions pos0,
    // pos0+1), the rest = lhs units of the tile three ahead (positions pos0+2, pos0+3).
    auto ring_load = [&](auto pos0, int slot, int soff_b, int soff_a) {
      if (slot < kHalf) load_b(slot, pos0, soff_b);
      else load_a(slot - kHalf, pos0 + 2, soff_a);
    };
    Frag af[kNPass ? 1 : 2][C::kTm], bf[2][kNPass ? kHalfTn : C::kTn];
    // A matrix instruction every 16 (32) clocks leaves the wave 12 (28) clocks to issue anything else before the matrix
    // pipe runs dry, and a vector ALU instruction takes 8 of them, a scalar or LDS or memory instruction 4 to 8.  The
    // steady-state loop therefore computes no address: a read at a compile-time ring position is one of three copies of the
    // lane's fragment offset (the 160 KiB ring seen as 64 KiB windows, the reach of a read's immediate) plus an immediate.
    // (The build for a partial last K-tile has no registers to spare for the copies: it forms the addresses as before.)
    constexpr bool kUseWindows = !KTAIL;
    constexpr int kWindows = kUseWindows ? (C::kLdsBytes + 65535) / 65536 : 1;
    // (a tile's units start at an even ring position, so the wave's own unit - wm for the lhs, wn for the rhs - never
    // wraps on its own and can sit in the register part: one set of copies per operand)
    uint32_t frag_win[2][kWindows][KK][CH];
#pragma unroll
    for (int o = 0; o < 2; ++o)
#pragma unroll
      for (int w = 0; w < kWindows; ++w)
#pragma unroll
        for (int kk = 0; kk < KK; ++kk)
#pragma unroll
          for (int c = 0; c < CH; ++c) {
            uint32_t v = (uint32_t)(uintptr_t)lds + frag_off[kk][c] + (uint32_t)(o ? wn : wm) * kUnit + (uint32_t)w * 65536u;
            asm volatile("" : "+v"(v));  // (opaque: registers that stay, not one register and an add at every read)
            frag_win[o][w][kk][c] = v;
          }
    // The 16 bytes of chunk c, slice kk of operand o (0 lhs, 1 rhs) whose unit 0 starts at ring byte `at`, `rows` bytes in.
    auto read_at = [&](int o, auto at, uint32_t rows, int kk, int c) -> u32x4 {
      if constexpr (std::is_integral_v<decltype(at)>) {
        return *(const u32x4 *)(lds + (at + (o ? wn : wm) * kUnit + frag_off[kk][c]) + rows);
      } else if constexpr (!kUseWindows) {
        return *(const u32x4 *)(lds + (decltype(at)::value + (o ? wn : wm) * kUnit + frag_off[kk][c]) + rows);
      } else {
        const uint32_t v = decltype(at)::value + rows;
        return *(const __attribute__((address_space(3))) u32x4 *)(uintptr_t)(frag_win[o][v >> 16][kk][c] + (v & 65535u));
      }
    };
    // prologue: tiles 0 and 1 whole (lhs units first, then rhs, as the tile steps count them)
#pragma unroll
    for (int t = 0; t < 2; ++t) {
#pragma unroll
      for (int idx = 0; idx < kHalf; ++idx) load_a(idx, 4 * t, k_off(t));
#pragma unroll
      for (int idx = 0; idx < kHalf; ++idx) load_b(idx, 4 * t + 2, k_off(t));
    }
    // ... and the part of the sequence [rhs of tile 1, lhs of tile 2] that a tile step issues in the
    // last slice of the tile before (there is none before tile 0)
    constexpr int kPrologueExtra = kEarly > kHalf ? kEarly - kHalf : 0;
#pragma unroll
    for (int slot = kHalf; slot < kHalf + kPrologueExtra; ++slot) ring_load(6, slot, 0, k_off(2));
    __builtin_amdgcn_s_waitcnt(vmcnt_imm(kLoadsPerTile + kPrologueExtra));
    __builtin_amdgcn_s_barrier();  // tile 0 published
    {
      const uint32_t a0 = wm * kUnit, b0 = (2 + wn) * kUnit;
      // (two passes: the lhs blocks and the first half of the rhs blocks)
#pragma unroll
      for (int idx = 0; idx < (kNPass ? (C::kTm + kHalfTn) * CH : kReads); ++idx) {
        const int blk = idx / CH, c = idx % CH;
        if (blk < C::kTm) af[0][blk].c[c] = *(const u32x4 *)(lds + a0 + frag_off[0][c] + blk * KM * C::kRowBytes);
        else bf[0][blk - C::kTm].c[c] = *(const u32x4 *)(lds + b0 + frag_off[0][c] + (blk - C::kTm) * KM * C::kRowBytes);
      }
    }
    // One tile at ring position `pos` (an int, or an integral_constant in the unrolled loop).  The
    // sequence after the barrier of tile kt-1 is [rhs of tile kt+1, lhs of tile kt+2]; its first
    // kEarly loads went out in the last slice of tile kt-1, the rest go out in the first slices of
    // tile kt.  (`first`: tile 0, where the prologue has issued the rhs part of that sequence.)
    // (`parity`: two passes only - which lhs fragment buffer holds this tile's blocks; it alternates from tile to tile)
    auto tile_step = [&](int kt, auto pos, auto first, auto parity) {
      const auto prev = ring_add(pos, Plus6{});
      const auto next = ring_add(pos, Plus4{});
      // LDS bases of this wave's operand units in this tile and the next one
      // (ring bytes of unit 0 of each operand - compile-time constants in the unrolled loop, see read_at)
      auto unit_base = [&](auto q) {
        if constexpr (std::is_integral_v<decltype(q)>) return (uint32_t)(q * kUnit);
        else return std::integral_constant<uint32_t, (uint32_t)(decltype(q)::value * kUnit)>{};
      };
      const auto a_cur_base = unit_base(pos);
      const auto b_cur_base = unit_base(ring_add(pos, Plus2{}));
      const auto a_nxt_base = unit_base(next);
      const auto b_nxt_base = unit_base(ring_add(pos, Plus6{}));
      const int soff_late_b = k_off(kt + 1), soff_late_a = k_off(kt + 2);   // sequence of tile kt-1
      const int soff_early_b = k_off(kt + 2), soff_early_a = k_off(kt + 3); // sequence of tile kt
      auto ring_read = [&](auto a_base, auto b_base, int kk, int idx, Frag *a_dst, Frag *b_dst) {
        const int blk = idx / CH, c = idx % CH;
        if (blk < C::kTm) a_dst[blk].c[c] = read_at(0, a_base, blk * KM * C::kRowBytes, kk, c);
        else b_dst[blk - C::kTm].c[c] = read_at(1, b_base, (blk - C::kTm) * KM * C::kRowBytes, kk, c);
      };
      if constexpr (kNPass) {
        (void)parity;
        Frag *a_cur = af[0];  // one buffer: a block is fetched again (for the next tile) right behind its last use in pass 1
#pragma unroll
        for (int ph = 0; ph < 2; ++ph) {
          Frag *b_cur = bf[ph];  // pass 0: rhs blocks 0 .. kHalfTn-1, pass 1: the others
          if (ph == 1) {
            // tile kt+1 has landed once only the kHalf youngest loads (lhs of tile kt+2) are in flight; this wave's reads
            // of tile kt (the last ones went out in pass 0) have returned
            __builtin_amdgcn_s_waitcnt(vmcnt_lgkm0_imm(kHalf));
            __builtin_amdgcn_s_barrier();
          }
#pragma unroll
          for (int g = 0; g < kPhaseMfmas; ++g) {
            const int i = g / kHalfTn, j = g % kHalfTn;  // lhs-block major: block i is used kHalfTn times in a row, then rests
            T::mfma_in_place(b_cur[j].c, a_cur[i].c, acc[i][ph * kHalfTn + j]);
            if (g % kLoadSpacing != 0) __builtin_amdgcn_sched_barrier(0);  // (a load's M0 write may move ahead of the matrix instruction)
            // (a read never shares the gap behind a matrix instruction with a load: the two together, with the scalar
            // instructions a load brings, outlast the instruction, and the matrix pipe would wait for the next one)
            if (ph == 0) {  // the second half of this tile's rhs blocks, in the first gaps that carry no load
              const int r = kSpread ? (g % kLoadSpacing ? g - 1 - g / kLoadSpacing : -1) : g;
              const int blk = r / CH, c = r % CH;
              if (r >= 0 && blk < kHalfTn) bf[1][blk].c[c] = read_at(1, b_cur_base, (kHalfTn + blk) * KM * C::kRowBytes, 0, c);
            } else {
              // the next tile: lhs block i into the registers its last use has just left ...
              const int jb = kSpread ? j - 1 : j;  // (loads go out behind j == 0 when kSpread)
              if (j == kHalfTn - 1) {
#pragma unroll
                for (int c = 0; c < CH; ++c) a_cur[i].c[c] = read_at(0, a_nxt_base, i * KM * C::kRowBytes, 0, c);
              } else if (kSpread && i < kHalfTn && jb >= 0 && jb < CH) {
                // ... and the first half of its rhs blocks (block i, chunk jb) into the buffer pass 0 has left
                bf[0][i].c[jb] = read_at(1, b_nxt_base, i * KM * C::kRowBytes, 0, jb);
              } else if (!kSpread && i * (kHalfTn - 1) + j < kHalfTn * CH) {
                // (without the spread placement: the same reads, one in each gap that refills no lhs block, in order)
                const int q = i * (kHalfTn - 1) + j;
                bf[0][q / CH].c[q % CH] = read_at(1, b_nxt_base, (q / CH) * KM * C::kRowBytes, 0, q % CH);
              }
            }
            if (g % kLoadSpacing == 0) {
              const int slot = (ph * kPhaseMfmas + g) / kLoadSpacing;
              if (ph == 1 && g / kLoadSpacing < kEarly) ring_load(pos, g / kLoadSpacing, soff_early_b, soff_early_a);
              if (ph == 0 && kEarly + slot < kLoadsPerTile && (!first.value || kEarly + slot >= kHalf))
                ring_load(prev, kEarly + slot, soff_late_b, soff_late_a);
            }
            __builtin_amdgcn_sched_barrier(0);
          }
        }
        return;
      }
#pragma unroll
      for (int kk = 0; kk < KK; ++kk) {
        Frag *a_cur = af[kk & 1], *b_cur = bf[kk & 1], *a_nxt = af[(kk + 1) & 1], *b_nxt = bf[(kk + 1) & 1];
        if (kk == KK - 1) {
          // tile kt+1 has landed once only the kHalf youngest loads (lhs of tile kt+2) are in flight
          __builtin_amdgcn_s_waitcnt(vmcnt_lgkm0_imm(kHalf));
          __builtin_amdgcn_s_barrier();
        } else if constexpr (!KTAIL) {
          // this slice's fragments, asked for during the previous slice, have long returned: one wait here, which never
          // waits, instead of the compiler's own wait in each of the first gaps, where it costs the gap a third of its slots
          __builtin_amdgcn_s_waitcnt(0xC07F);
        }
#pragma unroll
        for (int g = 0; g < kMfmas; ++g) {
          const int i = g / C::kTn, j = g % C::kTn;
          acc[i][j] = T::mfma(b_cur[j].c, a_cur[i].c, acc[i][j]);
          if (KTAIL || g % kLoadSpacing != 0) __builtin_amdgcn_sched_barrier(0);  // (a load's M0 write may move ahead of the matrix instruction)
#pragma unroll
          for (int t = 0; t < kReadsPerMfma; ++t) {
            // (kSpread: one read per gap, and none in the gaps that carry a load - see the two-pass step)
            const int idx = kSpread ? (g % kLoadSpacing ? g - 1 - g / kLoadSpacing : -1) : g * kReadsPerMfma + t;
            if (idx >= 0 && idx < kReads) {
              if (kk + 1 < KK) ring_read(a_cur_base, b_cur_base, kk + 1, idx, a_nxt, b_nxt);
              else ring_read(a_nxt_base, b_nxt_base, 0, idx, a_nxt, b_nxt);
            }
          }
          if (g % kLoadSpacing == 0) {
            const int slot = (kk * kMfmas + g) / kLoadSpacing;
            if (kk == KK - 1 && g / kLoadSpacing < kEarly) ring_load(pos, g / kLoadSpacing, soff_early_b, soff_early_a);
            if (kk < KK - 1 && kEarly + slot < kLoadsPerTile && (!first.value || kEarly + slot >= kHalf))
              ring_load(prev, kEarly + slot, soff_late_b, soff_late_a);
          }
          __builtin_amdgcn_sched_barrier(0);
        }
      }
    };
    using Even = std::integral_constant<int, 0>;
    tile_step(0, std::integral_constant<int, 0>{}, Yes{}, Even{});
    int kt = 1;
    for (; kt + 5 <= KT; kt += 5) {
      tile_step(kt, std::integral_constant<int, 4>{}, No{}, Even{});
      tile_step(kt + 1, std::integral_constant<int, 8>{}, No{}, Even{});
      tile_step(kt + 2, std::integral_constant<int, 2>{}, No{}, Even{});
      tile_step(kt + 3, std::integral_constant<int, 6>{}, No{}, Even{});
      tile_step(kt + 4, std::integral_constant<int, 0>{}, No{}, Even{});
    }
    for (int pos = 4; kt < KT; ++kt) {
      tile_step(kt, pos, No{}, Even{});
      pos = wrap(pos + 4);
    }
    __builtin_amdgcn_s_waitcnt(vmcnt_imm(0));  // loads issued for tiles past the end still target this workgroup's LDS
    if constexpr (kNPass) {
      // the in-place matrix instructions are opaque to the compiler, which therefore does not count the wait states their
      // results need before another kind of instruction may read the accumulators (up to 19 for this instruction)
      asm volatile("s_nop 15\n\ts_nop 7" ::: "memory");
    }
  } else if constexpr (STAGES == 2) {
    // Two stages (the ring depth of the reference fixture, matmul.mlir:19-22).  The one barrier per
    // tile sits BEFORE the tile's last K-slice: by then every wave has fetched the fragments of that
    // last slice, so the stage is free to be refilled, and the next tile is waited for and published.
    // The last slice's matrix instructions then cover the first fragment reads of the next tile.
    //
    // Pacing of the LDS-direct loads: the CU's texture path moves 64 bytes per clock, i.e. one 1 KiB
    // wave-load per 16 clocks, 64 clocks for one load from each of the 4 waves - two matrix
    // instructions.  Issued any faster the loads back up, a wave blocks at the load instruction and
    // its matrix pipe starves.  So one load goes behind every kLoadSpacing-th matrix instruction:
    // the first ones (tile kt+2) in the last slice of tile kt, right after the barrier, the rest in
    // the first slices of tile kt+1.
    static_assert(KK >= 2 && KK % 2 == 0, "needs an even number of K-slices per tile");
    // (narrower tiles have fewer matrix instructions per load: they fall back to a denser spacing)
    constexpr int kWanted = 64 / T::kMfmaClocks, kFit = ((KK - 1) * kMfmas) / kLoadsPerTile;
    constexpr int kLoadSpacing = kFit < 1 ? 1 : (kFit < kWanted ? kFit : kWanted);
    constexpr int kEarly = kMfmas / kLoadSpacing < kLoadsPerTile ? kMfmas / kLoadSpacing : kLoadsPerTile;  // issued in the last slice
    static_assert((kLoadsPerTile - kEarly) * kLoadSpacing <= (KK - 1) * kMfmas, "late loads must go out before the barrier that waits for them");
    Frag af[2][C::kTm], bf[2][C::kTn];
    issue_loads(0, 0);
    if (KT > 1) {
      issue_loads(1, 1);
      __builtin_amdgcn_s_waitcnt(vmcnt_imm(kLoadsPerTile));
    } else {
      __builtin_amdgcn_s_waitcnt(vmcnt_imm(0));
    }
    __builtin_amdgcn_s_barrier();  // tile 0 published
    read_frags(0, 0, af[0], bf[0]);
    // has_next: tile kt+1 exists.  early: tile kt+2 exists (its first loads go out in the last slice).
    // late: the remaining loads of tile kt+1 are still to be issued (false for tile 1: the prologue did).
    auto tile_step = [&](int kt, auto has_next, auto early, auto late) {
      const int stage = kt & 1;
#pragma unroll
      for (int kk = 0; kk < KK; ++kk) {
        Frag *a_cur = af[kk & 1], *b_cur = bf[kk & 1], *a_nxt = af[(kk + 1) & 1], *b_nxt = bf[(kk + 1) & 1];
        if (kk == KK - 1) {
          if constexpr (has_next.value) {
            __builtin_amdgcn_s_waitcnt(vmcnt_lgkm0_imm(0));  // own loads of tile kt+1 landed; own reads of this stage returned
            __builtin_amdgcn_s_barrier();
          }
        }
#pragma unroll
        for (int g = 0; g < kMfmas; ++g) {
          const int i = g / C::kTn, j = g % C::kTn;
          acc[i][j] = T::mfma(b_cur[j].c, a_cur[i].c, acc[i][j]);
          __builtin_amdgcn_sched_barrier(0);
#pragma unroll
          for (int t = 0; t < kReadsPerMfma; ++t) {
            const int idx = g * kReadsPerMfma + t;
            if (idx < kReads) {
              if (kk + 1 < KK) read_frag(stage, kk + 1, idx, a_nxt, b_nxt);
              else if constexpr (has_next.value) read_frag(stage ^ 1, 0, idx, a_nxt, b_nxt);
            }
          }
          if (g % kLoadSpacing == 0) {
            const int slot = (kk * kMfmas + g) / kLoadSpacing;  // load slots counted from the start of the tile
            if constexpr (early.value)
              if (kk == KK - 1 && g / kLoadSpacing < kEarly) issue_load(stage, kt + 2, g / kLoadSpacing);
            if constexpr (late.value)
              if (kk < KK - 1 && kEarly + slot < kLoadsPerTile) issue_load(stage ^ 1, kt + 1, kEarly + slot);
          }
          __builtin_amdgcn_sched_barrier(0);
        }
      }
    };
    if (KT == 1) {
      tile_step(0, No{}, No{}, No{});
    } else {
      if (KT > 2) tile_step(0, Yes{}, Yes{}, No{});
      else tile_step(0, Yes{}, No{}, No{});
      int kt = 1;
      for (; kt + 2 < KT; ++kt) tile_step(kt, Yes{}, Yes{}, Yes{});
      if (KT > 2) tile_step(KT - 2, Yes{}, No{}, Yes{});
      tile_step(KT - 1, No{}, No{}, No{});
    }
  } else {
    // Three or more stages: the barrier at the top of iteration kt publishes tile kt+1, so the
    // fragments of the next K-slice are always fetched one slice ahead, across tile boundaries
    // (the register double-buffering of the reference fixture, matmul.mlir:51-91).
    static_assert(KK % 2 == 0, "fragment double-buffering needs an even number of K-slices per tile");
    Frag af[2][C::kTm], bf[2][C::kTn];
#pragma unroll
    for (int s = 0; s < STAGES - 1; ++s)
      if (s < KT) issue_loads(s, s);
    if (KT > STAGES - 2) __builtin_amdgcn_s_waitcnt(vmcnt_imm(kLoadsPerTile * (STAGES - 2)));
    else __builtin_amdgcn_s_waitcnt(vmcnt_imm(0));
    __builtin_amdgcn_s_barrier();  // tile 0 published
    read_frags(0, 0, af[0], bf[0]);
    int stage = 0;  // stage of tile kt
    // One tile.  HAS_NEXT: tile kt+1 exists (publish it, prefetch its first fragments).
    // LOADS: tile kt+STAGES-1 exists (request it).  The flags are compile-time so that the
    // steady-state body is branch-free and the scheduler can interleave LDS reads with MFMAs.
    auto tile_step = [&](int kt, auto has_next, auto loads) {
      const int next_stage = stage + 1 == STAGES ? 0 : stage + 1;
      if constexpr (has_next.value) {
        // own loads of tile kt+1 have landed once only the younger tiles' loads remain in flight
        if constexpr (loads.value) __builtin_amdgcn_s_waitcnt(vmcnt_lgkm0_imm(kLoadsPerTile * (STAGES - 3)));
        else __builtin_amdgcn_s_waitcnt(vmcnt_lgkm0_imm(0));
        __builtin_amdgcn_s_barrier();  // tile kt+1 published; every wave has left tile kt-1
      }
      // Source order is issue order (sched_barrier pins it): behind each of the first matrix
      // instructions of a slice goes one LDS read of the next slice's fragments and, in the first
      // slice, one LDS-direct global load, so reads have the rest of the slice to land.
      static_assert(KK * kMfmas >= kLoadsPerTile, "not enough matrix instructions per tile to pace the global loads");
#pragma unroll
      for (int kk = 0; kk < KK; ++kk) {
        Frag *a_cur = af[kk & 1], *b_cur = bf[kk & 1], *a_nxt = af[(kk + 1) & 1], *b_nxt = bf[(kk + 1) & 1];
#pragma unroll
        for (int g = 0; g < kMfmas; ++g) {
          const int i = g / C::kTn, j = g % C::kTn;
          acc[i][j] = T::mfma(b_cur[j].c, a_cur[i].c, acc[i][j]);
          __builtin_amdgcn_sched_barrier(0);
#pragma unroll
          for (int t = 0; t < kReadsPerMfma; ++t) {
            const int idx = g * kReadsPerMfma + t;
            if (idx < kReads) {
              if (kk + 1 < KK) read_frag(stage, kk + 1, idx, a_nxt, b_nxt);
              else if constexpr (has_next.value) read_frag(next_stage, 0, idx, a_nxt, b_nxt);
            }
          }
          // the tile's LDS-direct loads are spread one per matrix instruction over the whole tile
          if constexpr (has_next.value && loads.value)
            if (kk * kMfmas + g < kLoadsPerTile) issue_load(stage == 0 ? STAGES - 1 : stage - 1, kt + STAGES - 1, kk * kMfmas + g);
          __builtin_amdgcn_sched_barrier(0);
        }
      }
      stage = next_stage;
    };
    int kt = 0;
    for (; kt + STAGES - 1 < KT; ++kt) tile_step(kt, Yes{}, Yes{});
    for (; kt + 1 < KT; ++kt) tile_step(kt, Yes{}, No{});
    tile_step(kt, No{}, No{});
  }

  if constexpr (kCanSplit) {
    if (p.split_k > 1) {
      __builtin_amdgcn_s_waitcnt(vmcnt_lgkm0_imm(0));
      __builtin_amdgcn_s_barrier();  // every wave has left the ring
      if (!split_k_meet<C::kThreads>(p, tm + tn * p.tiles_m, split, acc, m0 + wm * C::kWtm, KM, (uint32_t *)lds)) return;
    }
  }
  if constexpr (PACKED) {
    static_assert(PackedEpilogue<KM, C::kWtm, C::kWtn>::kBytesPerWave * C::kWaves <= C::kLdsBytes, "two strips per wavefront must fit the ring");
    __builtin_amdgcn_s_waitcnt(vmcnt_lgkm0_imm(0));
    __builtin_amdgcn_s_barrier();  // every wave has left the ring: it is reused as staging space
    PackedEpilogue<KM, C::kWtm, C::kWtn>::template run<TAIL>(p, acc, lds + wave * PackedEpilogue<KM, C::kWtm, C::kWtn>::kBytesPerWave, m0 + wm * C::kWtm,
                                              n0 + wn * C::kWtn, lane);
  } else {
#pragma unroll
    for (int i = 0; i < C::kTm; ++i)
#pragma unroll
      for (int j = 0; j < C::kTn; ++j) store_block_generic(p, m0 + wm * C::kWtm + i * KM, n0 + wn * C::kWtn + j * KM, lane, acc[i][j]);
  }
}

template <typename T, int BM, int BN, int BK, int WM, int WN, int STAGES, bool PACKED, bool KTAIL = false, bool TAIL = false>
int launch_tn_epi(GemmParams p, hipStream_t s) {
  using C = TnConfig<T, BM, BN, BK, WM, WN, STAGES>;
  auto kernel = tn_kernel<T, BM, BN, BK, WM, WN, STAGES, PACKED, KTAIL, TAIL>;
  p.tiles_m = (p.M + BM - 1) / BM;  // (only the ring variants are launched with tiles that hang over an edge)
  p.tiles_n = (p.N + BN - 1) / BN;
  constexpr bool kCanSplit = BM == 128 && BN == 128 && STAGES == kRing25;
  if (!kCanSplit) p.split_k = 1;
  if constexpr (C::kLdsBytes > 64 * 1024) {
    // A kernel whose LDS-direct loads address more than the 64 KiB every runtime grants: before its first launch on a device,
    // ask the runtime what it will give it - the code object's static size must be the kernel's own and within the device's
    // limit per workgroup - and refuse instead of launching loads that would land outside the workgroup's allocation.
    static int checked[kMaxDevices];  // 0 not asked, 1 fine, -1 refused (a race between two first calls only repeats the query)
    int dev = -1;
    KAPY_HIP_CHECK(hipGetDevice(&dev));
    if (dev < 0 || dev >= kMaxDevices) return fail(KAPY_ERR_UNSUPPORTED, "matmul: device ordinal %d beyond %d", dev, kMaxDevices);
    int state = __atomic_load_n(&checked[dev], __ATOMIC_ACQUIRE);
    if (state == 0) {
      hipFuncAttributes attr;
      int limit = 0;
      const hipError_t e1 = hipFuncGetAttributes(&attr, reinterpret_cast<const void *>(kernel));
      const hipError_t e2 = hipDeviceGetAttribute(&limit, hipDeviceAttributeMaxSharedMemoryPerBlock, dev);
      state = (e1 == hipSuccess && e2 == hipSuccess && (int64_t)attr.sharedSizeBytes == (int64_t)C::kLdsBytes && limit >= C::kLdsBytes) ? 1 : -1;
      (void)hipGetLastError();
      __atomic_store_n(&checked[dev], state, __ATOMIC_RELEASE);
    }
    if (state < 0) return fail(KAPY_ERR_HIP, "matmul: the runtime does not give this kernel the %d bytes of LDS it addresses (nothing was launched)", C::kLdsBytes);
  }
  kernel<<<dim3((unsigned)(p.tiles_m * p.tiles_n), (unsigned)p.split_k), dim3(C::kThreads), 0, s>>>(p);
  KAPY_HIP_CHECK(hipGetLastError());
  return KAPY_OK;
}


template <typename T, int BM, int BN, int BK, int WM, int WN, int STAGES>
int launch_tn(const GemmParams &p, hipStream_t s) {
  // a result that ends inside a 16-byte piece of a row takes the bounds-checked element stores
  // (tiles that hang over the edge: the ring builds' loads are bounded, the others fetch the last row again; the strip stores
  // are bounded for all of them)
  const bool whole_tiles = (p.M % BM == 0 && p.N % BN == 0) || ((STAGES == kRing25 || BM <= 128) && p.N % 8 == 0);
  const bool packed = packed_epilogue(p) && whole_tiles;
  if (host_has_tail(p)) {
    // a fused elementwise tail: the ring kernels on the 16x16 instruction have builds with it in the packed epilogue,
    // every other variant applies it in the element stores
    if constexpr (STAGES == kRing25 && T::kM == 16) {
      if (packed) return p.K % BK ? launch_tn_epi<T, BM, BN, BK, WM, WN, STAGES, true, true, true>(p, s) : launch_tn_epi<T, BM, BN, BK, WM, WN, STAGES, true, false, true>(p, s);
    }
    if constexpr (STAGES == kRing25) {
      if (p.K % BK) return launch_tn_epi<T, BM, BN, BK, WM, WN, STAGES, false, true>(p, s);
    }
    return launch_tn_epi<T, BM, BN, BK, WM, WN, STAGES, false>(p, s);
  }
  if constexpr (STAGES == kRing25) {
    if (p.K % BK)  // a partial last K-tile: the build of the kernel that masks the lanes past K
      return packed ? launch_tn_epi<T, BM, BN, BK, WM, WN, STAGES, true, true>(p, s) : launch_tn_epi<T, BM, BN, BK, WM, WN, STAGES, false, true>(p, s);
  }
  return packed ? launch_tn_epi<T, BM, BN, BK, WM, WN, STAGES, true>(p, s) : launch_tn_epi<T, BM, BN, BK, WM, WN, STAGES, false>(p, s);
}

}  // namespace
}  // namespace kapy

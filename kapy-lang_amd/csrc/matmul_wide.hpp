// matmul_wide.hpp — the tiled kernel with 256 rows per workgroup tile: 256 x 256 tiles for the operand layouts that need transposing
// LDS reads, 256 x 128 tiles for every layout.  Instantiated per element type and tile in matmul_wide_*.hip (they take minutes to
// compile).
//
// 4 wavefronts (2 x 2) with a wave tile of 128 x BN/2.  An operand is staged as it lies in memory by LDS-direct buffer loads (the
// cp_async of CpAsyncOpToLLVM.cpp:22-186).  K-contiguous (a row-major lhs, a column-major rhs): rows of 128 bytes under the tiled
// kernel's swizzle, read 16 bytes per lane.  Contiguous along its other extent (a column-major lhs, a row-major rhs): for each 128
// rows or columns an image [64 k-rows][128 elements] with 16-byte chunk c of k-row r at chunk c ^ transposed_key(r), the operand registers
// made on the way out of LDS by ds_read_b64_tr_b16 (the ldmatrix.trans of LdMatrixOpToLLVM.cpp:128-129).
//
// One barrier per K-tile, before the tile's second and last K-slice: by then every wave holds that slice's fragments, so the stage is
// free, and the loads of the tile STAGES further on go out into it.  Two stages of 64 KiB (256 x 256): all of them behind the matrix
// instructions of that last slice, with the next tile's first slice to land.  Three stages of 48 KiB (256 x 128): half of them
// there, half in the first slice of the next tile, with a whole tile time more to land - its slices are half as long.
//
// What bounds it: 256 x 256, the matrix cores at the clock the power limit leaves (matrix pipe busy for 88 % of the wave clocks at
// 8192^3); 256 x 128 with one tile per CU, what nothing else on that CU covers - first loads, epilogue, waits for loads (matrix pipe busy
// for 73 .. 75 % of the wave clocks with 64 K-tiles; LDS reads for 0.41 of the matrix clocks, 0.26 on 256 x 256 tiles; no bank
// conflicts in the loop).  Measured, 128 x 128 tiles (or the operands turned first) -> here: fp8 1000 x 8192 x 8192 60 -> 52 us;
// bf16 2048 x 4096 x 4096 row-major 63.5 -> 54, two transposed operands 66 -> 56; 8192^3 with two transposed operands, fp32 result,
// 0.84 ms for the turns and the product -> 0.74.
#pragma once
#include "matmul_tile.hpp"
#include "operand_pieces.hpp"

namespace kapy {
namespace {

// Waits for the transposing reads whose results sit in h0[j], h1[j] and hands those registers back as its own results (the
// registers of a read still pending must not be touched by anything before this).
__device__ __forceinline__ void wide_tr_wait(u32x2_lds (&h0)[4], u32x2_lds (&h1)[4]) { tr_reads_wait(h0, h1); }
__device__ __forceinline__ void wide_tr_wait(u32x2_lds (&h0)[8], u32x2_lds (&h1)[8]) {
  asm volatile("s_waitcnt lgkmcnt(0)"
               : "+v"(h0[0]), "+v"(h0[1]), "+v"(h0[2]), "+v"(h0[3]), "+v"(h0[4]), "+v"(h0[5]), "+v"(h0[6]), "+v"(h0[7]), "+v"(h1[0]), "+v"(h1[1]),
                 "+v"(h1[2]), "+v"(h1[3]), "+v"(h1[4]), "+v"(h1[5]), "+v"(h1[6]), "+v"(h1[7])
               :
               : "memory");
}

// A K-slice has G matrix instructions; what goes into the gap behind each: a load, spread evenly, or reads of the next slice's
// fragments, one per gap in the gaps without a load, first come - or, where those are too few, as many as needed in every gap.
constexpr int wide_load_at(int g, int loads, int G) {
  for (int i = 0; i < loads; ++i)
    if (i * G / loads == g) return i;
  return -1;
}
constexpr int wide_free_before(int g, int loads, int G) {
  int n = 0;
  for (int x = 0; x < g; ++x) n += wide_load_at(x, loads, G) < 0;
  return n;
}
struct WideReads {
  int first, count;
};
constexpr WideReads wide_reads_at(int g, int reads, int loads, int G) {
  if (reads <= G - loads) return {wide_free_before(g, loads, G), wide_load_at(g, loads, G) < 0 && wide_free_before(g, loads, G) < reads ? 1 : 0};
  const int per = (reads + G - 1) / G, left = reads - g * per;
  return {g * per, left <= 0 ? 0 : left < per ? left : per};
}

constexpr int kWideBM = 256;
constexpr int wide_stages(int bn) { return bn == 256 ? 2 : 3; }
constexpr int wide_lds_bytes(int bn) { return wide_stages(bn) * (kWideBM + bn) * 128; }

// TAIL: the build for calls with a fused elementwise tail (scale, bias, activation in the strip epilogue).
// KTAIL: K is not a multiple of the K-tile.  Of the last tile, the 16-byte pieces (K-contiguous operand; K a multiple of 8 then) or
// k-rows (transposed operand) beyond K are given an offset no descriptor covers, so that zeros arrive in their place; the switch
// is made once, when the last tile's loads come up.
template <typename T, int BN, bool A_TR, bool B_TR, bool TAIL, bool KTAIL>
__global__ __launch_bounds__(256) void wide_kernel(GemmParams p) {
  constexpr int EB = T::kBytes, CH = T::kChunks, KM = T::kM, BM = kWideBM, BK = 128 / EB, KK = BK / T::kSliceK;
  constexpr int kStages = wide_stages(BN), kImageB = BM * 128, kStageBytes = (BM + BN) * 128, kRowTr = 256, kHalfTr = 16384;
  constexpr int kTm = 128 / KM, kTn = BN / 2 / KM, kMfmas = kTm * kTn;
  constexpr int kLoadsA = BM / 32, kLoadsB = BN / 32, kLoads = kLoadsA + kLoadsB;  // LDS-direct loads per wavefront and K-tile
  constexpr int kEarly = kStages == 2 ? kLoads : kLoads / 2;                       // of them in the slice behind the barrier
  static_assert(KK == 2 && (!(A_TR || B_TR) || (EB == 2 && KM == 16)) && !(KTAIL && EB != 2), "two slices per K-tile; transposed operands and partial K-tiles in 16 bits");
  using L = TileLayout<128, T, KM>;
  static_assert(16 % L::kLineParam == 0 && (KM * 128) % (256 * L::kLineParam) == 0, "the swizzle key must depend neither on the load instruction nor on the block");
  __shared__ __attribute__((aligned(1024))) char lds[kStages * kStageBytes];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wm = wave & 1, wn = wave >> 1;
  int32_t tm, tn;
  tile_of_block(p, tm, tn);
  const int32_t m0 = tm * BM, n0 = tn * BN;
  const int KT = __builtin_amdgcn_readfirstlane(KTAIL ? (p.K + BK - 1) / BK : p.K / BK);
  // elements between neighbours along the staged rows' other extent: between rows (K-contiguous) or between k-rows (transposed)
  const int32_t a_ld = __builtin_amdgcn_readfirstlane((int32_t)(A_TR ? p.a_sk : p.a_sm)), b_ld = __builtin_amdgcn_readfirstlane((int32_t)(B_TR ? p.b_sk : p.b_sn));

  // Per-lane global byte offsets of the 16-byte pieces this lane fetches, one per load instruction: instruction q of an operand fills
  // bytes [(wave + 4q) * 1024, + 1024) of its image, 32 rows (K-contiguous) or 16 k-rows and, from q = 4 on, the other 128 rows or
  // columns (transposed) further on than instruction 0's - no key mixes in a bit that q changes.
  const uint32_t my_byte = (uint32_t)wave * 1024u + lane * 16u;
  uint32_t kc_row, kc_chunk;
  L::locate(my_byte, kc_row, kc_chunk);
  const uint32_t tr_krow = my_byte / kRowTr, tr_chunk = ((my_byte % kRowTr) / 16) ^ transposed_key(tr_krow);
  // (the lines and pieces a tile that hangs over an edge reads in place of those that do not exist: operand_pieces.hpp)
  using PiecesA = OperandPieces<A_TR, BK, EB>;
  using PiecesB = OperandPieces<B_TR, BK, EB>;
  auto line_of = [&](bool tr, int q) -> uint32_t { return tr ? tr_krow + 16 * (q % 4) : kc_row + 32 * q; };
  auto first_of = [&](bool tr, int q) -> uint32_t { return tr ? tr_chunk * 8 + 128 * (q / 4) : kc_chunk * (16 / EB); };
  uint32_t a_goff[kLoadsA], b_goff[kLoadsB];
  const uint32_t a_line0 = line_of(A_TR, 0) * (uint32_t)a_ld, b_line0 = line_of(B_TR, 0) * (uint32_t)b_ld;
#pragma unroll
  for (int q = 0; q < kLoadsA; ++q) a_goff[q] = PiecesA::lane(a_line0 + (uint32_t)((A_TR ? 16 * (q % 4) : 32 * q) * a_ld), first_of(A_TR, q), a_ld, p.M - m0);
#pragma unroll
  for (int q = 0; q < kLoadsB; ++q) b_goff[q] = PiecesB::lane(b_line0 + (uint32_t)((B_TR ? 16 * (q % 4) : 32 * q) * b_ld), first_of(B_TR, q), b_ld, p.N - n0);
  auto enter_k_tail = [&]() __attribute__((always_inline)) {
    const int32_t k_left = p.K - (KT - 1) * BK;
#pragma unroll
    for (int q = 0; q < kLoadsA; ++q) a_goff[q] = PiecesA::beyond_k(line_of(A_TR, q), first_of(A_TR, q), k_left) ? PiecesA::kNowhere : a_goff[q];
#pragma unroll
    for (int q = 0; q < kLoadsB; ++q) b_goff[q] = PiecesB::beyond_k(line_of(B_TR, q), first_of(B_TR, q), k_left) ? PiecesB::kNowhere : b_goff[q];
  };
  auto uniform_ptr = [](const char *ptr) {
    const uint64_t v = (uint64_t)ptr;
    const uint32_t lo = __builtin_amdgcn_readfirstlane((uint32_t)v), hi = __builtin_amdgcn_readfirstlane((uint32_t)(v >> 32));
    return (void *)(((uint64_t)hi << 32) | lo);
  };
  const int64_t a_left = PiecesA::bytes(p.K, A_TR ? p.a_sk : p.a_sm, p.M - m0), b_left = PiecesB::bytes(p.K, B_TR ? p.b_sk : p.b_sn, p.N - n0);
  const __amdgpu_buffer_rsrc_t a_rsrc = __builtin_amdgcn_make_buffer_rsrc(uniform_ptr(p.a + (int64_t)m0 * (A_TR ? 1 : p.a_sm) * EB), 0,
                                                                          __builtin_amdgcn_readfirstlane((int)(a_left < 0x7fffffff ? a_left : 0x7fffffff)), 0x00020000);
  const __amdgpu_buffer_rsrc_t b_rsrc = __builtin_amdgcn_make_buffer_rsrc(uniform_ptr(p.b + (int64_t)n0 * (B_TR ? 1 : p.b_sn) * EB), 0,
                                                                          __builtin_amdgcn_readfirstlane((int)(b_left < 0x7fffffff ? b_left : 0x7fffffff)), 0x00020000);
  const int wave_lds = wave * 1024;
  // load instruction idx (the lhs ones, then the rhs ones) of this wavefront for the K-tile at scalar offsets soff_a / soff_b
  auto issue_load = [&](int soff_a, int soff_b, int stage, int idx) __attribute__((always_inline)) {
    if (idx < kLoadsA)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(a_rsrc, (__attribute__((address_space(3))) void *)(lds + stage * kStageBytes + idx * 4096 + wave_lds), 16,
                                               (int)a_goff[idx], soff_a, 0, 0);
    else
      __builtin_amdgcn_raw_ptr_buffer_load_lds(b_rsrc, (__attribute__((address_space(3))) void *)(lds + stage * kStageBytes + kImageB + (idx - kLoadsA) * 4096 + wave_lds),
                                               16, (int)b_goff[idx - kLoadsA], soff_b, 0, 0);
  };
  auto soff_a_of = [&](int j) { return PiecesA::tile(j, KT, a_ld); };
  auto soff_b_of = [&](int j) { return PiecesB::tile(j, KT, b_ld); };

  // Operand reads, from the operand fragments of the instruction.  K-contiguous: row frag.row of each KM-row block, the 16-byte chunks
  // that hold its kpack consecutive K elements of the slice.  Transposed: the transposing read hands lane j of a 16-lane group
  // element j of the four k-rows whose 8-byte pieces the group's lanes address, so lane l16 addresses k-row 8 * grp + 4 * h + l16 / 4,
  // elements 4 * (l16 % 4) .. of the block.  One address register per stage and slice chunk (K-contiguous) or per stage and block
  // (transposed: the key enters by XOR); the rest is an immediate.
  const OperandLane frag_at = operand_lane(T::kShape, lane);
  const uint32_t grp = frag_at.k0 / T::kShape.kpack, l16 = frag_at.row;
  const uint32_t tr_row = 8 * grp + (l16 >> 2), tr_key = transposed_key(tr_row);  // (the key is the same for every slice and half)
  auto tr_at = [&](int first, int blk) -> uint32_t {  // `first`: the wave's first row or column of the tile
    return (first / 128) * kHalfTr + tr_row * kRowTr + ((((first % 128) / 8 + blk * 2 + ((l16 & 3) >> 1)) ^ tr_key) * 16) + (l16 & 1) * 8;
  };
  auto kc_at = [&](int first, int kk, int c) -> uint32_t { return L::offset(first + l16, ((kk * T::kSliceK + frag_at.k0) * EB) / 16 + c); };
  constexpr int kRegsA = A_TR ? kTm : KK * CH, kRegsB = B_TR ? kTn : KK * CH;
  uint32_t a_at[kStages][kRegsA], b_at[kStages][kRegsB];
#pragma unroll
  for (int st = 0; st < kStages; ++st) {
#pragma unroll
    for (int x = 0; x < kRegsA; ++x) {
      uint32_t v = (uint32_t)(uintptr_t)lds + st * kStageBytes + (A_TR ? tr_at(wm * 128, x) : kc_at(wm * 128, x / CH, x % CH));
      asm volatile("" : "+v"(v));  // (opaque: registers that stay, not one register and an add at every read)
      a_at[st][x] = v;
    }
#pragma unroll
    for (int x = 0; x < kRegsB; ++x) {
      uint32_t v = (uint32_t)(uintptr_t)lds + st * kStageBytes + kImageB + (B_TR ? tr_at(wn * (BN / 2), x) : kc_at(wn * (BN / 2), x / CH, x % CH));
      asm volatile("" : "+v"(v));
      b_at[st][x] = v;
    }
  }
  struct Frags {
    u32x4 a[A_TR ? 1 : kTm][CH], b[B_TR ? 1 : kTn][CH];
    u32x2_lds ah0[kTm], ah1[kTm], bh0[kTn], bh1[kTn];  // (used for transposed operands only)
  };
  constexpr int kReadsA = kTm * (A_TR ? 2 : CH), kReadsB = kTn * (B_TR ? 2 : CH), kReads = kReadsA + kReadsB;
  // read r (0 .. kReads - 1) of slice KKc of stage STc: the lhs blocks, then the rhs blocks
  auto read_op = [&](auto stage_c, auto kk_c, auto r_c, Frags &dst) __attribute__((always_inline)) {
    constexpr int st = decltype(stage_c)::value, kk = decltype(kk_c)::value, r = decltype(r_c)::value;
    if constexpr (r < kReadsA) {
      if constexpr (A_TR && r < kTm) dst.ah0[r] = tr_read_b64_at<(uint32_t)(kk * 32 * kRowTr)>(a_at[st][r]);
      else if constexpr (A_TR) dst.ah1[r - kTm] = tr_read_b64_at<(uint32_t)(kk * 32 * kRowTr + 4 * kRowTr)>(a_at[st][r - kTm]);
      else dst.a[r / CH][r % CH] = *(const __attribute__((address_space(3))) u32x4 *)(uintptr_t)(a_at[st][kk * CH + r % CH] + (uint32_t)(r / CH) * KM * 128);
    } else {
      constexpr int x = r - kReadsA;
      if constexpr (B_TR && x < kTn) dst.bh0[x] = tr_read_b64_at<(uint32_t)(kk * 32 * kRowTr)>(b_at[st][x]);
      else if constexpr (B_TR) dst.bh1[x - kTn] = tr_read_b64_at<(uint32_t)(kk * 32 * kRowTr + 4 * kRowTr)>(b_at[st][x - kTn]);
      else dst.b[x / CH][x % CH] = *(const __attribute__((address_space(3))) u32x4 *)(uintptr_t)(b_at[st][kk * CH + x % CH] + (uint32_t)(x / CH) * KM * 128);
    }
  };

  using Acc = typename T::Acc;
  Acc acc[kTm][kTn];
  {
    Acc zero;
#pragma unroll
    for (int v = 0; v < KM * KM / 64; ++v) zero[v] = 0.f;
#pragma unroll
    for (int i = 0; i < kTm; ++i)
#pragma unroll
      for (int j = 0; j < kTn; ++j) acc[i][j] = zero;
  }

  // prologue: tiles 0 .. STAGES - 2 and the early part of tile STAGES - 1
#pragma unroll
  for (int t = 0; t < kStages; ++t) {
    if (KTAIL && t == KT - 1) enter_k_tail();
#pragma unroll
    for (int idx = 0; idx < (t < kStages - 1 ? kLoads : kEarly); ++idx) issue_load(soff_a_of(t), soff_b_of(t), t, idx);
  }
  __builtin_amdgcn_s_waitcnt(vmcnt_imm((kStages - 2) * kLoads + kEarly));
  __builtin_amdgcn_s_barrier();  // tile 0 published
  Frags fr[2];
  using Zero = std::integral_constant<int, 0>;
  static_for<kReads>([&](auto r) __attribute__((always_inline)) { read_op(Zero{}, Zero{}, r, fr[0]); });

  // One K-tile in stage STAGE (compile time: every LDS address is then a register plus an immediate).
  auto tile_step = [&](int kt, auto stage_c) __attribute__((always_inline)) {
    constexpr int stage = decltype(stage_c)::value, next_stage = (stage + 1) % kStages, late_stage = (stage + kStages - 1) % kStages;
    int soff_a = __builtin_amdgcn_readfirstlane(soff_a_of(kt + kStages)), soff_b = __builtin_amdgcn_readfirstlane(soff_b_of(kt + kStages));
    int late_a = __builtin_amdgcn_readfirstlane(soff_a_of(kt + kStages - 1)), late_b = __builtin_amdgcn_readfirstlane(soff_b_of(kt + kStages - 1));
    asm volatile("" : "+s"(soff_a), "+s"(soff_b), "+s"(late_a), "+s"(late_b));
    static_for<2>([&](auto kk_c) __attribute__((always_inline)) {
      constexpr int kk = decltype(kk_c)::value, kLoadsHere = kk ? kEarly : kLoads - kEarly;
      constexpr bool last = kk == 1;
      Frags &cur = fr[kk], &nxt = fr[kk ^ 1];
      if constexpr (last) {
        // own loads of tile kt+1 have landed (those of younger tiles may be in flight) and own reads of this stage have returned
        // (the last slice's fragments among them: they were asked for during the slice before); then every wave's have
        __builtin_amdgcn_s_waitcnt(vmcnt_lgkm0_imm((kStages - 2) * kLoads));
        __builtin_amdgcn_s_barrier();
        if (KTAIL && kt + kStages == KT - 1) enter_k_tail();
      } else if constexpr (!A_TR && !B_TR) {
        __builtin_amdgcn_s_waitcnt(0xC07F);  // lgkmcnt(0): one wait, which never waits, instead of the compiler's in each of the first gaps
      }
      if constexpr (A_TR) wide_tr_wait(cur.ah0, cur.ah1);
      if constexpr (B_TR) wide_tr_wait(cur.bh0, cur.bh1);
      static_for<kMfmas>([&](auto g_c) __attribute__((always_inline)) {
        constexpr int g = decltype(g_c)::value, i = g / kTn, j = g % kTn;
        u32x4 a_op[CH], b_op[CH];
        if constexpr (A_TR) a_op[0] = u32x4{cur.ah0[i][0], cur.ah0[i][1], cur.ah1[i][0], cur.ah1[i][1]};
        else
#pragma unroll
          for (int c = 0; c < CH; ++c) a_op[c] = cur.a[i][c];
        if constexpr (B_TR) b_op[0] = u32x4{cur.bh0[j][0], cur.bh0[j][1], cur.bh1[j][0], cur.bh1[j][1]};
        else
#pragma unroll
          for (int c = 0; c < CH; ++c) b_op[c] = cur.b[j][c];
        T::mfma_in_place(b_op, a_op, acc[i][j]);
        __builtin_amdgcn_sched_barrier(0);
        constexpr WideReads reads = wide_reads_at(g, kReads, kLoadsHere, kMfmas);
        static_for<reads.count>([&](auto t) __attribute__((always_inline)) {
          using RS = std::integral_constant<int, (last ? next_stage : stage)>;
          using RK = std::integral_constant<int, (last ? 0 : 1)>;
          read_op(RS{}, RK{}, std::integral_constant<int, reads.first + decltype(t)::value>{}, nxt);
        });
        constexpr int load = wide_load_at(g, kLoadsHere, kMfmas);
        if constexpr (load >= 0 && last) issue_load(soff_a, soff_b, stage, load);
        else if constexpr (load >= 0) issue_load(late_a, late_b, late_stage, kEarly + load);
        __builtin_amdgcn_sched_barrier(0);
      });
    });
  };
  int kt = 0;
  for (; kt + kStages <= KT; kt += kStages)
    static_for<kStages>([&](auto u) __attribute__((always_inline)) { tile_step(kt + decltype(u)::value, u); });
  // (Every step ends with the reads of the next step's first slice in flight.  A step that does not run waits in its place: the
  // compiler does not know that the registers of transposing reads are pending.)
  static_for<kStages - 1>([&](auto u) __attribute__((always_inline)) {
    if (kt + decltype(u)::value < KT) tile_step(kt + decltype(u)::value, u);
    else asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
  });
  // (nobody waits for the last step's reads but this; the loads issued for tiles past the end of K still target this workgroup's LDS)
  asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
  __builtin_amdgcn_s_waitcnt(vmcnt_lgkm0_imm(0));
  // the in-place matrix instructions are opaque to the compiler, which therefore does not count the wait states their
  // results need before another kind of instruction may read the accumulators
  asm volatile("s_nop 15\n\ts_nop 7" ::: "memory");
  __builtin_amdgcn_s_barrier();  // every wave has left the stages: they are reused as staging space by the strip epilogue
  using Epilogue = PackedEpilogue<KM, 128, BN / 2>;
  static_assert(Epilogue::kBytesPerWave * 4 <= kStages * kStageBytes, "a strip per wavefront must fit the stages");
  Epilogue::template run<TAIL>(p, acc, lds + wave * Epilogue::kBytesPerWave, m0 + wm * 128, n0 + wn * (BN / 2), lane);
}

template <typename T, int BN, bool A_TR, bool B_TR, bool TAIL, bool KTAIL>
int launch_wide_build(GemmParams p, hipStream_t s) {
  auto kernel = wide_kernel<T, BN, A_TR, B_TR, TAIL, KTAIL>;
  p.tiles_m = (p.M + kWideBM - 1) / kWideBM;
  p.tiles_n = (p.N + BN - 1) / BN;
  p.split_k = 1;
  // Before the first launch on a device: the runtime must give the kernel the LDS its loads address.
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
    state = (e1 == hipSuccess && e2 == hipSuccess && (int64_t)attr.sharedSizeBytes == wide_lds_bytes(BN) && limit >= wide_lds_bytes(BN)) ? 1 : -1;
    (void)hipGetLastError();
    __atomic_store_n(&checked[dev], state, __ATOMIC_RELEASE);
  }
  if (state < 0) return fail(KAPY_ERR_HIP, "matmul: the runtime does not give this kernel the %d bytes of LDS it addresses (nothing was launched)", wide_lds_bytes(BN));
  kernel<<<dim3((unsigned)(p.tiles_m * p.tiles_n), 1), dim3(256), 0, s>>>(p);
  KAPY_HIP_CHECK(hipGetLastError());
  return KAPY_OK;
}

// The 16-bit builds of one tile width: a row-major rhs beside a row-major lhs, a row-major rhs beside a column-major lhs (without a
// fused tail) and, 256 x 128 only, two K-contiguous operands (whole K-tiles).
template <typename T, int BN>
int launch_wide_16bit(const GemmParams &p, bool a_tr, bool b_tr, hipStream_t s) {
  const bool tail = host_has_tail(p), k_tail = p.K % 64 != 0;
  if (a_tr) return k_tail ? launch_wide_build<T, BN, true, true, false, true>(p, s) : launch_wide_build<T, BN, true, true, false, false>(p, s);
  if (b_tr) {
    if (tail) return k_tail ? launch_wide_build<T, BN, false, true, true, true>(p, s) : launch_wide_build<T, BN, false, true, true, false>(p, s);
    return k_tail ? launch_wide_build<T, BN, false, true, false, true>(p, s) : launch_wide_build<T, BN, false, true, false, false>(p, s);
  }
  if constexpr (BN == 128) return tail ? launch_wide_build<T, BN, false, false, true, false>(p, s) : launch_wide_build<T, BN, false, false, false, false>(p, s);
  return fail(KAPY_ERR_INVALID, "matmul: no such tile configuration");
}

}  // namespace
}  // namespace kapy

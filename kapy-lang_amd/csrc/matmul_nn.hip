// matmul_nn.hip — the tiled kernel for 16-bit operands of which at least one is contiguous along its other extent, or whose lines end
// inside a 16-byte piece (128 x 128 tiles).
#include "matmul_tile.hpp"
#include "operand_pieces.hpp"

namespace kapy {
namespace {

// ---------------------------------------------------------------------------------------------
// NN kernel: 128 x 128 x BK tiles of operands in any layout with 16-byte aligned lines along the contiguous axis (A_TR / B_TR below),
// any N and K, any M of a K-contiguous lhs, M a multiple of 8 of a transposed one.  4 wavefronts (2x2), wave tile 64x64 = 4x4
// blocks of the 16x16x32 instruction.  An operand tile is staged as it lies in memory - a transposed one as [BK][128] - by
// LDS-direct buffer loads; the K-contiguous operand registers that the matrix instruction wants of a transposed operand are
// made on the way out of LDS by ds_read_b64_tr_b16: a 16-lane group hands in 16 addresses of 8 bytes (4 k-rows x 16 columns) and
// lane i gets column i of the four rows.  This replaces the ldmatrix.trans of the reference (LdMatrixOpToLLVM.cpp:128-129).
// STAGES-deep ring; the barrier at the top of iteration kt publishes tile kt+1 and frees the stage of
// tile kt-1 for the loads of tile kt+STAGES-1.  Loads past the end of K re-read the last tile into
// a stage nobody reads again, so every iteration is identical.
constexpr int kNBM = 128, kNBN = 128;

// A_TR / B_TR: how each operand lies in memory and in LDS.  false: K-contiguous (a row-major lhs, a column-major rhs): rows
// of BK elements staged under the tiled kernel's swizzle and read 16 bytes per lane.  true: contiguous along its other
// extent (a column-major lhs, a row-major rhs): k-rows of 128 elements staged as they lie and read with the transposing
// read.  <false, true> is the reference fixture's row-major x row-major; <false, false> is the tiled kernel's business
// except where lines end inside a 16-byte piece, which its ring does not cut.
// KTAIL: K is not a multiple of BK.  The loads of the last K-tile are then issued with the per-lane offsets of the
// 16-byte pieces (K-contiguous operand) or k-rows (transposed operand) beyond K moved out of the descriptor's range, so that
// zeros arrive in their place; the switch is made once, beside a barrier, when the last tile's loads come up.
template <typename T, int BK, int STAGES, bool PACKED, bool A_TR = false, bool B_TR = true, bool KTAIL = false, bool RAG_N = false>
__global__ __launch_bounds__(256) void nn_kernel(GemmParams p) {
  static_assert(T::kM == 16 && T::kBytes == 2 && BK % 32 == 0 && STAGES >= 3, "16x16x32 instruction, 16-bit operands");
  static_assert(A_TR || B_TR || KTAIL, "two K-contiguous operands are the tiled kernel's, but for lines that end inside a 16-byte piece");
  using LA = TileLayout<BK * 2, T, 16>;
  constexpr int kRowKc = BK * 2, kRowTr = 128 * 2;   // bytes per staged row: a row / column of BK elements, or a k-row of 128
  constexpr int kBytesOp = 128 * BK * 2, kBytesA = kBytesOp, kStage = 2 * kBytesOp;
  constexpr int kLoadsOp = kBytesOp / 1024 / 4, kLoads = 2 * kLoadsOp;  // per wavefront per tile
  constexpr int KK = BK / 32, kTm = 4, kTn = 4, kMfmas = kTm * kTn;
  static_assert(kNBM == 128 && kNBN == 128, "both operands stage 128 rows, columns or elements per k-row");
  __shared__ __attribute__((aligned(1024))) char lds[STAGES * kStage];  // static: see tn_kernel
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wm = wave & 1, wn = wave >> 1;
  int32_t tm, tn;
  tile_of_block(p, tm, tn);
  const int32_t m0 = tm * kNBM, n0 = tn * kNBN;
  const int32_t split = enter_split(p, 2);
  // (a scalar: in the builds whose epilogue calls the element store out of line the parameters live in scratch memory, and a
  // count read back from there would make every branch on it a vector compare)
  const int KT = __builtin_amdgcn_readfirstlane(KTAIL ? (p.K + BK - 1) / BK : p.K / BK);
  // elements between neighbours along the staged rows' other extent: between rows (K-contiguous) or between k-rows (transposed)
  const int32_t a_ld = (int32_t)(A_TR ? p.a_sk : p.a_sm), b_ld = (int32_t)(B_TR ? p.b_sk : p.b_sn);

  // Per-lane global byte offsets of the 16-byte pieces this lane fetches, one per load instruction (instruction q of an operand
  // fills LDS bytes [q*1024, q*1024 + 1024) of its image), with what a tile that hangs over an edge reads in place of rows, columns
  // and pieces that do not exist (operand_pieces.hpp).
  using PiecesA = OperandPieces<A_TR, BK, 2>;
  using PiecesB = OperandPieces<B_TR, BK, 2>;
  // Row (k-row) and first element along it of the piece that instruction 0 brings this lane; instruction q's is as many rows further on
  // as 4 KiB hold (no key mixes in a bit that q changes).
  constexpr int kStepKc = 4096 / kRowKc, kStepTr = 4096 / kRowTr;
  static_assert(16 % LA::kLineParam == 0 && kStepTr % 16 == 0, "the pieces of one lane must lie at one place along their rows");
  const uint32_t my_byte = (uint32_t)wave * 1024u + lane * 16u;
  uint32_t kc_row, kc_chunk;
  LA::locate(my_byte, kc_row, kc_chunk);
  const uint32_t tr_krow = my_byte / kRowTr, tr_chunk = ((my_byte % kRowTr) / 16) ^ transposed_key(tr_krow);
  const uint32_t a_first = (A_TR ? tr_chunk : kc_chunk) * 8, b_first = (B_TR ? tr_chunk : kc_chunk) * 8;
  const uint32_t a_line0 = (A_TR ? tr_krow : kc_row) * (uint32_t)a_ld, b_line0 = (B_TR ? tr_krow : kc_row) * (uint32_t)b_ld;
  uint32_t a_goff[kLoadsOp], b_goff[kLoadsOp];
#pragma unroll
  for (int q = 0; q < kLoadsOp; ++q) {
    a_goff[q] = PiecesA::lane(a_line0 + (uint32_t)(q * (A_TR ? kStepTr : kStepKc) * a_ld), a_first, a_ld, p.M - m0);
    b_goff[q] = PiecesB::lane(b_line0 + (uint32_t)(q * (B_TR ? kStepTr : kStepKc) * b_ld), b_first, b_ld, p.N - n0);
  }
  // From the last K-tile on (the loads past the end of K repeat it): pieces at or beyond K get an offset no descriptor covers.
  // (a K-contiguous operand's line does not matter here: its first element is its K position)
  auto enter_k_tail = [&]() __attribute__((always_inline)) {
    const int32_t k_left = p.K - (KT - 1) * BK;
#pragma unroll
    for (int q = 0; q < kLoadsOp; ++q) {
      a_goff[q] = PiecesA::beyond_k(tr_krow + q * kStepTr, a_first, k_left) ? PiecesA::kNowhere : a_goff[q];
      b_goff[q] = PiecesB::beyond_k(tr_krow + q * kStepTr, b_first, k_left) ? PiecesB::kNowhere : b_goff[q];
    }
  };
  // (KTAIL) Of a K-contiguous operand the piece that K ends inside has arrived with what lies behind K: this lane's copy of it in the
  // last K-tile's stage is cut to zeros from K on - other lanes' products with it are zeros times whatever lies there, which
  // may be a NaN.  Between the wait for the tile's loads and the barrier that publishes it.
  auto cut_k_tail = [&](int stage) __attribute__((always_inline)) {
    const int32_t k_left = p.K - (KT - 1) * BK;
#pragma unroll
    for (int q = 0; q < kLoadsOp; ++q) {
      char *piece = lds + stage * kStage + q * 4096 + wave * 1024 + lane * 16;
#pragma unroll
      for (int e = 1; e < 8; ++e) {
        const int32_t from = k_left - (int32_t)kc_chunk * 8;   // (one compare per element: the piece K ends inside has 1 .. 7 left)
        if (from > 0 && from <= e) {
          if constexpr (!A_TR) ((uint16_t *)piece)[e] = 0;
          if constexpr (!B_TR) ((uint16_t *)(piece + kBytesA))[e] = 0;
        }
      }
    }
  };
  auto uniform_ptr = [](const char *ptr) {
    const uint64_t v = (uint64_t)ptr;
    const uint32_t lo = __builtin_amdgcn_readfirstlane((uint32_t)v), hi = __builtin_amdgcn_readfirstlane((uint32_t)(v >> 32));
    return (void *)(((uint64_t)hi << 32) | lo);
  };
  const int64_t a_left = PiecesA::bytes(p.K, A_TR ? p.a_sk : p.a_sm, p.M - m0), b_left = PiecesB::bytes(p.K, B_TR ? p.b_sk : p.b_sn, p.N - n0);
  const __amdgpu_buffer_rsrc_t a_rsrc = __builtin_amdgcn_make_buffer_rsrc(uniform_ptr(p.a + (int64_t)m0 * (A_TR ? 1 : p.a_sm) * 2), 0,
                                                                          __builtin_amdgcn_readfirstlane((int)(a_left < 0x7fffffff ? a_left : 0x7fffffff)), 0x00020000);
  const __amdgpu_buffer_rsrc_t b_rsrc = __builtin_amdgcn_make_buffer_rsrc(uniform_ptr(p.b + (int64_t)n0 * (B_TR ? 1 : p.b_sn) * 2), 0,
                                                                          __builtin_amdgcn_readfirstlane((int)(b_left < 0x7fffffff ? b_left : 0x7fffffff)), 0x00020000);
  const int wave_lds = wave * 1024;
  // (the scalar offsets of K-tile j, clamped to the last tile: loads past the end of K are still issued, into stages nobody reads)
  auto soff_a_of = [&](int j) { return PiecesA::tile(j, KT, a_ld); };
  auto soff_b_of = [&](int j) { return PiecesB::tile(j, KT, b_ld); };
  auto issue_load_at = [&](int soff_a, int soff_b, int stage, int idx) __attribute__((always_inline)) {
    if (idx < kLoadsOp)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(a_rsrc, (__attribute__((address_space(3))) void *)(lds + stage * kStage + idx * 4096 + wave_lds), 16,
                                               (int)a_goff[idx], soff_a, 0, 0);
    else
      __builtin_amdgcn_raw_ptr_buffer_load_lds(b_rsrc, (__attribute__((address_space(3))) void *)(lds + stage * kStage + kBytesA + (idx - kLoadsOp) * 4096 + wave_lds),
                                               16, (int)b_goff[idx - kLoadsOp], soff_b, 0, 0);
  };
  auto issue_load = [&](int j, int stage, int idx) __attribute__((always_inline)) { issue_load_at(soff_a_of(j), soff_b_of(j), stage, idx); };

  // Operand reads, from the operand fragments of the instruction (l16: the lane's row of an lhs block = its column of
  // an rhs block; grp: which 8 of a slice's 32 K positions its registers hold).  K-contiguous operand: row / column l16 of each
  // 16-wide block, 16-byte chunk 4*kk + grp.  Transposed operand: the transposing read hands lane j of a 16-lane group element j
  // of the four k-rows whose 8-byte pieces the group's lanes address, so lane l16 addresses k-row (8*grp + 4*h + l16/4),
  // elements 4*(l16%4).. of the block.
  const OperandLane frag_at = operand_lane(T::kShape, lane);
  const uint32_t grp = frag_at.k0 / T::kShape.kpack, l16 = frag_at.row;
  static_assert((16 * kRowKc) % (256 * LA::kLineParam) == 0, "an operand block must span whole swizzle periods");
  const uint32_t tr_row = 8 * grp + (l16 >> 2), tr_key = transposed_key(tr_row);  // the key is the same for every kk and h
  // Byte offset, inside an operand's image of a stage, of this lane's read for block `blk` (transposed) or slice kk (K-contiguous)
  // of the wave's half `w` of the operand.
  auto tr_off = [&](int w, int blk) { return tr_row * kRowTr + (((w * 8 + blk * 2 + ((l16 & 3) >> 1)) ^ tr_key) * 16) + (l16 & 1) * 8; };
  auto kc_off = [&](int w, int kk) { return LA::offset(w * 64 + l16, 4 * kk + grp); };
  // a transposed operand's fragment comes out of LDS as two 8-byte halves (k-rows +0..3 and +4..7 of the lane's K-group)
  // (kept as two arrays of halves per fragment buffer, the form the wait for these reads takes its operands in)
  struct Frags {
    u32x4 c[4];               // K-contiguous operand: one 16-byte read per block
    u32x2_lds h0[4], h1[4];   // transposed operand
  };
  static_assert(kTm == 4 && kTn == 4, "tr_reads_wait takes the halves of four fragments");
  // Every operand read of the main loop is `register + immediate`: the stage is a compile-time constant there (the loop is
  // unrolled over the ring), and where the ring is longer than a read's 64 KiB immediate reaches, the per-lane offsets
  // are kept once per 64 KiB window (a vector add per read would cost the matrix pipe more than the read itself).
  constexpr int kWindows = (STAGES * kStage + 65535) / 65536;
  constexpr int kRegsA = A_TR ? kTm : KK, kRegsB = B_TR ? kTn : KK;
  uint32_t a_win[kWindows][kRegsA], b_win[kWindows][kRegsB];
#pragma unroll
  for (int w = 0; w < kWindows; ++w) {
#pragma unroll
    for (int x = 0; x < kRegsA; ++x) {
      uint32_t v = (uint32_t)(uintptr_t)lds + (A_TR ? tr_off(wm, x) : kc_off(wm, x)) + (uint32_t)w * 65536u;
      asm volatile("" : "+v"(v));  // (opaque: registers that stay, not one register and an add at every read)
      a_win[w][x] = v;
    }
#pragma unroll
    for (int x = 0; x < kRegsB; ++x) {
      uint32_t v = (uint32_t)(uintptr_t)lds + kBytesA + (B_TR ? tr_off(wn, x) : kc_off(wn, x)) + (uint32_t)w * 65536u;
      asm volatile("" : "+v"(v));
      b_win[w][x] = v;
    }
  }
  // read `r` (0 .. 3) of slice kk of the stage: block r of the operand
  auto read_op = [&](auto is_b, auto stage, auto kk, auto blk, Frags &dst) __attribute__((always_inline)) {
    constexpr bool kIsB = decltype(is_b)::value, kTr = kIsB ? B_TR : A_TR;
    constexpr int b = decltype(blk)::value;
    auto win = [&](uint32_t w, int x) { if constexpr (kIsB) return b_win[w][x]; else return a_win[w][x]; };
    if constexpr (kTr) {
      constexpr uint32_t c0 = decltype(stage)::value * kStage + decltype(kk)::value * 32 * kRowTr, c1 = c0 + 4 * kRowTr;
      dst.h0[b] = tr_read_b64_at<(c0 & 65535u)>(win(c0 >> 16, b));
      dst.h1[b] = tr_read_b64_at<(c1 & 65535u)>(win(c1 >> 16, b));
    } else {
      constexpr uint32_t c = decltype(stage)::value * kStage + (uint32_t)b * 16 * kRowKc;
      dst.c[b] = *(const __attribute__((address_space(3))) u32x4 *)(uintptr_t)(win(c >> 16, decltype(kk)::value) + (c & 65535u));
    }
  };
  using IsA = std::integral_constant<bool, false>;
  using IsB = std::integral_constant<bool, true>;
  auto operand_of = [](auto tr, const Frags &f, int b) __attribute__((always_inline)) -> u32x4 {
    if constexpr (decltype(tr)::value) return u32x4{f.h0[b][0], f.h0[b][1], f.h1[b][0], f.h1[b][1]};
    else return f.c[b];
  };
  using ATr = std::integral_constant<bool, A_TR>;
  using BTr = std::integral_constant<bool, B_TR>;

  using Acc = typename T::Acc;
  Acc acc[kTm][kTn];
#pragma unroll
  for (int i = 0; i < kTm; ++i)
#pragma unroll
    for (int j = 0; j < kTn; ++j) acc[i][j] = Acc{0.f, 0.f, 0.f, 0.f};

#pragma unroll
  for (int j = 0; j < STAGES - 1; ++j) {
    if (KTAIL && j == KT - 1) enter_k_tail();
#pragma unroll
    for (int idx = 0; idx < kLoads; ++idx) issue_load(j, j, idx);
  }
  __builtin_amdgcn_s_waitcnt(vmcnt_imm(kLoads * (STAGES - 2)));
  const bool cut = KTAIL && (!A_TR || !B_TR) && (p.K & 7) != 0;
  if (cut && KT == 1) {
    cut_k_tail(0);
    __builtin_amdgcn_s_waitcnt(0xC07F);  // lgkmcnt(0)
  }
  __builtin_amdgcn_s_barrier();  // tile 0 published
  Frags af[2], bf[2];
  using Zero = std::integral_constant<int, 0>;
  static_for<kTm>([&](auto i) { read_op(IsA{}, Zero{}, Zero{}, i, af[0]); });
  static_for<kTn>([&](auto j) { read_op(IsB{}, Zero{}, Zero{}, j, bf[0]); });

  constexpr int kReads = kTm + kTn;
  constexpr int kLoadSpacing = (KK * kMfmas) / kLoads;  // matrix instructions between two loads
  static_assert(kLoadSpacing >= 2 && kReads <= kMfmas - (kMfmas + kLoadSpacing - 1) / kLoadSpacing, "a slice has a gap without a load for each of its reads");
  // (Every lambda that touches the fragment buffers is always_inline.  Left to its cost model the compiler once kept tile_step
  // out of line in one build - both operands transposed, 64-deep, partial last K-tile - and the buffers it captures by
  // reference then live in scratch memory: registers with a transposing read still pending were stored there before their
  // data had arrived, and the products were wrong.)
  // One K-tile in ring stage STAGE (a type: every LDS address of the step is then a constant).  `parity` says which
  // fragment buffer holds slice 0 of this tile: with an odd number of slices per tile it alternates from tile to tile.
  // What goes behind which matrix instruction follows the tiled kernel's rule: a read never shares a gap with a load,
  // and a load's gap is left to the scheduler, which moves the M0 write ahead of the matrix instruction.
  auto tile_step = [&](int kt, auto stage_c, auto parity) __attribute__((always_inline)) {
    constexpr int stage = decltype(stage_c)::value, par = decltype(parity)::value;
    constexpr int next_stage = stage + 1 == STAGES ? 0 : stage + 1, free_stage = stage == 0 ? STAGES - 1 : stage - 1;
    // (the scalar offsets of this step's loads are formed here, beside the barrier, not in the gaps of the loads)
    int soff_a = __builtin_amdgcn_readfirstlane(soff_a_of(kt + STAGES - 1)), soff_b = __builtin_amdgcn_readfirstlane(soff_b_of(kt + STAGES - 1));
    asm volatile("" : "+s"(soff_a), "+s"(soff_b));
    if (KTAIL && kt + STAGES - 1 == KT - 1) enter_k_tail();
    // own loads of tile kt+1 have landed once only the younger tiles' loads remain in flight
    __builtin_amdgcn_s_waitcnt(vmcnt_lgkm0_imm(kLoads * (STAGES - 3)));
    if (cut && kt + 1 == KT - 1) {
      cut_k_tail(next_stage);
      __builtin_amdgcn_s_waitcnt(0xC07F);  // lgkmcnt(0)
    }
    __builtin_amdgcn_s_barrier();  // tile kt+1 published; every wave has left tile kt-1
    static_for<KK>([&](auto kk_c) __attribute__((always_inline)) {
      constexpr int kk = decltype(kk_c)::value;
      Frags &a_cur = af[(kk + par) & 1], &a_nxt = af[(kk + par + 1) & 1];
      Frags &b_cur = bf[(kk + par) & 1], &b_nxt = bf[(kk + par + 1) & 1];
      // the transposed fragments of this slice were requested during the previous one
      if constexpr (A_TR) tr_reads_wait(a_cur.h0, a_cur.h1);
      if constexpr (B_TR) tr_reads_wait(b_cur.h0, b_cur.h1);
      static_for<kMfmas>([&](auto g_c) __attribute__((always_inline)) {
        constexpr int g = decltype(g_c)::value, i = g / kTn, j = g % kTn;
        constexpr bool load_here = (kk * kMfmas + g) % kLoadSpacing == kLoadSpacing - 1 && (kk * kMfmas + g) / kLoadSpacing < kLoads;
        const u32x4 a_op = operand_of(ATr{}, a_cur, i), b_op = operand_of(BTr{}, b_cur, j);
        T::mfma_in_place(&b_op, &a_op, acc[i][j]);
        if constexpr (!load_here) __builtin_amdgcn_sched_barrier(0);
        constexpr int r = load_here ? -1 : g - (g + 1) / kLoadSpacing;  // this gap's read: the gaps without a load, in order
        if constexpr (r >= 0 && r < kReads) {
          using RS = std::integral_constant<int, (kk + 1 < KK ? stage : next_stage)>;
          using RK = std::integral_constant<int, (kk + 1 < KK ? kk + 1 : 0)>;
          if constexpr (r < kTm) read_op(IsA{}, RS{}, RK{}, std::integral_constant<int, r>{}, a_nxt);
          else read_op(IsB{}, RS{}, RK{}, std::integral_constant<int, r - kTm>{}, b_nxt);
        }
        if constexpr (load_here) issue_load_at(soff_a, soff_b, free_stage, (kk * kMfmas + g) / kLoadSpacing);
        __builtin_amdgcn_sched_barrier(0);
      });
    });
  };
  // the loop is unrolled over the ring (and over the fragment-buffer parity)
  constexpr int kUnroll = (KK & 1) && (STAGES & 1) ? 2 * STAGES : STAGES;
  int kt = 0;
  for (; kt + kUnroll <= KT; kt += kUnroll)
    static_for<kUnroll>([&](auto u) __attribute__((always_inline)) { tile_step(kt + decltype(u)::value, std::integral_constant<int, decltype(u)::value % STAGES>{}, std::integral_constant<int, (decltype(u)::value * KK) & 1>{}); });
  // Every step ends with the transposing reads of the NEXT step's first slice in flight, and only that step waits for them.  A
  // step that does not run (past the last K-tile) waits in its place, first thing, and so does the end of the kernel: the
  // compiler does not know that those registers are pending and, once nobody reads them any more, hands them out again - a
  // late result would land on top of the new value.  (These waits name no register: an asm operand may be given another
  // register than the read's, and the copy into it would itself read the pending one.  That no instruction names a pending
  // register before its wait is checked on the library's machine code by the build tests.)
  static_for<kUnroll - 1>([&](auto u) __attribute__((always_inline)) {
    if (kt + decltype(u)::value < KT)
      tile_step(kt + decltype(u)::value, std::integral_constant<int, decltype(u)::value % STAGES>{}, std::integral_constant<int, (decltype(u)::value * KK) & 1>{});
    else if constexpr (A_TR || B_TR)
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
  });
  __builtin_amdgcn_s_waitcnt(vmcnt_lgkm0_imm(0));
  // the in-place matrix instructions are opaque to the compiler, which therefore does not count the wait states their
  // results need before another kind of instruction may read the accumulators
  asm volatile("s_nop 15\n\ts_nop 7" ::: "memory");
  __builtin_amdgcn_s_barrier();  // every wave has left the ring: it is reused as staging space by the packed epilogue
  if (p.split_k > 1 && !split_k_meet<256>(p, tm + tn * p.tiles_m, split, acc, m0 + wm * 64, 16, (uint32_t *)lds)) return;
  if constexpr (PACKED) {
    static_assert(PackedEpilogue<16, 64, 64>::kBytesPerWave * 4 <= STAGES * kStage, "two strips per wavefront must fit the ring");
    PackedEpilogue<16, 64, 64>::template run<false, RAG_N>(p, acc, lds + wave * PackedEpilogue<16, 64, 64>::kBytesPerWave, m0 + wm * 64, n0 + wn * 64, lane);
  } else {
#pragma unroll
    for (int i = 0; i < kTm; ++i)
#pragma unroll
      for (int j = 0; j < kTn; ++j) store_block_generic(p, m0 + wm * 64 + i * 16, n0 + wn * 64 + j * 16, lane, acc[i][j]);
  }
}

template <typename T, int BK, int STAGES, bool A_TR = false, bool B_TR = true, bool KTAIL = false>
int launch_nn(GemmParams p, hipStream_t s) {
  p.tiles_m = (p.M + kNBM - 1) / kNBM;
  p.tiles_n = (p.N + kNBN - 1) / kNBN;
  const bool packed = packed_epilogue(p) && !host_has_tail(p);  // (a fused tail goes through the element stores here)
  dim3 grid((unsigned)(p.tiles_m * p.tiles_n), (unsigned)p.split_k);
  if (packed && p.N % 8) nn_kernel<T, BK, STAGES, true, A_TR, B_TR, KTAIL, true><<<grid, dim3(256), 0, s>>>(p);
  else if (packed) nn_kernel<T, BK, STAGES, true, A_TR, B_TR, KTAIL><<<grid, dim3(256), 0, s>>>(p);
  else nn_kernel<T, BK, STAGES, false, A_TR, B_TR, KTAIL><<<grid, dim3(256), 0, s>>>(p);
  KAPY_HIP_CHECK(hipGetLastError());
  return KAPY_OK;
}

}  // namespace

// form: 0 lhs K-contiguous x rhs transposed, 1 both transposed, 2 lhs transposed x rhs K-contiguous, 3 (k_tail only) both K-contiguous.
int launch_nn_config(const GemmParams &p, bool bf16, int form, int bk, int stages, bool k_tail, hipStream_t s) {
#define KAPY_NN_FORMS(BK, ST, KT)                                                                                                             \
  switch (form + (bf16 ? 0 : 3)) {                                                                                                            \
  case 0: return launch_nn<Bf16M16, BK, ST, false, true, KT>(p, s);                                                                           \
  case 1: return launch_nn<Bf16M16, BK, ST, true, true, KT>(p, s);                                                                            \
  case 2: return launch_nn<Bf16M16, BK, ST, true, false, KT>(p, s);                                                                           \
  case 3: return launch_nn<F16M16, BK, ST, false, true, KT>(p, s);                                                                            \
  case 4: return launch_nn<F16M16, BK, ST, true, true, KT>(p, s);                                                                             \
  default: return launch_nn<F16M16, BK, ST, true, false, KT>(p, s);                                                                           \
  }
  if (k_tail && form == 3) {
    if (bk == 64) return bf16 ? launch_nn<Bf16M16, 64, 4, false, false, true>(p, s) : launch_nn<F16M16, 64, 4, false, false, true>(p, s);
    return bf16 ? launch_nn<Bf16M16, 32, 4, false, false, true>(p, s) : launch_nn<F16M16, 32, 4, false, false, true>(p, s);
  }
  if (k_tail) {
    if (bk == 64) { KAPY_NN_FORMS(64, 4, true) }
    KAPY_NN_FORMS(32, 4, true)
  }
  if (bk == 64 && stages == 4) { KAPY_NN_FORMS(64, 4, false) }
  if (bk == 64) { KAPY_NN_FORMS(64, 3, false) }
  KAPY_NN_FORMS(32, 4, false)
#undef KAPY_NN_FORMS
}

}  // namespace kapy

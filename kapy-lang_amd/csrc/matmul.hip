// matmul.hip — kapy.matmul over whole views on CDNA4 matrix cores (f16 / bf16 operands).
//
// Reference: kapy.matmul (include/kapy/Dialect/Kapy/IR/Ops.td:416-439, verifier
// lib/Dialect/Kapy/IR/Kapy.cpp:451-574) lowered by MatmulOpToLLVM.cpp:58-311 to mma.sync, fed by
// the cp.async ring of CpAsyncOpToLLVM.cpp:22-186 and ldmatrix (LdMatrixOpToLLVM.cpp:21-174);
// the kernel shape is the fixture test/Conversion/KapyToKgpu/matmul.mlir: a 2-stage shared-memory
// ring, fragments prefetched one k-slice ahead, one barrier per wait.
//
// gfx950 counterparts used here:
//   mma.sync m16n8k16          -> v_mfma_f32_32x32x16_{f16,bf16} (fp32 accumulate)
//   cp.async + wait_group      -> global_load_lds_dwordx4 (16 B per lane, written straight into
//                                 LDS) + s_waitcnt vmcnt
//   per-lane swizzled cp.async destination (CpAsyncOpToLLVM.cpp:124-139)
//                              -> the destination of an LDS-direct load is wave-contiguous, so the
//                                 XOR swizzle is applied to WHICH global chunk a lane fetches; the
//                                 LDS image is the same swizzled one
//   ldmatrix                   -> ds_read_b128 of 8 K-contiguous elements per lane
//   swizzle (4,8) for 32 banks -> searched at compile time for 64 banks from the MFMA operand
//                                 layout (layout.hpp first_swizzle)
//
// Kernels:
//   tn_kernel      both operands contiguous along K (lhs row-major, rhs column-major): the roofline path (matmul_tn.hpp).
//   nn_kernel      an operand contiguous along its other extent, read with transposing LDS reads (matmul_nn.hip).
//   wide_kernel    256-row tiles: 256 x 256 for an operand contiguous along its other extent, 256 x 128 for any (matmul_wide.hpp).
//   staged_kernel  any strides, ragged extents: tiles go global -> registers -> LDS, transposing
//                  on the way when an operand is contiguous along M/N.  128x128x32 tiles.
#include <algorithm>
#include <type_traits>
#include <utility>

#include "common.hpp"
#include "layout.hpp"
#include "matmul_params.hpp"
#include "mfma.hpp"
#include "ew_machine.hpp"
#include "numeric.hpp"

// Workspace of a split K for callers that cannot bring one (kapy_matmul_static_workspace): arrival counters, then
// partial sums.  Part of the device image, so every GPU the library runs on holds its own copy until the process ends;
// zero when the image is loaded, and every kernel that uses the counters leaves them zero.  (A launch the runtime refuses has
// not run and leaves them as they were; a kernel that dies on the way takes the process's context with it, array included: there
// is no state in between for the host to repair.)
static __device__ __align__(256) unsigned char scratch[kapy::kSplitCounterBytes + (16 << 20)];

#include "matmul_tile.hpp"
#include "wide_rule.hpp"

namespace kapy {
namespace {

// ---------------------------------------------------------------------------------------------
// Staged kernel: 128x128x32 tile, 4 wavefronts (2x2), wave tile 64x64.  Any operand strides, ragged
// extents (out-of-range elements read as zero: the padding-ZERO ld_global of the reference).
constexpr int kNBM = 128, kNBN = 128;  // nn_kernel's tile
constexpr int kSBM = 128, kSBN = 128, kSBK = 32;

// One operand tile [128 rows][32 k] is 512 16-byte vectors: 2 per thread.  In "k contiguous" mode a
// vector is 8 consecutive k of one row; in "row contiguous" mode it is 8 consecutive rows at one k
// and is scattered into the K-contiguous LDS image element by element.
struct StagedRegs {
  u32x4 v[2];
};

__device__ __forceinline__ u32x4 load_vec8(const char *base, int64_t s_row, int64_t s_k, int32_t row, int32_t k, int32_t rows,
                                           int32_t K, bool k_contig) {
  u32x4 r = {0, 0, 0, 0};
  const uint16_t *e = (const uint16_t *)base;
  if (k_contig) {
    if (row >= rows || k >= K) return r;
    const uint16_t *ptr = e + row * s_row + k;
    if (k + 8 <= K && (((uintptr_t)ptr) & 15) == 0) return *(const u32x4 *)ptr;
    uint16_t t[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) t[i] = (k + i < K) ? ptr[i] : (uint16_t)0;
#pragma unroll
    for (int w = 0; w < 4; ++w) r[w] = t[2 * w] | ((uint32_t)t[2 * w + 1] << 16);
    return r;
  }
  if (row >= rows || k >= K) return r;
  const uint16_t *ptr = e + row + k * s_k;  // s_row == 1
  if (row + 8 <= rows && (((uintptr_t)ptr) & 15) == 0) return *(const u32x4 *)ptr;
  uint16_t t[8];
#pragma unroll
  for (int i = 0; i < 8; ++i) t[i] = (row + i < rows) ? ptr[i] : (uint16_t)0;
#pragma unroll
  for (int w = 0; w < 4; ++w) r[w] = t[2 * w] | ((uint32_t)t[2 * w + 1] << 16);
  return r;
}

// Fully strided operand (no contiguous axis): element-wise gather of 8 consecutive k of one row.
__device__ __forceinline__ u32x4 gather_vec8(const char *base, int64_t s_row, int64_t s_k, int32_t row, int32_t k, int32_t rows,
                                             int32_t K) {
  u32x4 r = {0, 0, 0, 0};
  if (row >= rows) return r;
  const uint16_t *e = (const uint16_t *)base + row * s_row;
  uint16_t t[8];
#pragma unroll
  for (int i = 0; i < 8; ++i) t[i] = (k + i < K) ? e[(k + i) * s_k] : (uint16_t)0;
#pragma unroll
  for (int w = 0; w < 4; ++w) r[w] = t[2 * w] | ((uint32_t)t[2 * w + 1] << 16);
  return r;
}

enum OperandMode { kKContig = 0, kRowContig = 1, kStrided = 2 };

template <typename T, bool PACKED>
__global__ __launch_bounds__(256) void staged_kernel(GemmParams p, int a_mode, int b_mode) {
  using L = TileLayout<kSBK * 2, T>;
  __shared__ __attribute__((aligned(1024))) char lds[(kSBM + kSBN) * kSBK * 2];
  char *sa = lds, *sb = lds + kSBM * kSBK * 2;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int wm = wave & 1, wn = wave >> 1;
  int32_t tm, tn;
  tile_of_block(p, tm, tn);
  const int32_t m0 = tm * kSBM, n0 = tn * kSBN;

  auto fetch = [&](const char *base, int64_t s_row, int64_t s_k, int32_t row0, int32_t rows, int mode, int kt, StagedRegs &r) {
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      int v = tid + h * 256;
      if (mode == kRowContig) {
        int k = v >> 4, rchunk = v & 15;  // 16 chunks of 8 rows at each of 32 k
        r.v[h] = load_vec8(base, s_row, s_k, row0 + rchunk * 8, kt * kSBK + k, rows, p.K, false);
      } else {
        int row = v >> 2, kchunk = v & 3;  // 4 chunks of 8 k in each of 128 rows
        r.v[h] = mode == kKContig ? load_vec8(base, s_row, s_k, row0 + row, kt * kSBK + kchunk * 8, rows, p.K, true)
                                  : gather_vec8(base, s_row, s_k, row0 + row, kt * kSBK + kchunk * 8, rows, p.K);
      }
    }
  };
  auto stash = [&](char *tile, int mode, const StagedRegs &r) {
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      int v = tid + h * 256;
      if (mode == kRowContig) {
        int k = v >> 4, rchunk = v & 15;
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          uint16_t x = (uint16_t)(r.v[h][e >> 1] >> ((e & 1) * 16));
          *(uint16_t *)(tile + L::offset(rchunk * 8 + e, k >> 3) + (k & 7) * 2) = x;
        }
      } else {
        int row = v >> 2, kchunk = v & 3;
        *(u32x4 *)(tile + L::offset(row, kchunk)) = r.v[h];
      }
    }
  };

  f32x16 acc[2][2];
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int v = 0; v < 16; ++v) acc[i][j][v] = 0.f;

  const int KT = (p.K + kSBK - 1) / kSBK;
  StagedRegs ra, rb;
  fetch(p.a, p.a_sm, p.a_sk, m0, p.M, a_mode, 0, ra);
  fetch(p.b, p.b_sn, p.b_sk, n0, p.N, b_mode, 0, rb);
  const OperandLane frag_at = operand_lane(T::kShape, lane);
  const uint32_t frag_row = frag_at.row, frag_half = frag_at.k0 / T::kShape.kpack;  // the lane's row of a block; which half of a slice's 16 K
  for (int kt = 0; kt < KT; ++kt) {
    __syncthreads();  // every wave has finished reading the previous tile
    stash(sa, a_mode, ra);
    stash(sb, b_mode, rb);
    __syncthreads();
    if (kt + 1 < KT) {  // next tile's global loads fly while this one is multiplied
      fetch(p.a, p.a_sm, p.a_sk, m0, p.M, a_mode, kt + 1, ra);
      fetch(p.b, p.b_sn, p.b_sk, n0, p.N, b_mode, kt + 1, rb);
    }
#pragma unroll
    for (int kk = 0; kk < kSBK / 16; ++kk) {
      u32x4 af[2], bf[2];
#pragma unroll
      for (int i = 0; i < 2; ++i) af[i] = *(const u32x4 *)(sa + L::offset(wm * 64 + i * 32 + frag_row, 2 * kk + frag_half));
#pragma unroll
      for (int j = 0; j < 2; ++j) bf[j] = *(const u32x4 *)(sb + L::offset(wn * 64 + j * 32 + frag_row, 2 * kk + frag_half));
#pragma unroll
      for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j) acc[i][j] = T::mfma(&bf[j], &af[i], acc[i][j]);
    }
  }
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      const int32_t mb = m0 + wm * 64 + i * 32, nb = n0 + wn * 64 + j * 32;
      if (PACKED && mb + 32 <= p.M && nb + 32 <= p.N) store_block_packed(p, mb, nb, lane, acc[i][j]);
      else store_block_generic(p, mb, nb, lane, acc[i][j]);
    }
}

// ---------------------------------------------------------------------------------------------
// Host side.
template <typename T>
int launch_staged(GemmParams p, int a_mode, int b_mode, hipStream_t s) {
  p.tiles_m = (p.M + kSBM - 1) / kSBM;
  p.tiles_n = (p.N + kSBN - 1) / kSBN;
  p.split_k = 1;
  dim3 grid((unsigned)(p.tiles_m * p.tiles_n));
  if (packed_epilogue(p) && p.d_dtype != KAPY_F32 && p.acc_dtype < 0) staged_kernel<T, true><<<grid, dim3(256), 0, s>>>(p, a_mode, b_mode);  // (its packed stores are 16-bit, without accumulator input)
  else staged_kernel<T, false><<<grid, dim3(256), 0, s>>>(p, a_mode, b_mode);
  KAPY_HIP_CHECK(hipGetLastError());
  return KAPY_OK;
}

// The shape and element-type rules of Kapy.cpp:451-487, with the reference's wording.  Not taken over: the minimum
// extents of :491-564 (acc at least 16x8, lhs / rhs at least 16x8, 16x16 or 8x8 per MMA way) - they bound a warp's
// register tile, and this entry point takes whole views of any extent (a decode-shaped M = 1 included) - and the rule
// that the RESULT is f16 or f32: it is applied to the accumulator operand only, because `result` here is the view the
// kernel's final fptofp stores into (f16, bf16 or f32).
int verify_matmul(const kapy_global *lhs, const kapy_global *rhs, const kapy_global *acc, const kapy_global *res, int impl_way) {
  int rc = check_global(lhs, "matmul lhs");
  if (!rc) rc = check_global(rhs, "matmul rhs");
  if (!rc) rc = check_global(res, "matmul result");
  if (!rc && acc) rc = check_global(acc, "matmul acc");
  if (rc) return rc;
  if (extent1(lhs) != extent0(rhs))
    return fail(KAPY_ERR_VERIFY, "matmul: number of columns of lhs must be equal to number of rows of rhs");
  if (extent0(res) != extent0(lhs) || (acc && extent0(acc) != extent0(lhs)))
    return fail(KAPY_ERR_VERIFY, "matmul: number of rows of acc must be equal to number of rows of lhs");
  if (extent1(res) != extent1(rhs) || (acc && extent1(acc) != extent1(rhs)))
    return fail(KAPY_ERR_VERIFY, "matmul: number of columns of acc must be equal to number of columns of rhs");
  if (dtype_bytes(lhs->dtype) != dtype_bytes(rhs->dtype))
    return fail(KAPY_ERR_VERIFY, "matmul: lhs and rhs must have same element bit width");
  if (acc && acc->dtype != KAPY_F16 && acc->dtype != KAPY_F32)
    return fail(KAPY_ERR_VERIFY, "matmul: result must have f16 or f32 element type");
  if (acc && lhs->dtype == KAPY_BF16 && rhs->dtype == KAPY_BF16 && acc->dtype == KAPY_F16)
    return fail(KAPY_ERR_VERIFY, "matmul: result must have f32 element type when operands are bf16 element type");
  if (!is_f8(lhs->dtype) && lhs->dtype != rhs->dtype)
    return fail(KAPY_ERR_VERIFY, "matmul: lhs and rhs must have same element type unless they have f8 element type");
  bool f16ish = lhs->dtype == KAPY_F16 || lhs->dtype == KAPY_BF16;
  switch (impl_way) {
  case KAPY_MATMUL_AUTO: break;
  case KAPY_MMA_M16N8K8_F16: case KAPY_MMA_M16N8K16_F16: case KAPY_MFMA_32X32X16_16B: case KAPY_MFMA_16X16X32_16B:
    if (!f16ish) return fail(KAPY_ERR_VERIFY, "matmul: mma f16 operands must have f16 or bf16 element type");
    break;
  case KAPY_MMA_M16N8K8_TF32:
    if (lhs->dtype != KAPY_F32) return fail(KAPY_ERR_VERIFY, "matmul: mma_m16n8k8_tf32 operands must have f32 element type");
    return fail(KAPY_ERR_UNSUPPORTED, "matmul: mma_m16n8k8_tf32 has no counterpart on gfx950 (no tf32 matrix instruction)");
  case KAPY_MMA_M16N8K16_F8: case KAPY_MFMA_16X16X128_F8: case KAPY_MFMA_32X32X64_F8:
    if (!is_f8(lhs->dtype) || !is_f8(rhs->dtype))
      return fail(KAPY_ERR_VERIFY, "matmul: mma f8 operands must have f8E4M3 or f8E5M2 element type");
    break;
  default: return fail(KAPY_ERR_INVALID, "matmul: unknown implement way %d", impl_way);
  }
  for (const kapy_global *g : {lhs, rhs, res, acc})
    if (g && (g->start0 < 0 || g->start1 < 0)) return fail(KAPY_ERR_INVALID, "matmul: negative view start");
  return KAPY_OK;
}

// Compiled configurations of the TN kernel, in order of preference.
struct TnVariant {
  int bm, bn, bk, waves, stages, mfma;  // mfma: rows of the matrix instruction's operand block (16 or 32)
};
const TnVariant kTnVariants[kTnConfigCount] = {
#define KAPY_TN_CONFIG(BM, BN, BK, WM, WN, S, MFMA) {BM, BN, BK, (WM) * (WN), S, MFMA},
    KAPY_TN_CONFIGS
#undef KAPY_TN_CONFIG
};
// Launches the configuration with this tile, instruction and ring depth (one of the table's).
int launch_tn(const GemmParams &p, bool bf16, int bm, int bn, int bk, int stages, int mfma, hipStream_t s) {
  for (int k = 0; k < kTnConfigCount; ++k) {
    const TnVariant &v = kTnVariants[k];
    if (v.bm == bm && v.bn == bn && v.bk == bk && v.stages == stages && v.mfma == mfma) return bf16 ? launch_tn_bf16(k, p, s) : launch_tn_f16(k, p, s);
  }
  return fail(KAPY_ERR_INVALID, "matmul: no such tile configuration");
}

int operand_mode(int64_t s_row, int64_t s_k) { return s_k == 1 ? kKContig : (s_row == 1 ? kRowContig : kStrided); }

int64_t split_workspace_bytes(int64_t tiles, int split) { return kSplitCounterBytes + tiles * split * (128 * 128 * 4); }

// Whether K falls into `sp` parts of whole K-tiles whose partial sums fit the workspace.
bool split_fits(const GemmParams &p, const kapy_matmul_cfg &c, int tile_k, int sp) {
  const int64_t tiles = (int64_t)((p.M + 127) / 128) * ((p.N + 127) / 128);
  return p.K % (tile_k * sp) == 0 && tiles <= kSplitCounterBytes / 4 && split_workspace_bytes(tiles, sp) <= c.workspace_bytes && ((uintptr_t)c.workspace & 15) == 0;
}
bool split_is_valid(int split) { return split >= 0 && split <= kMaxSplitK && !(split & (split - 1)); }

// Whether plan_split_k honours cfg.split_k.
bool split_is_honoured(const GemmParams &p, const kapy_matmul_cfg &c, int tile_k) {
  return c.split_k == 0 || c.split_k == 1 || (split_is_valid(c.split_k) && c.workspace && split_fits(p, c, tile_k, c.split_k));
}

}  // namespace

// Decides whether the 128 x 128 tiled kernels split K for this problem and points the parameters at the workspace.
// cfg.split_k = 1 or no workspace: never.  0: when the tiles alone would leave at least half the device idle, the
// largest power of two that keeps tiles * split within the CUs, leaves every part at least sixteen K-tiles and fits the
// workspace.  An explicit split that cannot be honoured is an error.
int plan_split_k(GemmParams &p, const kapy_matmul_cfg &c, int tile_k) {
  p.split_k = 1;
  p.partial = nullptr;
  p.counters = nullptr;
  if (!split_is_valid(c.split_k))
    return fail(KAPY_ERR_INVALID, "matmul: split_k must be 0 (library's choice) or a power of two up to %d, not %d", kMaxSplitK, c.split_k);
  if (c.split_k == 1) return KAPY_OK;
  if (!c.workspace) {
    if (c.split_k > 1) return fail(KAPY_ERR_INVALID, "matmul: split_k = %d needs a workspace (kapy_matmul_workspace_bytes)", c.split_k);
    return KAPY_OK;
  }
  const int64_t tiles = (int64_t)((p.M + 127) / 128) * ((p.N + 127) / 128);
  int split = 1;
  if (c.split_k > 1) {
    if (!split_fits(p, c, tile_k, c.split_k))
      return fail(KAPY_ERR_UNSUPPORTED, "matmul: cannot split K = %d into %d parts of whole %d-wide K-tiles with a 16-byte aligned workspace of %lld bytes (%lld needed)",
                  p.K, c.split_k, tile_k, (long long)c.workspace_bytes, (long long)split_workspace_bytes(tiles, c.split_k));
    split = c.split_k;
  } else if (tiles * 2 <= device_cus()) {
    // (meeting in the workspace costs about 10 us: parts shorter than 16 K-tiles do not earn it back)
    for (int sp = 2; sp <= kMaxSplitK && tiles * sp <= device_cus(); sp *= 2)
      if (split_fits(p, c, tile_k, sp) && p.K / (tile_k * sp) >= 16) split = sp;
  }
  if (split > 1) {
    p.split_k = split;
    p.counters = (uint32_t *)c.workspace;
    p.partial = (float *)((char *)c.workspace + kSplitCounterBytes);
  }
  return KAPY_OK;
}

// What the 256-row tiles take (the caller has made sure that each operand has 16-byte aligned lines along its contiguous axis): the
// strip epilogue's results, whole 16-byte pieces, offsets that fit the loader's 32 bits, and a K that ends on a tile or can be
// masked - by pieces of 8 in a K-contiguous operand, by k-rows in a transposed one (two K-contiguous operands: whole tiles only).
bool wide_serves(const GemmParams &p, int bn, bool a_tr, bool b_tr) {
  const int64_t limit = int64_t(1) << 31;
  if (p.M <= 0 || p.N <= 0 || p.K < 128 || p.N % 8 || p.rz || !packed_epilogue(p) || (a_tr && host_has_tail(p))) return false;
  if (p.K % 64 && !b_tr) return false;
  if (p.K % 8 && !a_tr) return false;
  const bool a_fits = a_tr ? p.M % 8 == 0 && p.a_sk > 0 && ((int64_t)p.K + 64) * p.a_sk * 2 < limit : p.a_sm > 0 && p.a_sm * 2 * 256 + (int64_t)p.K * 2 < limit;
  const bool b_fits = b_tr ? p.b_sk > 0 && ((int64_t)p.K + 64) * p.b_sk * 2 < limit : p.b_sn > 0 && p.b_sn * 2 * bn + (int64_t)p.K * 2 < limit;
  return a_fits && b_fits && ((int64_t)(p.M + 255) / 256) * ((p.N + bn - 1) / bn) < limit;
}

// Implemented in matmul_f8.hip.
int matmul_f8(const kapy_global *a, const kapy_global *b, const float *row_scale, const float *col_scale, const kapy_global *acc,
              const kapy_global *result, const kapy_matmul_cfg *cfg, hipStream_t s);

namespace {
// kapy.matmul with, optionally, the elementwise ops that follow it on the accumulator fused into the kernel's epilogue.
int matmul_16bit(const kapy_global *lhs, const kapy_global *rhs, const kapy_global *acc, const kapy_global *result,
                 const kapy_matmul_cfg *cfg, const kapy_matmul_epilogue *epi, void *stream) {
  kapy_matmul_cfg c = {KAPY_MATMUL_AUTO, 0, 0, 0, KAPY_RN, 0, 0, 0, nullptr, 0};
  if (cfg) c = *cfg;
  int rc = verify_matmul(lhs, rhs, acc, result, c.impl_way);
  if (rc) return rc;
  if (c.rmode != KAPY_RN && c.rmode != KAPY_RZ) return fail(KAPY_ERR_INVALID, "matmul: unknown rounding mode %d", c.rmode);
  if (result->dtype != KAPY_F16 && result->dtype != KAPY_BF16 && result->dtype != KAPY_F32)
    return fail(KAPY_ERR_VERIFY, "matmul: result must have f16, bf16 or f32 element type");
  if (c.accumulate != KAPY_ACCUMULATE_F32 && c.accumulate != KAPY_ACCUMULATE_ELEMENT) return fail(KAPY_ERR_INVALID, "matmul: unknown accumulate mode %d", c.accumulate);
  rc = ensure_device();
  if (rc) return rc;
  hipStream_t s = (hipStream_t)stream;
  if (c.accumulate == KAPY_ACCUMULATE_ELEMENT) {
    if (epi) return fail(KAPY_ERR_UNSUPPORTED, "matmul_fused: the fused tail exists with fp32 accumulators only");
    if (c.rmode != KAPY_RN) return fail(KAPY_ERR_UNSUPPORTED, "matmul: f16 accumulators round to nearest even, as the instruction they restate");
    return run_matmul_f16acc(lhs, rhs, acc, result, c.impl_way == KAPY_MMA_M16N8K8_F16 ? 8 : 16, s);
  }
  if (is_f8(lhs->dtype)) {
    if (epi) return fail(KAPY_ERR_UNSUPPORTED, "matmul_fused: fp8 operands take kapy_matmul_scaled_f8");
    return matmul_f8(lhs, rhs, nullptr, nullptr, acc, result, &c, s);
  }
  if (lhs->dtype != KAPY_F16 && lhs->dtype != KAPY_BF16)
    return fail(KAPY_ERR_UNSUPPORTED, "matmul: %s operands have no matrix instruction on gfx950", dtype_name(lhs->dtype));

  // A column-major result: D^T = B^T . A^T is the same problem with a row-major result, which the strip epilogues store (a
  // column-major one goes element by element).  Every dot product sums the same products in the same order, so the bits are
  // those of the problem as given.  (A bias row would turn into a bias column, which no epilogue adds: such calls stay.)
  if (result->stride0 == 1 && result->stride1 != 1 && extent0(result) > 1 && !(epi && epi->bias)) {
    auto turned = [](const kapy_global &g) {
      kapy_global t = g;
      std::swap(t.start0, t.start1);
      std::swap(t.end0, t.end1);
      std::swap(t.stride0, t.stride1);
      return t;
    };
    const kapy_global at = turned(*lhs), bt = turned(*rhs), dt = turned(*result);
    kapy_global acct;
    if (acc) acct = turned(*acc);
    kapy_matmul_cfg inner = c;
    std::swap(inner.tile_m, inner.tile_n);
    return matmul_16bit(&bt, &at, acc ? &acct : nullptr, &dt, &inner, epi, stream);
  }

  GemmParams p;
  p.a = view_base(lhs);
  p.b = view_base(rhs);
  p.acc = acc ? view_base(acc) : nullptr;
  p.d = (char *)view_base(result);
  p.row_scale = p.col_scale = nullptr;
  p.bias = epi && epi->bias ? view_base(epi->bias) : nullptr;
  p.bias_dtype = epi && epi->bias ? epi->bias->dtype : KAPY_F32;
  p.alpha = epi ? epi->alpha : 1.0f;
  p.act = epi ? epi->act : -1;
  p.act_operand = epi ? epi->act_operand : 0.f;
  p.a_sm = lhs->stride0; p.a_sk = lhs->stride1;
  p.b_sk = rhs->stride0; p.b_sn = rhs->stride1;
  p.acc_sm = acc ? acc->stride0 : 0; p.acc_sn = acc ? acc->stride1 : 0;
  p.d_sm = result->stride0; p.d_sn = result->stride1;
  p.M = (int32_t)extent0(lhs); p.K = (int32_t)extent1(lhs); p.N = (int32_t)extent1(rhs);
  p.acc_dtype = acc ? acc->dtype : -1;
  p.d_dtype = result->dtype;
  p.rz = c.rmode == KAPY_RZ;
  p.tiles_m = p.tiles_n = 0;
  p.split_k = 1;
  p.partial = nullptr;
  p.counters = nullptr;
  // The 256-row tiles.  An operand that is contiguous along its other extent is read in place with transposing LDS reads.
  const bool row_lhs = lhs->stride1 == 1 && vector_bytes(lhs, 1) == 16, column_lhs = !row_lhs && lhs->stride0 == 1 && vector_bytes(lhs, 0) == 16;
  const bool row_rhs = rhs->stride1 == 1 && vector_bytes(rhs, 1) == 16, column_rhs = !row_rhs && rhs->stride0 == 1 && vector_bytes(rhs, 0) == 16;
  const bool wide_form = (row_lhs && (row_rhs || column_rhs)) || (column_lhs && row_rhs);
  const bool wide_free = !c.tile_m && !c.tile_n && !c.tile_k && !c.stages && !c.waves && c.split_k <= 1 && c.impl_way != KAPY_MFMA_32X32X16_16B && !(column_rhs && c.impl_way >= KAPY_MFMA_32X32X16_16B);
  const bool wide_asked = c.tile_m == 256 && c.tile_n == 128 && (!c.tile_k || c.tile_k == 64) && !c.stages && (!c.waves || c.waves == 4) && c.split_k <= 1 && c.impl_way != KAPY_MFMA_32X32X16_16B;
  // (a split that is no split at all is left to the kernels below, which refuse it; two row-major operands on 256 x 256 tiles never
  // looked at it)
  const bool split_said = c.split_k >= 0;
  int wide_bn = 0;
  if (wide_form && (wide_free || wide_asked)) {
    if (split_said && (wide_asked || wide128_wins(p.M, p.N, p.K, row_rhs ? 0 : 512, device_cus())) && wide_serves(p, 128, column_lhs, row_rhs)) wide_bn = 128;
    // (KAPY_NN256=0 in the environment: never the 256 x 256 form; KAPY_NN256_FROM: the least number of its tiles per 100 CUs, for
    // measurements)
    static const bool wide256 = !(getenv("KAPY_NN256") && getenv("KAPY_NN256")[0] == '0');
    static const int wide256_from_pct = getenv("KAPY_NN256_FROM") ? atoi(getenv("KAPY_NN256_FROM")) : 55;
    if (!wide_bn && wide_free && (split_said || row_lhs) && wide256 && row_rhs && wide_serves(p, 256, column_lhs, row_rhs) &&
        (int64_t)((p.M + 255) / 256) * ((p.N + 255) / 256) * 100 >= (int64_t)device_cus() * wide256_from_pct)
      wide_bn = 256;
  }

  // A large problem with an operand that is contiguous along its OTHER extent (a row-major rhs, a column-major lhs).  The kernel
  // that reads such operands with transposing LDS reads works on 128 x 128 tiles and reaches 1.05-1.12 PFLOP/s where the
  // K-contiguous kernel's 256 x 256 tiles reach 1.35-1.55.  Turning the operand first costs one pass of the transposing copy
  // over it (its bytes read and written once, at 0.68 of the HBM rate) and pays from about six thousand rows on - if the caller's
  // workspace has room for the turned operand(s) behind the 16 KiB of split-K counters, which stay untouched.
  if (c.workspace && !c.tile_m && !c.tile_n && !c.tile_k && !c.stages && !c.waves && c.split_k <= 1 && c.impl_way < KAPY_MFMA_32X32X16_16B) {
    const int64_t M = extent0(lhs), K = extent1(lhs), N = extent1(rhs);
    const bool a_turn = lhs->stride0 == 1 && lhs->stride1 != 1, b_turn = rhs->stride1 == 1 && rhs->stride0 != 1;
    const bool a_kc = lhs->stride1 == 1, b_kc = rhs->stride0 == 1;
    const int64_t a_bytes = a_turn ? ((M * K * 2 + 255) & ~int64_t(255)) : 0, b_bytes = b_turn ? ((K * N * 2 + 255) & ~int64_t(255)) : 0;
    // (measured, bf16, in place -> turned: 8192^3 1237 -> 1485 TFLOP/s, 8192 x 2048 x 4096 1130 -> 1317, 8192 x 8192 x 1024 924 -> 1106;
    // 4096^3 and 2048 x 8192 x 4096 the same either way; 2048^2 x K slower by a third: the turn is paid once per operand and
    // earned back over the rows - or, for a turned lhs, the columns - that use it)
    // (what the 256-row tiles read in place is not turned: 8192^3 bf16, row-major rhs 0.683 ms against 0.727 for turn and product, both
    // operands transposed 0.72 against 0.83)
    if (!wide_bn && (a_turn || b_turn) && (a_turn || a_kc) && (b_turn || b_kc) && (!b_turn || M >= 6144) && (!a_turn || N >= 6144) && M >= 2048 && N >= 2048 && K >= 1024 &&
        M % 8 == 0 && N % 8 == 0 && K % 8 == 0 &&
        M * K < (int64_t(1) << 31) && K * N < (int64_t(1) << 31) && kSplitCounterBytes + a_bytes + b_bytes <= c.workspace_bytes &&
        ((uintptr_t)c.workspace & 255) == 0) {
      char *at = (char *)c.workspace + kSplitCounterBytes;
      kapy_global a2 = *lhs, b2 = *rhs;
      const kapy_copy_cfg turn = {1, KAPY_PAD_ZERO, 0, 0, 0, 0};
      auto dense = [](void *ptr, int64_t rows, int64_t cols, int32_t dtype) {
        kapy_global g;
        g.ptr = ptr;
        g.start0 = g.start1 = 0;
        g.end0 = (int32_t)rows;
        g.end1 = (int32_t)cols;
        g.stride0 = (int32_t)cols;
        g.stride1 = 1;
        g.dtype = dtype;
        g.alignment = 16;
        return g;
      };
      if (b_turn) {  // rhs [K x N] row-major -> [N x K] row-major in the workspace, read back as a [K x N] view with K contiguous
        const kapy_global turned = dense(at, N, K, rhs->dtype);
        rc = copy_impl(rhs, &turned, &turn, nullptr, stream);
        if (rc) return rc;
        b2 = turned;
        b2.end0 = (int32_t)K; b2.end1 = (int32_t)N;
        b2.stride0 = 1; b2.stride1 = (int32_t)K;
        at += b_bytes;
      }
      if (a_turn) {  // lhs [M x K] column-major -> row-major
        const kapy_global turned = dense(at, M, K, lhs->dtype);
        kapy_global as_rows = *lhs;  // the same memory seen as the row-major [K x M] it is, which the copy transposes
        std::swap(as_rows.start0, as_rows.start1);
        std::swap(as_rows.end0, as_rows.end1);
        std::swap(as_rows.stride0, as_rows.stride1);
        rc = copy_impl(&as_rows, &turned, &turn, nullptr, stream);
        if (rc) return rc;
        a2 = turned;
      }
      kapy_matmul_cfg inner = c;
      inner.workspace = nullptr;
      inner.workspace_bytes = 0;
      return matmul_16bit(&a2, &b2, acc, result, &inner, epi, stream);
    }
  }

  if (p.M == 0 || p.N == 0) return KAPY_OK;
  const bool bf16 = lhs->dtype == KAPY_BF16;
  if (wide_bn == 128) return bf16 ? launch_wide128_bf16(p, column_lhs, row_rhs, s) : launch_wide128_f16(p, column_lhs, row_rhs, s);
  if (wide_bn == 256) return bf16 ? launch_wide256_bf16(p, column_lhs, row_rhs, s) : launch_wide256_f16(p, column_lhs, row_rhs, s);

  // Roofline path: both operands K-contiguous, 16-byte aligned rows, extents multiples of the tile,
  // and offsets that fit the 32-bit per-lane address arithmetic of the loader.
  bool tn = p.a_sk == 1 && p.b_sk == 1 && vector_bytes(lhs, 1) == 16 && vector_bytes(rhs, 0) == 16 && p.K > 0 &&
            p.a_sm * 2 * 256 + (int64_t)p.K * 2 < (int64_t(1) << 31) && p.b_sn * 2 * 256 + (int64_t)p.K * 2 < (int64_t(1) << 31) && p.a_sm >= 0 && p.b_sn >= 0;
  if (tn) {
    const bool free_choice = !c.tile_m && !c.tile_n && !c.tile_k && !c.stages && !c.waves && c.impl_way < KAPY_MFMA_32X32X16_16B;
    for (const TnVariant &v : kTnVariants) {
      if ((c.tile_m && c.tile_m != v.bm) || (c.tile_n && c.tile_n != v.bn) || (c.tile_k && c.tile_k != v.bk) ||
          (c.stages && c.stages != v.stages) || (c.waves && c.waves != v.waves) ||
          (c.impl_way == KAPY_MFMA_32X32X16_16B && v.mfma != 32) || (c.impl_way == KAPY_MFMA_16X16X32_16B && v.mfma != 16))
        continue;
      // the ring variants' bounded loads let a tile hang over the last rows of either operand; the others need whole tiles
      const bool whole_tiles = p.M % v.bm == 0 && p.N % v.bn == 0;
      const bool whole_k = p.K % v.bk == 0;  // the ring variants also take a partial last K-tile of whole 16-byte chunks
      if ((!whole_k && (v.stages != kRing25 || p.K % 8)) || (!whole_tiles && v.stages != kRing25)) continue;
      // with a free choice, a 256x256 tiling of too few tiles yields to 128x128
      if (free_choice && v.bm == 256 && !enough_256_tiles(p.M, p.N, device_cus())) continue;
      // an explicit split of K is a request for a variant that can split: with a free tile choice the others are passed over
      // (plan_split_k then honours the split or says why it cannot)
      if (c.split_k > 1 && !c.tile_m && !(v.bm == 128 && v.stages == kRing25)) continue;
      if (v.bm == 128 && v.stages == kRing25) {
        rc = plan_split_k(p, c, v.bk);
        if (rc) return rc;
        // A result with N no multiple of 8: the ring's builds store it element by element, nn_kernel's in strips (f16, K-contiguous
        // operands: 1000 x 4097 x 4096 98 -> 54 us, 1500 x 2047 x 2048 59 -> 18, 64 x 300 x 256 40 -> 6).
        if (free_choice && !host_has_tail(p) && p.N % 8 && packed_epilogue(p)) return launch_nn_config(p, bf16, 3, 64, 4, true, s);
        // Tiles for at most half the CUs and K not split: a workgroup alone on its CU waits for the ring's 2.5 tiles of loads.
        // The four-stage build on the 32-row instruction keeps three tiles in flight: bf16 N = K = 8192, 128 / 256 rows
        // 54 / 55 -> 48 / 52 us (level at 384 rows, behind from 512; the same depth on the 16-row instruction: 71 us).
        // Fewer still: smaller tiles put every CU to work on the operand streams.  bf16 N = K = 8192, 64 / 128 rows on
        // 64 x 64 x 128 tiles 48 / 47 -> 30 / 30 us, 256 rows on 128 x 64 x 64 tiles 47.5 -> 43; from 384 rows on (more small
        // tiles than CUs) they lose to the 128 x 128 ring.
        if (free_choice && p.split_k <= 1 && !host_has_tail(p) && p.N % 8 == 0) {
          const int64_t n64 = (p.N + 63) / 64;
          if (p.K % 128 == 0 && (int64_t)((p.M + 63) / 64) * n64 <= device_cus())
            return launch_tn(p, bf16, 64, 64, 128, 4, 32, s);
          if (p.K % 64 == 0 && (int64_t)((p.M + 127) / 128) * n64 <= device_cus())
            return launch_tn(p, bf16, 128, 64, 64, 4, 32, s);
        }
        if (free_choice && p.split_k <= 1 && !host_has_tail(p) && p.K % 64 == 0 && p.N % 8 == 0 &&
            (int64_t)((p.M + 127) / 128) * ((p.N + 127) / 128) * 2 <= device_cus())
          return launch_tn(p, bf16, 128, 128, 64, 4, 32, s);
      } else if (c.split_k > 1 && c.tile_m) {
        return fail(KAPY_ERR_UNSUPPORTED, "matmul: only the 128 x 128 tiles split K");
      }
      return launch_tn(p, bf16, v.bm, v.bn, v.bk, v.stages, v.mfma, s);
    }
  }
  // An operand that is contiguous along its other extent - a row-major rhs (with a row-major lhs: the reference fixture's
  // layout, matmul.mlir), a column-major lhs - is staged as it lies and read with the transposing read.
  const bool a_kc = p.a_sk == 1 && vector_bytes(lhs, 1) == 16 && p.a_sm >= 0 && p.a_sm * 2 * kNBM + (int64_t)p.K * 2 < (int64_t(1) << 31);
  const bool a_tr = !a_kc && p.a_sm == 1 && vector_bytes(lhs, 0) == 16 && p.a_sk >= 0 && p.M % 8 == 0 && (int64_t)p.K * p.a_sk * 2 < (int64_t(1) << 31);
  const bool b_tr = p.b_sn == 1 && vector_bytes(rhs, 1) == 16 && p.b_sk >= 0 && (int64_t)p.K * p.b_sk * 2 < (int64_t(1) << 31);
  const bool b_kc = !b_tr && p.b_sk == 1 && vector_bytes(rhs, 0) == 16 && p.b_sn >= 0 && p.b_sn * 2 * kNBN + (int64_t)p.K * 2 < (int64_t(1) << 31);
  bool nn = (a_kc || a_tr) && (b_kc || b_tr) && (a_tr || b_tr || p.K % 8) && p.M > 0 && p.K > 0 &&
            c.impl_way != KAPY_MFMA_32X32X16_16B && (!c.tile_m || c.tile_m == kNBM) && (!c.tile_n || c.tile_n == kNBN) && (!c.waves || c.waves == 4);
  if (nn) {
    struct NnVariant {
      int bk, stages;
    };
    static const NnVariant kNn[] = {{64, 4}, {64, 3}, {32, 4}};
    const int form = !a_tr ? (b_tr ? 0 : 3) : (b_tr ? 1 : 2);
    // A split that cannot be honoured is refused, except where lines end inside the tiles' pieces (a row-major result's in N, a
    // column-major lhs's in M): such calls keep going to the general kernel, which does not split.
    const bool any_split = p.N % 8 || (a_tr && p.M % kNBM);
    for (const NnVariant &v : kNn) {
      if ((c.tile_k && c.tile_k != v.bk) || (c.stages && c.stages != v.stages) || p.K % v.bk) continue;
      if (any_split && !split_is_honoured(p, c, v.bk)) break;
      rc = plan_split_k(p, c, v.bk);
      if (rc) return rc;
      return launch_nn_config(p, bf16, form, v.bk, v.stages, false, s);
    }
    // K that no variant's K-tile divides: the builds with a partial last K-tile (never split).  Operands that lie K-row by K-row are
    // masked row by row; of a K-contiguous operand the pieces beyond K are masked and the piece K ends inside is cut.  (us, on the
    // general kernel before: the weight gradient of 1973 tokens, 3072 x 2560 bf16 -> fp32 226 -> 33; f16, row-major operands: 1000 x 4096 x 4095 288 -> 34,
    // 999 x 4097 x 4096 332 -> 60; K-contiguous ones: 1000 x 4096 x 4095 229 -> 33.)
    if (!c.stages && c.split_k <= 1) {
      const int bk = c.tile_k ? c.tile_k : (p.K >= 256 ? 64 : 32);
      if (bk == 64 || bk == 32) {
        p.split_k = 1;
        return launch_nn_config(p, bf16, form, bk, 4, true, s);
      }
    }
  }
  if ((c.tile_m && c.tile_m != kSBM) || (c.tile_n && c.tile_n != kSBN) || (c.tile_k && c.tile_k != kSBK) || (c.stages && c.stages != 1) ||
      (c.waves && c.waves != 4))
    return fail(KAPY_ERR_UNSUPPORTED, "matmul: no kernel with tile %dx%dx%d, %d stages, %d waves serves these operands "
                                      "(the general kernel is 128x128x32, 1 stage, 4 waves)",
                c.tile_m, c.tile_n, c.tile_k, c.stages, c.waves);
  int a_mode = operand_mode(p.a_sm, p.a_sk), b_mode = operand_mode(p.b_sn, p.b_sk);
  return bf16 ? launch_staged<Bf16>(p, a_mode, b_mode, s) : launch_staged<F16>(p, a_mode, b_mode, s);
}


}  // namespace
}  // namespace kapy

using namespace kapy;

extern "C" {

int kapy_matmul(const kapy_global *lhs, const kapy_global *rhs, const kapy_global *acc, const kapy_global *result,
                const kapy_matmul_cfg *cfg, void *stream) {
  return matmul_16bit(lhs, rhs, acc, result, cfg, nullptr, stream);
}

int64_t kapy_matmul_turn_workspace_bytes(const kapy_global *lhs, const kapy_global *rhs) {
  if (!lhs || !rhs) return 0;
  const int64_t M = extent0(lhs), K = extent1(lhs), N = extent1(rhs);
  const bool a_turn = lhs->stride0 == 1 && lhs->stride1 != 1, b_turn = rhs->stride1 == 1 && rhs->stride0 != 1;
  if (!a_turn && !b_turn) return 0;
  return kSplitCounterBytes + (a_turn ? ((M * K * 2 + 255) & ~int64_t(255)) : 0) + (b_turn ? ((K * N * 2 + 255) & ~int64_t(255)) : 0);
}

int64_t kapy_matmul_workspace_bytes(int64_t m, int64_t n) {
  if (m <= 0 || n <= 0) return 0;
  // a split keeps tiles * parts within the CUs of the device; without a device, the largest split of every tile
  const int64_t tiles = ((m + 127) / 128) * ((n + 127) / 128);
  return split_workspace_bytes(tiles, kMaxSplitK);
}

int kapy_matmul_static_workspace(const kapy_global *lhs, const kapy_global *rhs, const kapy_global *acc, const kapy_global *result,
                                 const kapy_matmul_cfg *cfg, void *stream) {
  kapy_matmul_cfg c = {KAPY_MATMUL_AUTO, 0, 0, 0, KAPY_RN, 0, 0, 0, nullptr, 0};
  if (cfg) c = *cfg;
  int rc = ensure_device();
  if (rc) return rc;
  // The array's name is a host-side handle, not a device address: ask the runtime once per device where this device's
  // copy lives, and hand that pointer to the kernels.
  static void *scratch_on_device[kMaxDevices];  // (a race between two first calls only repeats the query)
  int dev = -1;
  KAPY_HIP_CHECK(hipGetDevice(&dev));
  if (dev < 0 || dev >= kMaxDevices) return fail(KAPY_ERR_UNSUPPORTED, "matmul_static_workspace: device ordinal %d beyond %d", dev, kMaxDevices);
  void *ws = __atomic_load_n(&scratch_on_device[dev], __ATOMIC_ACQUIRE);
  if (!ws) {
    KAPY_HIP_CHECK(hipGetSymbolAddress(&ws, HIP_SYMBOL(scratch)));
    if (!ws) return fail(KAPY_ERR_HIP, "matmul_static_workspace: the runtime reports no address for the workspace array");
    __atomic_store_n(&scratch_on_device[dev], ws, __ATOMIC_RELEASE);
  }
  c.workspace = ws;
  c.workspace_bytes = (int64_t)sizeof(scratch);
  return matmul_16bit(lhs, rhs, acc, result, &c, nullptr, stream);
}

int kapy_matmul_fused(const kapy_global *lhs, const kapy_global *rhs, const kapy_global *result, const kapy_matmul_epilogue *epi,
                      const kapy_matmul_cfg *cfg, void *stream) {
  if (!epi) return fail(KAPY_ERR_INVALID, "matmul_fused: null epilogue");
  switch (epi->act) {
  case -1: case KAPY_EW_GELU_TANH: case KAPY_EW_MAXIMUMF: case KAPY_EW_MINIMUMF: case KAPY_EW_NEGF: case KAPY_EW_ABSF:
    break;
  case KAPY_EW_EXP: case KAPY_EW_EXP2: case KAPY_EW_LOG: case KAPY_EW_LOG2: case KAPY_EW_SQRT: case KAPY_EW_RSQRT: case KAPY_EW_TANH: case KAPY_EW_ERF:
    return fail(KAPY_ERR_UNSUPPORTED, "matmul_fused: this activation is not compiled into the matmul kernels; run it as an elementwise program on the result");
  default: return fail(KAPY_ERR_INVALID, "matmul_fused: act must be a unary elementwise op, maximumf / minimumf (against act_operand) or -1, not %d", epi->act);
  }
  if (epi->bias) {
    int rc = check_global(epi->bias, "matmul_fused bias");
    if (rc) return rc;
    if (epi->bias->dtype != KAPY_F16 && epi->bias->dtype != KAPY_BF16 && epi->bias->dtype != KAPY_F32)
      return fail(KAPY_ERR_VERIFY, "matmul_fused: bias must have f16, bf16 or f32 element type");
    if (!rhs || extent0(epi->bias) != 1 || extent1(epi->bias) != extent1(rhs) || epi->bias->stride1 != 1)
      return fail(KAPY_ERR_VERIFY, "broadcast: the bias must be one contiguous row [1 x N]");
  }
  return matmul_16bit(lhs, rhs, nullptr, result, cfg, epi, stream);
}

int kapy_matmul_lds_layout(int32_t operand_dtype, int32_t tile_k, kapy_swizzling *out) {
  if (!out) return fail(KAPY_ERR_INVALID, "matmul_lds_layout: null result");
  if (operand_dtype != KAPY_F16 && operand_dtype != KAPY_BF16)
    return fail(KAPY_ERR_UNSUPPORTED, "matmul_lds_layout: only f16 / bf16 operand tiles are described here");
  Swizzle s;
  switch (tile_k) {
  case 32: s = TileLayout<64, Bf16>::kSwizzle; break;      // (f16 and bf16 share the operand layouts; the 32-deep tiles are built
  case 64: s = TileLayout<128, Bf16M16>::kSwizzle; break;  //  on the 32x32x16 instruction, the 64-deep ones on 16x16x32)
  default: return fail(KAPY_ERR_UNSUPPORTED, "matmul_lds_layout: tile_k must be 32 or 64");
  }
  s.stride0 = tile_k;  // the search runs on bytes; report the row stride in elements
  out->stride0 = s.stride0;
  out->stride1 = s.stride1;
  out->bank_param = s.bank_param;
  out->line_param = s.line_param;
  out->rotate = s.rotate;
  return KAPY_OK;
}

}  // extern "C"

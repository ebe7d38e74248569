// Interpolation on gfx950: 2:4 sparse MFMA (v_smfmac_f32_16x16x32_f16) over the
// reference's packed tiles, a dense-MFMA control, and the plain FP32 CSR path.
//
// Semantics follow the reference's fused complex kernel
// (experiments/production/src/nufft_spmma_bench.cu:377-663): for every 16-row
// group, sum over its K32 tiles of A_re/A_im (16x32, 2:4) times the panel rows
// named by the tile's 32 column ids (16 channels = Re/Im of 8 coils), complex
// combine (conjugate for the adjoint), scale, store or accumulate.
//
// MI355X design (not a translation): one wave64 per work item; the tile is
// re-laid out at upload so each lane fetches its MFMA operands with one 16-byte
// load (A_re|A_im) and one 2-byte load (both sparse index bytes); hi and
// residual panels accumulate into the same FP32 accumulators in one pass; the
// Re/Im combine is one cross-lane swap (lane n <-> n^8); long groups are split
// over several waves and reduced deterministically; block -> item mapping
// keeps Morton-adjacent groups on one XCD (shared L2).
#include <algorithm>
#include <atomic>
#include <cmath>
#include <cstdlib>
#include <initializer_list>
#include <memory>
#include <mutex>
#include <new>
#include <numeric>
#include <system_error>
#include <thread>
#include <type_traits>

#include "tsn_internal.h"

using namespace tsn;

typedef _Float16 half4_t __attribute__((ext_vector_type(4)));
typedef _Float16 half8_t __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x4_t __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef float float4_t __attribute__((ext_vector_type(4)));
typedef float float2_t __attribute__((ext_vector_type(2)));
typedef uint32_t u32x2_t __attribute__((ext_vector_type(2)));

namespace tsn {

// kOutBlockRows (host side only): row-major float2 in blocks of 8 coils, block
// b of rows at b * n_out * 8 (64-byte rows), launched as kOutRowMajor with
// the block stride set.
enum OutMode { kOutCoilMajor = 0, kOutRowMajor = 1, kOutSplit16IL = 3, kOutSplitBF16IL = 4,
               kOutBlockRows = 5 };
// Tile kinds: FP16 tiles x FP16 hi + residual on smfmac, the same on dense
// MFMA, FP16 hi only, and BF16 tiles x BF16 hi + residual on smfmac.
enum TileKind { kSparseSplit = 0, kDenseSplit = 1, kSparseHi = 2, kSparseSplitBF16 = 3 };

struct InterpArgs {
  const WorkItem* items;
  uint32_t n_items;
  const ChunkItem* chunks;  // long-group chunks
  uint32_t n_chunks;
  const uint32_t* order;    // [n_items + n_chunks] launch order (kChunkTag marks chunks)
  float* partials;          // their partial slots [slot][kSlotFloats]
  uint32_t* counters;       // arrival counter per long group
  const int32_t* group_rows;
  const uint32_t* group_offsets;
  const uint32_t* tile_cols;  // column * 32 | last-tile flag (bit 31 of word 2 of each lane segment)
  uint32_t n_tiles, n_groups;
  const uint4* tile_a;
  const uint16_t* tile_idx;
  const uint4* tile_dense;
  const _Float16* panel_hi;
  const _Float16* panel_res;
  const uint32_t* panel_il;  // interleaved hi|res panel (plan-internal layout)
  uint64_t panel_stride;     // elements between coil blocks of the input panel
  uint32_t coils;
  uint32_t n_out;         // output rows (for layouts)
  float scale;
  float* out_f32;         // float2 output (coil- or row-major)
  uint32_t* out_il;       // interleaved split output panel blocks, or line rows
  uint32_t lines;         // one wave per coil block (WB = 2): the interleaved panels hold line rows, not blocks
  // row-major float2 output: (row, coil) at float2 (coil >> 3) * out_bs +
  // row * out_rs + (coil & 7) ([row][coils]: out_rs = coils, out_bs = 8)
  uint32_t out_rs;
  uint64_t out_bs;
  uint32_t coil_base;     // first coil of block 0 in the output (batched launches)
  uint32_t depth;         // tiles in flight ahead of the multiply: 0 = PipeDepth, else 1..3
  // Batched launches (one coil block of one problem per entry; NB = 1,
  // interleaved panels): items[i] belongs to problems[item_problem[i]].
  const struct InterpProblem* problems;
  const uint32_t* item_problem;
  // Data-consistency epilogue of split outputs: each value v becomes
  // (v - dc_scale * y) * w before the split.  y is read at
  // row * dc_row_stride + coil * dc_coil_stride + part (floats); null = off.
  const float* dc_meas;
  const float* dc_density;  // w per output row, or null (all ones)
  float dc_scale;
  uint32_t dc_row_stride, dc_coil_stride;
};

// One coil block of one problem of a batched interpolation launch.
struct InterpProblem {
  const int32_t* group_rows;
  const uint32_t* tile_cols;
  const uint4* tile_a;
  const uint16_t* tile_idx;
  const uint4* tile_dense;
  uint32_t n_tiles, n_groups, n_out, n_cols;
  uint32_t coils;       // coils of the problem (output row layouts)
  uint32_t coil_base;   // first coil of this block
  const uint32_t* panel_il;  // this block's input panel [n_cols][16]
  float* out_f32;       // the problem's float2 output
  uint32_t* out_il;     // this block's split output panel
  uint32_t out_rs;      // row-major output strides (as InterpArgs)
  uint64_t out_bs;
  uint32_t lines;       // both panels hold two coil blocks as 128-byte line rows
};

// Global-space view of a plain pointer.  The kernel's loads and stores after
// the first tile go through it: a generic (flat) access counts on both the
// vector-memory and the LDS wait counters, and while one is outstanding the
// compiler drains every later wait to zero, which stalls the tile pipeline at
// each epilogue.
template <typename T>
__device__ __forceinline__ __attribute__((address_space(1))) T* glb(T* p) {
  return (__attribute__((address_space(1))) T*)(p);
}

__device__ __forceinline__ InterpArgs problem_args(const InterpArgs& a, uint32_t vp) {
  const InterpProblem& q = a.problems[vp];
  InterpArgs v = a;
  v.group_rows = q.group_rows;
  v.tile_cols = q.tile_cols;
  v.tile_a = q.tile_a;
  v.tile_idx = q.tile_idx;
  v.tile_dense = q.tile_dense;
  v.n_tiles = q.n_tiles;
  v.n_groups = q.n_groups;
  v.n_out = q.n_out;
  v.coils = q.coils;
  v.coil_base = q.coil_base;
  v.panel_il = q.panel_il;
  v.panel_stride = static_cast<uint64_t>(q.n_cols) * kN;
  v.lines = q.lines;
  v.out_f32 = q.out_f32;
  v.out_il = q.out_il;
  v.out_rs = q.out_rs;
  v.out_bs = q.out_bs;
  return v;
}

// hi | res << 16 of one value: FP16 (RN) or BF16 (RNE) halves, res = v - hi.
// v is pinned as an FP32 value first: otherwise the compiler may fold the
// multiply that produced it into the FP16 conversion (v_fma_mix, one rounding
// instead of two), and identical inputs would split differently in different
// kernels.
template <bool BF16>
__device__ __forceinline__ uint32_t split_word(float v) {
  asm volatile("" : "+v"(v));
  if constexpr (BF16) {
    const uint16_t hb = bf16_rne_bits(v);
    return static_cast<uint32_t>(hb) | (static_cast<uint32_t>(bf16_rne_bits(v - bf16_to_float(hb))) << 16);
  } else {
    const _Float16 h = static_cast<_Float16>(v);
    const _Float16 r = static_cast<_Float16>(v - static_cast<float>(h));
    return static_cast<uint32_t>(__builtin_bit_cast(uint16_t, h)) |
           (static_cast<uint32_t>(__builtin_bit_cast(uint16_t, r)) << 16);
  }
}

// Data-consistency residual (prediction - scale * y) * w, every step rounded
// on its own (no contraction into fma), so that the fused epilogue and the
// materialized pass over stored predictions produce the same bits.
__device__ __forceinline__ float dc_residual(float pred, float y, float scale, float w) {
#pragma clang fp contract(off)
  const float m = y * scale;
  return (pred - m) * w;
}

__device__ __forceinline__ float dc_apply(const InterpArgs& a, float v, uint32_t coil, int row, int part) {
  asm volatile("" : "+v"(v));  // v is final here, as if loaded from memory
  const float y = coil < a.coils ? glb(a.dc_meas)[static_cast<size_t>(row) * a.dc_row_stride +
                                             static_cast<size_t>(coil) * a.dc_coil_stride + part]
                                 : 0.0f;
  const float w = a.dc_density ? glb(a.dc_density)[row] : 1.0f;
  return dc_residual(v, y, a.dc_scale, w);
}

// Exchanges within the wave's 16-lane rows by DPP.  lane_xor: the value of lane
// n ^ OFF.  swap_lanes: lanes with bit OFF of n clear take the partner's x into
// y, the others the partner's y into x.
constexpr int kRor8 = 0x128, kShl4 = 0x104, kShr4 = 0x114;  // row rotate by 8, lane n reads n + 4, n - 4
template <int OFF>
__device__ __forceinline__ float lane_xor(float v) {
  const int i = __builtin_bit_cast(int, v);
  if constexpr (OFF == 8) return __builtin_bit_cast(float, __builtin_amdgcn_mov_dpp(i, kRor8, 0xF, 0xF, true));
  const int up = __builtin_amdgcn_update_dpp(i, i, kShl4, 0xF, 0x5, false);
  return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(up, i, kShr4, 0xF, 0xA, false));
}
template <int OFF>
__device__ __forceinline__ void swap_lanes(uint32_t& x, uint32_t& y) {
  static_assert(OFF == 4 || OFF == 8, "lane bit 2 or 3");
  const int x0 = static_cast<int>(x), y0 = static_cast<int>(y);
  y = static_cast<uint32_t>(OFF == 8 ? __builtin_amdgcn_update_dpp(y0, x0, kRor8, 0xF, 0x3, false)
                                     : __builtin_amdgcn_update_dpp(y0, x0, kShl4, 0xF, 0x5, false));
  x = static_cast<uint32_t>(OFF == 8 ? __builtin_amdgcn_update_dpp(x0, y0, kRor8, 0xF, 0xC, false)
                                     : __builtin_amdgcn_update_dpp(x0, y0, kShr4, 0xF, 0xA, false));
}
template <int OFF>
__device__ __forceinline__ void swap_lanes(float& x, float& y) {
  uint32_t u = __builtin_bit_cast(uint32_t, x), v = __builtin_bit_cast(uint32_t, y);
  swap_lanes<OFF>(u, v);
  x = __builtin_bit_cast(float, u);
  y = __builtin_bit_cast(float, v);
}

// One float2 output value from the Re and the Im channel's sums.
template <int OM, bool CONJ, bool ACC>
__device__ __forceinline__ void store_value(const InterpArgs& a, int row, uint32_t coil, float rr, float ri, float ir,
                                            float ii) {
  float2_t v = {(CONJ ? rr + ii : rr - ii) * a.scale, (CONJ ? ir - ri : ir + ri) * a.scale};
  if (row < 0 || coil >= a.coils) return;
  size_t o;
  if constexpr (OM == kOutCoilMajor) o = static_cast<size_t>(coil) * a.n_out + row;
  else o = (coil >> 3) * a.out_bs + static_cast<size_t>(row) * a.out_rs + (coil & 7);
  auto* out = glb(reinterpret_cast<float2_t*>(a.out_f32));
  if constexpr (ACC) v += out[o];
  out[o] = v;
}

// One coil block's rows from the wave's accumulators.  Lane n of a quarter
// holds part n >> 3 (Re or Im) of coil n & 7 for four rows, lane n ^ 8 the
// coil's other part.  Split outputs write a word a lane and row.  For float2
// outputs the two lanes exchange accumulators, so that the Re lane holds both
// parts of rows 0 and 1 and the Im lane those of rows 2 and 3: two 8-byte stores
// a lane, where a store per part took four of 4 bytes (adjoint, 512^2 / 8 coils:
// 17.9 -> 17.2 us).
template <int OM, bool CONJ, bool ACC, int WB>
__device__ __forceinline__ void interp_epilogue(const InterpArgs& a, const int4& rows, int b,
                                                const float4_t& acc_re, const float4_t& acc_im,
                                                int lane) {
  const int n = lane & 15;
  const uint32_t coil = a.coil_base + b * kCoilsPerBlock + (n & 7);
  if constexpr (OM == kOutSplitBF16IL || OM == kOutSplit16IL) {
    const int rr[4] = {rows.x, rows.y, rows.z, rows.w};
    const bool im = n & 8;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const float x = lane_xor<8>(acc_im[i]);
      float v = (im == CONJ ? acc_re[i] - x : acc_re[i] + x) * a.scale;
      const int row = rr[i];
      if (row < 0) continue;
      if (a.dc_meas) v = dc_apply(a, v, coil, row, im ? 1 : 0);
      const size_t o = WB > 1 && a.lines ? (static_cast<size_t>(row) * 2 + b) * kN
                                         : (static_cast<size_t>(b) * a.n_out + row) * kN;
      glb(a.out_il)[o + n] = split_word<OM == kOutSplitBF16IL>(v);
    }
  } else {
    // rows.x and rows.y: rows 0 and 1 in the Re lane, 2 and 3 in the Im lane (group_rows_of)
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      float rr = acc_re[i], ir = acc_re[2 + i], ri = acc_im[i], ii = acc_im[2 + i];
      swap_lanes<8>(rr, ir);
      swap_lanes<8>(ri, ii);
      store_value<OM, CONJ, ACC>(a, i ? rows.y : rows.x, coil, rr, ri, ir, ii);
    }
  }
}

// The epilogue of both coil blocks of kLines panels.  Accumulator b of lane n
// of a quarter is word 16 ((n >> 1) & 1) + 8 ((n >> 2) & 1) + 4 (n & 1) +
// 2 (n >> 3) + b of the 32-word row (see fetch_ops): part (n >> 2) & 1 (Re or
// Im) of coil 8 ((n >> 1) & 1) + 4 (n & 1) + 2 (n >> 3) + b, and lane n ^ 4
// holds the coil's other part.  Split outputs write the two words with one
// 8-byte store (128 contiguous bytes a row); float2 outputs exchange
// accumulators so that the Re lane holds both parts of its b = 0 coil and the
// Im lane both parts of its b = 1 coil, one 8-byte store each.
template <int OM, bool CONJ, bool ACC>
__device__ __forceinline__ void interp_epilogue_lines(const InterpArgs& a, const int4& rows,
                                                      const float4_t (&acc_re)[2], const float4_t (&acc_im)[2],
                                                      int lane) {
  const uint32_t n = lane & 15;
  const bool im = n & 4u;
  const uint32_t coil0 = a.coil_base + ((n >> 1) & 1u) * kCoilsPerBlock + 4 * (n & 1) + 2 * (n >> 3);
  const int rr[4] = {rows.x, rows.y, rows.z, rows.w};
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int row = rr[i];
    if constexpr (OM == kOutSplitBF16IL || OM == kOutSplit16IL) {
      float v[2];
#pragma unroll
      for (int b = 0; b < 2; ++b) {
        const float x = lane_xor<4>(acc_im[b][i]);
        v[b] = (im == CONJ ? acc_re[b][i] - x : acc_re[b][i] + x) * a.scale;
      }
      if (row < 0) continue;
      if (a.dc_meas) {
#pragma unroll
        for (int b = 0; b < 2; ++b) v[b] = dc_apply(a, v[b], coil0 + b, row, im ? 1 : 0);
      }
      const u32x2_t w = {split_word<OM == kOutSplitBF16IL>(v[0]), split_word<OM == kOutSplitBF16IL>(v[1])};
      glb(reinterpret_cast<u32x2_t*>(a.out_il))[static_cast<size_t>(row) * kN + 8 * ((n >> 1) & 1u) +
                                                4 * ((n >> 2) & 1u) + 2 * (n & 1u) + (n >> 3)] = w;
    } else {
      float re = acc_re[0][i], ir = acc_re[1][i], ri = acc_im[0][i], ii = acc_im[1][i];
      swap_lanes<4>(re, ir);
      swap_lanes<4>(ri, ii);
      store_value<OM, CONJ, ACC>(a, row, coil0 + (im ? 1u : 0u), re, ri, ir, ii);
    }
  }
}

// Rows of a group from the wave's accumulators (or from summed chunk slots).
template <int NB, int IL, int OM, bool CONJ, bool ACC, int WB>
__device__ __forceinline__ void write_group(const InterpArgs& a, const int4& rows, const float4_t (&acc_re)[NB],
                                            const float4_t (&acc_im)[NB], int lane) {
  if constexpr (IL == kLines) {
    interp_epilogue_lines<OM, CONJ, ACC>(a, rows, acc_re, acc_im, lane);
  } else {
#pragma unroll
    for (int b = 0; b < NB; ++b) interp_epilogue<OM, CONJ, ACC, WB>(a, rows, b, acc_re[b], acc_im[b], lane);
  }
}

// Buffer resources of one launch (wave-uniform, in scalar registers).  Every
// per-tile operand is a buffer load at a scalar tile offset plus a
// loop-invariant lane offset, and every gather one buffer load whose lane
// offset is one VALU op from the stored column word, so the tile loop spends
// almost no vector instructions on addresses.  Out-of-range offsets read 0.
typedef uint32_t u32x4_t __attribute__((ext_vector_type(4)));
typedef __amdgpu_buffer_rsrc_t rsrc_t;

__device__ __forceinline__ rsrc_t make_rsrc(const void* p, uint64_t bytes) {
  const uint32_t n = bytes > 0xFFFFFFFFull ? 0xFFFFFFFFu : static_cast<uint32_t>(bytes);
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(p), static_cast<short>(0), static_cast<int>(n),
                                           0x00020000);
}

template <int NB>
struct TileRsrc {
  rsrc_t cols, a, idx, dense, rows, hi[NB], res[NB];
};

template <int NB, int IL, int WB>
__device__ __forceinline__ TileRsrc<NB> make_tile_rsrc(const InterpArgs& a, uint32_t end_cut = 0) {
  TileRsrc<NB> r;
  const uint64_t tiles = a.n_tiles;
  r.cols = make_rsrc(a.tile_cols, tiles * kK * 4);
  r.a = make_rsrc(a.tile_a, tiles * 64 * 16);
  r.idx = make_rsrc(a.tile_idx, tiles * 64 * 2);
  r.dense = make_rsrc(a.tile_dense, a.tile_dense ? tiles * 64 * 32 : 0);
  r.rows = make_rsrc(a.group_rows, static_cast<uint64_t>(a.n_groups) * 64);
#pragma unroll
  for (int b = 0; b < NB; ++b) {
    if constexpr (IL != kHalves) {
      // (WB = 2: panel_il already points at the wave's block, to the panel's end in line rows)
      if constexpr (IL == kLines) r.hi[b] = make_rsrc(a.panel_il, a.panel_stride * 8);
      else r.hi[b] = make_rsrc(a.panel_il + b * a.panel_stride, a.panel_stride * (WB > 1 && a.lines ? 8 : 4) - end_cut);
      r.res[b] = r.hi[b];
    } else {
      r.hi[b] = make_rsrc(a.panel_hi + b * a.panel_stride, a.panel_stride * 2);
      r.res[b] = make_rsrc(a.panel_res ? a.panel_res + b * a.panel_stride : a.panel_hi, a.panel_stride * 2);
    }
  }
  return r;
}

// Where a lane's output rows of a group start among its 16 (in bytes): the
// quarter's four accumulator rows 4q .. 4q + 3, or, for one coil block's float2
// output, the two of them that the lane stores (interp_epilogue).
template <int IL, int OM>
__device__ __forceinline__ int rows_offset(int lane) {
  constexpr bool kPair = IL != kLines && (OM == kOutCoilMajor || OM == kOutRowMajor);
  return (lane >> 4) * 16 + (kPair && (lane & 8) ? 8 : 0);
}

// Output rows of group g (x and y only where a lane stores two rows; past the
// table's end the buffer range check returns zeros for the unused z and w).
template <int NB, int IL, int OM>
__device__ __forceinline__ int4 load_rows(const TileRsrc<NB>& r, int g, int lane) {
  const u32x4_t v = __builtin_amdgcn_raw_buffer_load_b128(r.rows, rows_offset<IL, OM>(lane), g * 64, 0);
  return make_int4(static_cast<int>(v.x), static_cast<int>(v.y), static_cast<int>(v.z), static_cast<int>(v.w));
}

template <int IL, int OM>
__device__ __forceinline__ int4 group_rows_of(const InterpArgs& a, uint32_t group, int lane) {
  const auto* p = glb(a.group_rows + static_cast<size_t>(group) * 16) + rows_offset<IL, OM>(lane) / 4;
  if constexpr (IL != kLines && (OM == kOutCoilMajor || OM == kOutRowMajor)) return make_int4(p[0], p[1], -1, -1);
  return make_int4(p[0], p[1], p[2], p[3]);
}

// Stage 1 of a tile: the lane's 8 device column words (tile columns
// 8q .. 8q+7).  A word holds the byte offset of the column's row in a half
// panel (column * 32); bit 31 of word 2 is set on the last tile of a group.
struct TileCols {
  u32x4_t c0, c1;
};

// The column words of a unit or chunk (at most kSplitAboveTiles tiles, 128
// bytes each) are copied once into the wave's LDS slice, so the gathers of a
// tile wait for an LDS read instead of a global load issued one step earlier
// (the chain column word -> gather address -> gather otherwise costs a full
// memory latency per tile).  Words past the range read neighbours or zeros
// (unused).
constexpr int kStageWords = kSplitAboveTiles * kK;  // per wave

template <int NB>
__device__ __forceinline__ void stage_cols(const TileRsrc<NB>& r, int first, int n, uint32_t* stage, int lane) {
  // both halves are loaded before either is stored (one memory round trip);
  // past the last tile the buffer range check returns zeros
  (void)n;
  first = __builtin_amdgcn_readfirstlane(first);
  const u32x4_t v0 = __builtin_amdgcn_raw_buffer_load_b128(r.cols, lane * 16, first * (kK * 4), 0);
  const u32x4_t v1 = __builtin_amdgcn_raw_buffer_load_b128(r.cols, 1024 + lane * 16, first * (kK * 4), 0);
  reinterpret_cast<u32x4_t*>(stage)[lane] = v0;
  reinterpret_cast<u32x4_t*>(stage)[64 + lane] = v1;
  __builtin_amdgcn_wave_barrier();
}

// Column words of the unit's k-th tile from the stage (the 16 lanes of a
// quarter read the same 32 bytes: LDS broadcast).
template <int IL>
__device__ __forceinline__ TileCols staged_cols(const uint32_t* stage, int k, int lane) {
  TileCols c;
  if constexpr (IL == kLines) {  // four columns a lane (fetch_ops)
    c.c0 = reinterpret_cast<const u32x4_t*>(stage + k * kK)[lane >> 3];
    c.c1 = c.c0;
  } else {
    const u32x4_t* p = reinterpret_cast<const u32x4_t*>(stage + k * kK) + (lane >> 4) * 2;
    c.c0 = p[0];
    c.c1 = p[1];
  }
  return c;
}

// Stage 2 of a tile: A fragment, sparse index bytes, last-tile flag and the
// raw gathered panel words (kept unpacked until the multiply so no wait is
// forced before then).  IL: one dword (hi | res << 16) per row; otherwise one
// zero-extended half per row for hi (w[0..7]) and for the residual (w[8..15]).
template <int NB, int IL>
struct TileOps {
  u32x4_t a0, a1;
  uint32_t idx, last;
  uint32_t w[NB][IL == kHalves ? 16 : 8];
};

template <int KIND, int NB, int IL, int WB>
__device__ __forceinline__ void fetch_ops(const TileRsrc<NB>& r, int t, const TileCols& c, int lane, uint32_t shift,
                                          TileOps<NB, IL>& o) {
  const uint32_t n = lane & 15;
  const uint32_t cw[8] = {c.c0.x, c.c0.y, c.c0.z, c.c0.w, c.c1.x, c.c1.y, c.c1.z, c.c1.w};
  if constexpr (IL == kLines) {
    // Whole 128-byte lines, 16 bytes a lane: lanes n < 8 of quarter q read its
    // columns 8q .. 8q + 3, lanes n >= 8 columns 8q + 4 .. 8q + 7, 16-byte quad
    // 4 ((n >> 1) & 1) + 2 ((n >> 2) & 1) + (n & 1) of each (block, part, coil
    // half; mma_tile exchanges half of the words with lane n ^ 8).  Rows of 128
    // bytes in L2, 32 columns a step, 16 waves a CU: 80 cycles a CU, against
    // 104 as two 64-byte halves in 4-byte loads and 140 in 8-byte loads.
    static_assert(NB == 2, "line rows hold two coil blocks");
    const uint32_t quad = ((n & 2) << 5) | ((n & 4) << 3) | ((n & 1) << 4);
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const u32x4_t v =
          __builtin_amdgcn_raw_buffer_load_b128(r.hi[0], static_cast<int>((cw[j] << 2) | quad), 0, 0);
      o.w[0][j] = v.x;
      o.w[1][j] = v.y;
      o.w[0][4 + j] = v.z;
      o.w[1][4 + j] = v.w;
    }
  } else {
#pragma unroll
  for (int b = 0; b < NB; ++b) {
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      if constexpr (IL == kBlocks) {
        // row byte offset in the interleaved panel: column * 64 (128 in line rows) + n * 4
        const uint32_t off = (cw[j] << (WB > 1 ? shift : 1u)) | (n << 2);
        o.w[b][j] = __builtin_amdgcn_raw_buffer_load_b32(r.hi[b], static_cast<int>(off), 0, 0);
      } else {
        const uint32_t off = (j == 2 ? (cw[j] & 0x7FFFFFFFu) : cw[j]) | (n << 1);
        o.w[b][j] = __builtin_amdgcn_raw_buffer_load_b16(r.hi[b], static_cast<int>(off), 0, 0);
        o.w[b][8 + j] = KIND == kSparseHi ? 0u
                                          : __builtin_amdgcn_raw_buffer_load_b16(r.res[b], static_cast<int>(off), 0, 0);
      }
    }
  }
  }
  if constexpr (KIND == kDenseSplit) {
    o.a0 = __builtin_amdgcn_raw_buffer_load_b128(r.dense, lane * 32, t * (64 * 32), 0);
    o.a1 = __builtin_amdgcn_raw_buffer_load_b128(r.dense, lane * 32 + 16, t * (64 * 32), 0);
    o.idx = 0;
  } else {
    o.a0 = __builtin_amdgcn_raw_buffer_load_b128(r.a, lane * 16, t * (64 * 16), 0);
    o.a1 = u32x4_t{0u, 0u, 0u, 0u};
    o.idx = __builtin_amdgcn_raw_buffer_load_b16(r.idx, lane * 2, t * (64 * 2), 0);
  }
  o.last = c.c0.z >> 31;
}

// hi (sel 0x05040100) or residual (sel 0x07060302) halves of 8 words as half8.
__device__ __forceinline__ half8_t pack_halves(const uint32_t* w, uint32_t sel) {
  u32x4_t v;
  v.x = __builtin_amdgcn_perm(w[1], w[0], sel);
  v.y = __builtin_amdgcn_perm(w[3], w[2], sel);
  v.z = __builtin_amdgcn_perm(w[5], w[4], sel);
  v.w = __builtin_amdgcn_perm(w[7], w[6], sel);
  return __builtin_bit_cast(half8_t, v);
}
constexpr uint32_t kSelLo = 0x05040100u, kSelHi = 0x07060302u;

template <int KIND, int NB, int IL>
__device__ __forceinline__ void mma_tile(TileOps<NB, IL>& o, float4_t (&acc_re)[NB],
                                         float4_t (&acc_im)[NB]) {
#pragma unroll
  for (int b = 0; b < NB; ++b) {
    if constexpr (IL == kLines) {
      // every lane gets words 2 (n >> 3) + b of its quad of all 8 columns
#pragma unroll
      for (int j = 0; j < 4; ++j) swap_lanes<8>(o.w[b][j], o.w[b][4 + j]);
    }
    const half8_t hi = pack_halves(o.w[b], kSelLo);
    half8_t res;
    if constexpr (IL == kHalves) res = pack_halves(o.w[b] + 8, kSelLo);
    else res = pack_halves(o.w[b], kSelHi);
    if constexpr (KIND == kDenseSplit) {
      const half8_t dre = __builtin_bit_cast(half8_t, o.a0);
      const half8_t dim = __builtin_bit_cast(half8_t, o.a1);
      acc_re[b] = __builtin_amdgcn_mfma_f32_16x16x32_f16(dre, hi, acc_re[b], 0, 0, 0);
      acc_im[b] = __builtin_amdgcn_mfma_f32_16x16x32_f16(dim, hi, acc_im[b], 0, 0, 0);
      acc_re[b] = __builtin_amdgcn_mfma_f32_16x16x32_f16(dre, res, acc_re[b], 0, 0, 0);
      acc_im[b] = __builtin_amdgcn_mfma_f32_16x16x32_f16(dim, res, acc_im[b], 0, 0, 0);
    } else if constexpr (KIND == kSparseSplitBF16) {
      const bf16x4_t are = __builtin_bit_cast(bf16x4_t, make_uint2(o.a0.x, o.a0.y));
      const bf16x4_t aim = __builtin_bit_cast(bf16x4_t, make_uint2(o.a0.z, o.a0.w));
      const bf16x8_t bhi = __builtin_bit_cast(bf16x8_t, hi);
      const bf16x8_t bres = __builtin_bit_cast(bf16x8_t, res);
      const int idx = static_cast<int>(o.idx);
      acc_re[b] = __builtin_amdgcn_smfmac_f32_16x16x32_bf16(are, bhi, acc_re[b], idx, 0, 0);
      acc_im[b] = __builtin_amdgcn_smfmac_f32_16x16x32_bf16(aim, bhi, acc_im[b], idx, 0, 1);
      acc_re[b] = __builtin_amdgcn_smfmac_f32_16x16x32_bf16(are, bres, acc_re[b], idx, 0, 0);
      acc_im[b] = __builtin_amdgcn_smfmac_f32_16x16x32_bf16(aim, bres, acc_im[b], idx, 0, 1);
    } else {
      const half4_t are = __builtin_bit_cast(half4_t, make_uint2(o.a0.x, o.a0.y));
      const half4_t aim = __builtin_bit_cast(half4_t, make_uint2(o.a0.z, o.a0.w));
      const int idx = static_cast<int>(o.idx);
      acc_re[b] = __builtin_amdgcn_smfmac_f32_16x16x32_f16(are, hi, acc_re[b], idx, 0, 0);
      acc_im[b] = __builtin_amdgcn_smfmac_f32_16x16x32_f16(aim, hi, acc_im[b], idx, 0, 1);
      if constexpr (KIND == kSparseSplit) {
        acc_re[b] = __builtin_amdgcn_smfmac_f32_16x16x32_f16(are, res, acc_re[b], idx, 0, 0);
        acc_im[b] = __builtin_amdgcn_smfmac_f32_16x16x32_f16(aim, res, acc_im[b], idx, 0, 1);
      }
    }
  }
}

// Gather stages in flight ahead of the multiply: 2 for one coil block of the
// interleaved panel, 0 for two coil blocks of separate panels or of
// dense-control tiles, else 1 (deeper stages measured no faster and cost
// occupancy).
template <int KIND, int NB, int IL>
struct PipeDepth {
  static constexpr int value = (IL != kHalves && NB == 1 && KIND != kDenseSplit) ? 2
                               : (NB == 2 && (IL == kHalves || KIND == kDenseSplit)) ? 0
                                                                          : 1;
};

// Stream tiles first .. end - 1 (at most kSplitAboveTiles, column words
// staged) of one wave through a software pipeline.  Step i reads the column
// words of tile i + D + 1 from the stage, issues the operand loads of tile
// i + D, then multiplies tile i (D: PipeDepth, or the autotuner's choice);
// operand loads return in issue order, so the multiply's wait leaves D tiles
// of loads in flight.
// Tile i lives in register slot i % U of both rings (U = max(D + 1, 2), the
// loop unrolled U times so every slot index is a constant).  Indices past the
// end are clamped to the last tile (valid, unused loads).  The tiles are
// those of the consecutive groups group, group + 1, ... (< group_end); with
// last_mask 1 the last tile of each runs the epilogue with the group's rows
// (loaded one group ahead) and resets the accumulators; with 0 (a chunk of a
// long group) everything accumulates.  One loop for both keeps the kernel's
// register count at that of the regular units.
template <int KIND, int NB, int IL, int OM, bool CONJ, bool ACC, int WB, int D>
__device__ __forceinline__ void stream_tiles(const InterpArgs& a, const TileRsrc<NB>& r, int first, int end,
                                             int group, int group_end, uint32_t last_mask, float4_t (&acc_re)[NB],
                                             float4_t (&acc_im)[NB], int lane, const uint32_t* stage) {
  constexpr int U = D + 1 > 2 ? D + 1 : 2;
  // wave-uniform bounds: scalar control flow and scalar tile offsets
  first = __builtin_amdgcn_readfirstlane(first);
  end = __builtin_amdgcn_readfirstlane(end);
  int g = __builtin_amdgcn_readfirstlane(group);
  const int g_last = __builtin_amdgcn_readfirstlane(group_end) - 1;
  if (first >= end) return;
  const int n = end - first;
  const int last = end - 1;
  auto tile = [&](int i) { return min(first + i, last); };
  auto cols_of = [&](int i) { return staged_cols<IL>(stage, tile(i) - first, lane); };
  last_mask = __builtin_amdgcn_readfirstlane(last_mask);
  int4 rows = load_rows<NB, IL, OM>(r, g, lane);
  TileCols cols[U];
  TileOps<NB, IL> ops[U];
  // The scheduler must keep the issue order: the wait counter is in order, and
  // the loop's waits are computed over both the prologue and the back edge.
#pragma unroll
  for (int i = 0; i <= D; ++i) cols[i % U] = cols_of(i);
  __builtin_amdgcn_sched_barrier(0);
#pragma unroll
  for (int i = 0; i < D; ++i) {
    fetch_ops<KIND, NB, IL, WB>(r, tile(i), cols[i % U], lane, 1u + a.lines, ops[i % U]);
    __builtin_amdgcn_sched_barrier(0);
  }
  for (int base = 0; base < n; base += U) {
#pragma unroll
    for (int j = 0; j < U; ++j) {
      const int i = base + j;
      __builtin_amdgcn_sched_barrier(0);
      // loads run unconditionally (clamped), only the multiply is skipped past
      // the end, so no loaded register is merged across a branch
      cols[(j + D + 1) % U] = cols_of(i + D + 1);
      __builtin_amdgcn_sched_barrier(0);
      fetch_ops<KIND, NB, IL, WB>(r, tile(i + D), cols[(j + D) % U], lane, 1u + a.lines, ops[(j + D) % U]);
      if (i < n) {
        mma_tile<KIND, NB, IL>(ops[j], acc_re, acc_im);
        if (__builtin_amdgcn_readfirstlane(ops[j].last) & last_mask) {
          write_group<NB, IL, OM, CONJ, ACC, WB>(a, rows, acc_re, acc_im, lane);
#pragma unroll
          for (int b = 0; b < NB; ++b) {
            acc_re[b] = float4_t{0.f, 0.f, 0.f, 0.f};
            acc_im[b] = float4_t{0.f, 0.f, 0.f, 0.f};
          }
          g = min(g + 1, g_last);
          rows = load_rows<NB, IL, OM>(r, g, lane);
        }
      }
    }
  }
}

// After a chunk of a long group has streamed its tiles: publish the partial
// sums, and if this wave is the group's last arrival, add every chunk's slot in
// chunk order and write the group's rows.  Slots are written and read with
// device-scope (sc1) 16-byte buffer accesses, the access a relaxed agent-scope
// atomic of each word compiles to: they reach past the per-XCD L2 without a
// cache flush.  The stores complete (vmcnt 0) before the arrival is counted,
// and the slots are read only after the count shows every chunk done.  A full
// agent-scope fence here would write back the whole L2 per chunk (measured:
// the launch went from 29 to 230 us).  The last wave resets the counter for
// the next launch.  No wave waits on another.
// The protocol rests on gfx950's mapping of device-scope accesses (sc1
// stores and loads reach the coherent level past the per-XCD L2, in issue
// order with respect to the counter's atomic after the store wait) rather
// than on language-level acquire/release; other targets are refused here.
#if defined(__HIP_DEVICE_COMPILE__) && !defined(__gfx950__)
#error "the chunk-slot protocol of the interpolation kernels is written for gfx950"
#endif
constexpr int kCpolDevice = 16;  // cache policy bits of a buffer access: sc1 (device scope)
constexpr uint32_t kSlotBatch = 8;  // slots loaded before the first add (one round trip for <= 8 chunks)
// Slot byte offsets are 32-bit buffer offsets: at most 2^31 bytes of slots.
constexpr uint32_t kMaxSlots = (1u << 31) / (kSlotFloats * 4);

// WB > 1 (one wave per coil block of the entry): wave wb publishes its
// accumulators as block wb, the group's last arrival of all chunks and waves
// adds the slots of every block; a holds the unshifted (block 0) arguments.
template <int OM, bool CONJ, bool ACC, int NB, int IL, int WB = 1>
__device__ __forceinline__ void chunk_finish(const InterpArgs& a, const ChunkItem& c, float4_t (&acc_re)[NB],
                                             float4_t (&acc_im)[NB], int lane, int wb = 0) {
  // slot layout: [coil block][re, im][lane][4] floats; slot offsets stay below
  // 2^32 bytes (kSlotFloats * 4 bytes per chunk)
  static_assert(NB * WB <= 2, "a slot holds two coil blocks");
  const rsrc_t slots = make_rsrc(a.partials, uint64_t{1} << 32);
  const int mine = static_cast<int>((c.slot0 + c.chunk) * kSlotFloats * 4);
#pragma unroll
  for (int b = 0; b < NB; ++b) {
    __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4_t, acc_re[b]), slots,
                                           (((b + wb) * 2 + 0) * 64 + lane) * 16, mine, kCpolDevice);
    __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4_t, acc_im[b]), slots,
                                           (((b + wb) * 2 + 1) * 64 + lane) * 16, mine, kCpolDevice);
  }
  __builtin_amdgcn_s_waitcnt(0);  // every slot store acknowledged
  asm volatile("" ::: "memory");
  uint32_t arrived = 0;
  if (lane == 0)
    arrived = __hip_atomic_fetch_add(a.counters + c.counter, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  arrived = __builtin_amdgcn_readfirstlane(arrived);
  if (arrived + 1 != c.n_chunks * WB) return;
  asm volatile("" ::: "memory");
  if (lane == 0) __hip_atomic_store(a.counters + c.counter, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  const int first = static_cast<int>(c.slot0 * kSlotFloats * 4);
  const int4 rows = group_rows_of<IL, OM>(a, static_cast<uint32_t>(c.group), lane);
  const uint32_t n = c.n_chunks;
  float4_t sum_re[NB * WB], sum_im[NB * WB];
#pragma unroll
  for (int b = 0; b < NB * WB; ++b) {
    float4_t re = float4_t{0.f, 0.f, 0.f, 0.f}, im = re;
    // kSlotBatch slots are loaded (all before the first add), then added in
    // chunk order: ceil(n / kSlotBatch) memory round trips
    for (uint32_t q0 = 0; q0 < n; q0 += kSlotBatch) {
      float4_t pr[kSlotBatch], pi[kSlotBatch];
#pragma unroll
      for (uint32_t j = 0; j < kSlotBatch; ++j) {
        const int so = first + static_cast<int>(min(q0 + j, n - 1) * kSlotFloats * 4);
        pr[j] = __builtin_bit_cast(float4_t, __builtin_amdgcn_raw_buffer_load_b128(
                                                 slots, ((b * 2 + 0) * 64 + lane) * 16, so, kCpolDevice));
        pi[j] = __builtin_bit_cast(float4_t, __builtin_amdgcn_raw_buffer_load_b128(
                                                 slots, ((b * 2 + 1) * 64 + lane) * 16, so, kCpolDevice));
      }
#pragma unroll
      for (uint32_t j = 0; j < kSlotBatch; ++j) {
        if (q0 + j >= n) break;
        if (q0 + j == 0) {
          re = pr[j];
          im = pi[j];
        } else {
          re += pr[j];
          im += pi[j];
        }
      }
    }
    sum_re[b] = re;
    sum_im[b] = im;
  }
  write_group<NB * WB, IL, OM, CONJ, ACC, WB>(a, rows, sum_re, sum_im, lane);
}

// One wave per block, one entry of the launch order each (a regular unit, a
// run of whole groups, or a chunk of a long group), the entries of one XCD
// contiguous in pack order.  One-wave blocks let the dispatcher start a new
// entry whenever a wave slot frees, so uneven entries balance themselves
// across the CUs.  Units and chunks share one tile loop (one inlined copy
// keeps the register count of the regular units).
// WB = 2 (entries of two coil blocks, NB = 1): a block of two waves per
// entry, wave w computing coil block w.  Both stream the entry's tile operands
// (the second read comes from cache: the two waves share a CU), each with the
// one-block register budget and pipeline, and gather only its own panel.
// (the arguments by value: a reference to the kernel's by-value argument
// would make the compiler copy it to scratch and read it back through flat
// loads)
template <int KIND, int NB, int IL, int OM, bool CONJ, bool ACC, int WB, int D>
__device__ __forceinline__ void tiles_entry(InterpArgs a) {
  static_assert(WB == 1 || NB == 1, "one wave per coil block covers one block");
  __shared__ uint32_t stages[WB][kStageWords];
  const int lane = threadIdx.x & 63;
  const int wb = WB > 1 ? __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x >> 6)) : 0;
  uint32_t* stage = stages[wb];
  float4_t acc_re[NB], acc_im[NB];
#pragma unroll
  for (int b = 0; b < NB; ++b) {
    acc_re[b] = float4_t{0.f, 0.f, 0.f, 0.f};
    acc_im[b] = float4_t{0.f, 0.f, 0.f, 0.f};
  }
  const uint32_t entry = glb(a.order)[xcd_remap(blockIdx.x, gridDim.x)];
  const bool is_chunk = (entry & kChunkTag) != 0;
  ChunkItem c{};
  WorkItem u;
  uint32_t problem = 0;
  if (is_chunk) {
    c = a.chunks[entry & ~kChunkTag];
    u = {c.group, c.group + 1, c.tile_begin, c.tile_end};
    problem = c.problem;
  } else {
    u = a.items[entry];
    if (a.problems) problem = glb(a.item_problem)[entry];
  }
  InterpArgs v = a;
  if constexpr (IL != kHalves) {
    if (a.problems) v = problem_args(a, problem);
  }
  // this wave's coil block: input panel, output coils and split-panel block
  InterpArgs vw = v;
  uint32_t end_cut = 0;
  if constexpr (WB > 1) {
    // separate blocks, or this block's half of every line row
    vw.lines = __builtin_amdgcn_readfirstlane(v.lines);
    end_cut = vw.lines ? wb * kN * 4 : 0;
    vw.panel_il = v.panel_il ? v.panel_il + wb * (vw.lines ? static_cast<uint64_t>(kN) : v.panel_stride) : nullptr;
    vw.panel_hi = v.panel_hi ? v.panel_hi + wb * v.panel_stride : nullptr;
    vw.panel_res = v.panel_res ? v.panel_res + wb * v.panel_stride : nullptr;
    vw.coil_base = v.coil_base + wb * kCoilsPerBlock;
    const size_t out_block = static_cast<size_t>(wb) * v.n_out * kN;
    vw.out_il = v.out_il ? v.out_il + (vw.lines ? static_cast<size_t>(wb) * kN : out_block) : nullptr;
  }
  if (u.tile_begin == u.tile_end) {  // empty group: zero rows
    const int4 rows = group_rows_of<IL, OM>(vw, static_cast<uint32_t>(u.group), lane);
    write_group<NB, IL, OM, CONJ, ACC, WB>(vw, rows, acc_re, acc_im, lane);
    return;
  }
  const TileRsrc<NB> r = make_tile_rsrc<NB, IL, WB>(vw, end_cut);
  stage_cols(r, u.tile_begin, u.tile_end - u.tile_begin, stage, lane);
  stream_tiles<KIND, NB, IL, OM, CONJ, ACC, WB, D>(vw, r, u.tile_begin, u.tile_end, u.group, u.group_end,
                                               is_chunk ? 0u : 1u, acc_re, acc_im, lane, stage);
  if (is_chunk) chunk_finish<OM, CONJ, ACC, NB, IL, WB>(v, c, acc_re, acc_im, lane, wb);
}

template <int KIND, int NB, int IL, int OM, bool CONJ, bool ACC, int WB = 1>
__global__ __launch_bounds__(64 * WB) void interp_tiles_kernel(InterpArgs a) {
  tiles_entry<KIND, NB, IL, OM, CONJ, ACC, WB, PipeDepth<KIND, NB, IL>::value>(a);
}

// The same with another pipeline depth D (the autotuner's alternatives).
template <int KIND, int NB, int IL, int OM, bool CONJ, bool ACC, int WB, int D>
__global__ __launch_bounds__(64 * WB) void interp_tiles_depth_kernel(InterpArgs a) {
  tiles_entry<KIND, NB, IL, OM, CONJ, ACC, WB, D>(a);
}


struct CsrArgs {
  const CsrBlock* blocks;
  uint32_t n_blocks, n_active;  // (the rest: trailing runs of empty rows)
  const CsrRound* rounds;  // rounds after the first of each block
  const int32_t* row_ids;
  const uint32_t* cols;    // distinct columns of each round
  const float2* vals;      // [steps][64] entry values (see CsrBlock)
  const uint32_t* idx;     // [ceil(steps / 4)][64] local columns, one byte a step
  float2* partials;        // [slots][kMaxCoils] partial sums of long-row chunks
  uint32_t* counters;      // one arrival counter per group of long rows, zero between launches
  const float2* in;
  uint32_t n_cols;
  uint32_t coils;
  uint32_t n_out;
  float scale;
  float2* out;
  uint32_t skip_empty;  // the output's empty rows already hold zeros: runs of empty rows write nothing
};

// Plain FP32 path.  A block of four waves takes one CsrBlock: rows neighbouring
// in k-space, in rounds of at most kCsrCols distinct input rows that their
// entries name.  A round copies those input rows (float2 [row][coils]) into LDS
// once and forms every product from there: neighbouring rows share most of
// their columns, so an input row is fetched once per block instead of once per
// entry (205,824 samples / 512^2 / 8 coils: 47 MB of gathers a launch instead
// of 474 MB).  Four lanes (a quad) work on a row, CPL coils each; lane k of the
// quad holds entries 4t + k, so one coalesced load brings 4 entries of 16 rows,
// and the quad shares them by DPP broadcasts folded into the arithmetic (no LDS
// traffic but the input rows, one 16-byte read a lane and entry at 8 coils).
// The four input rows of a step are read before the first is used (two at a
// time: 256^2 solve of 6 steps 531 -> 517 us at 8 coils).  Values and one-byte
// local columns stream from memory, the next four steps loaded ahead.
// Rows of up to kCsrShortEntries entries are summed in entry order.  Chunks (at
// most kCsrChunkEntries entries) of longer rows take four quads, quad p the
// entries p mod 4, in 4 SUMS strided partial sums combined in a fixed tree;
// the chunks of a row publish partial sums that the last arrival adds in chunk
// order (the slot protocol of the packed kernel's long groups).  No sum depends
// on the schedule: SUMS follows from the coil count alone (4 up to 4 coils, 2 up
// to 8, else 1).
// A launch of many blocks covers all coils in each (CPL = 4 / SUMS).  One of up
// to kCsrFewBlocks leaves compute units idle and lasts as long as one wave's
// chain of LDS reads and multiply-adds: it takes CPL = 1 and blockIdx.y runs
// over groups of four coils.  Measured, one group of coils -> groups of four:
// 272 blocks (32^2 image, 16 coils) 7.4 -> 5.3 us, 392 blocks (64^2, 6 coils)
// 5.4 -> 5.0, 456 blocks (128^2, 8 coils) 6.0 -> 5.8; 584 blocks 7.8 -> 7.7 at 8
// coils, 11.6 -> 11.9 at 16; 960 blocks 7.8 -> 8.1, 1392 blocks 8.6 -> 9.5.
// Measured against one lane group per row that gathered every entry from memory
// (512^2 / 8 coils): forward 43-46 -> 20 us, adjoint 59-65 -> 26 us, sums bit
// for bit the same.
template <int CTRL>
__device__ __forceinline__ float quad_bcast(float v) {
  return __builtin_bit_cast(float, __builtin_amdgcn_mov_dpp(__builtin_bit_cast(int, v), CTRL, 0xF, 0xF, true));
}
template <int CTRL>
__device__ __forceinline__ uint32_t quad_bcast(uint32_t v) {
  return static_cast<uint32_t>(__builtin_amdgcn_mov_dpp(static_cast<int>(v), CTRL, 0xF, 0xF, true));
}

template <int CPL>
struct CsrCoils {
  float2_t v[CPL];
};

// acc += v * x (conj(v) * x) for the CPL coils of a lane: each product rounded
// as a multiply and a fused multiply-add, then added.
template <int CPL, bool CONJ>
__device__ __forceinline__ void csr_mac(float vr, float vi, const CsrCoils<CPL>& x, CsrCoils<CPL>& acc) {
#pragma clang fp contract(off)
#pragma unroll
  for (int c = 0; c < CPL; ++c) {
    const float a = vi * x.v[c].y, b = vi * x.v[c].x;
    acc.v[c].x += __builtin_fmaf(vr, x.v[c].x, CONJ ? a : -a);
    acc.v[c].y += __builtin_fmaf(vr, x.v[c].y, CONJ ? -b : b);
  }
}

// Input row of entry 4t + K of the quad's row (lane K's local column).
template <int CPL, int K>
__device__ __forceinline__ void csr_read(const char* stage, uint32_t at, uint32_t lane_off, CsrCoils<CPL>& x) {
  const uint32_t o = quad_bcast<K * 0x55>(at) + lane_off;  // quad_perm [K, K, K, K]
  if constexpr (CPL == 1) {
    x.v[0] = *reinterpret_cast<const float2_t*>(stage + o);
  } else {
#pragma unroll
    for (int c = 0; c < CPL; c += 2) {
      const float4_t q = *reinterpret_cast<const float4_t*>(stage + o + c * 8);
      x.v[c] = float2_t{q.x, q.y};
      x.v[c + 1] = float2_t{q.z, q.w};
    }
  }
}

template <int OM, bool ACC>
__device__ __forceinline__ void csr_store(const CsrArgs& a, int32_t row, uint32_t c, float re, float im) {
  float2_t v = float2_t{re * a.scale, im * a.scale};
  size_t o;
  if constexpr (OM == kOutCoilMajor) o = static_cast<size_t>(c) * a.n_out + row;
  else o = static_cast<size_t>(row) * a.coils + c;
  float2_t* out = reinterpret_cast<float2_t*>(a.out);
  if constexpr (ACC) v += glb(out)[o];
  glb(out)[o] = v;
}

// The entry values and local columns of one wave's round (wave-uniform bases,
// so that a load needs no address registers: a step is a scalar offset).
struct CsrStream {
  rsrc_t vals, idx;
  uint32_t steps;
};
__device__ __forceinline__ float2_t csr_value(const CsrStream& s, uint32_t t, uint32_t lane) {
  return __builtin_bit_cast(float2_t, __builtin_amdgcn_raw_buffer_load_b64(
                                          s.vals, lane * 8, static_cast<int>(min(t, s.steps - 1) * 512), 0));
}
__device__ __forceinline__ uint32_t csr_columns(const CsrStream& s, uint32_t word, uint32_t lane) {
  return __builtin_amdgcn_raw_buffer_load_b32(s.idx, lane * 4, static_cast<int>(word * 256), 0);
}

// The entries of one round of the wave's quads.  STRIDED: entry i of a quad
// goes to sum i mod NA, else all to sum 0.
template <int CPL, bool CONJ, bool STRIDED, int NA>
__device__ __forceinline__ void csr_round(const CsrStream& s, const char* stage, uint32_t lane, uint32_t lane_off,
                                          float2_t (&val)[4], uint32_t at, CsrCoils<CPL> (&acc)[NA]) {
  float2_t next_val[4];
  uint32_t next_at = 0;
  for (uint32_t t0 = 0; t0 < s.steps; t0 += 4) {
    if (t0 + 4 < s.steps) {
#pragma unroll
      for (int i = 0; i < 4; ++i) next_val[i] = csr_value(s, t0 + 4 + i, lane);
      next_at = csr_columns(s, t0 / 4 + 1, lane);
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      if (t0 + i < s.steps) {
        const uint32_t o = ((at >> (8 * i)) & 0xFFu) * (4 * CPL * 8);
        CsrCoils<CPL> x[4];
        csr_read<CPL, 0>(stage, o, lane_off, x[0]);
        csr_read<CPL, 1>(stage, o, lane_off, x[1]);
        csr_read<CPL, 2>(stage, o, lane_off, x[2]);
        csr_read<CPL, 3>(stage, o, lane_off, x[3]);
        if constexpr (CPL < 4) __builtin_amdgcn_sched_barrier(0);
        csr_mac<CPL, CONJ>(quad_bcast<0x00>(val[i].x), quad_bcast<0x00>(val[i].y), x[0], acc[0]);
        csr_mac<CPL, CONJ>(quad_bcast<0x55>(val[i].x), quad_bcast<0x55>(val[i].y), x[1], acc[STRIDED ? 1 % NA : 0]);
        csr_mac<CPL, CONJ>(quad_bcast<0xAA>(val[i].x), quad_bcast<0xAA>(val[i].y), x[2], acc[STRIDED ? 2 % NA : 0]);
        csr_mac<CPL, CONJ>(quad_bcast<0xFF>(val[i].x), quad_bcast<0xFF>(val[i].y), x[3], acc[STRIDED ? 3 % NA : 0]);
      }
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) val[i] = next_val[i];
    at = next_at;
  }
}

template <int CPL, int SUMS, int OM, bool CONJ, bool ACC>
__global__ __launch_bounds__(256) void interp_csr_kernel(CsrArgs a) {
  constexpr int kCoils = 4 * CPL;  // coils of an LDS row
  __shared__ __align__(16) float2_t stage[(kCsrCols + 1) * kCoils];
  __shared__ uint32_t last_arrival;
  const uint32_t tid = threadIdx.x, lane = tid & 63u, l = tid & 3u, quad = tid >> 2;
  const uint32_t w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const uint32_t coil0 = blockIdx.y * kCoils, coil = coil0 + l * CPL;
  // csr_balance cut the active blocks for the XCDs; runs of empty rows follow
  // (both remapped as one, every XCD's range shifted: an adjoint into a new
  // output timed by events, 8 coils, 512^2 39 -> 34 us, 768^2 74 -> 61 us)
  const CsrBlock it = a.blocks[blockIdx.x < a.n_active ? xcd_remap(blockIdx.x, a.n_active) : blockIdx.x];
  if (it.n_rounds == 0) {
    // a run of empty rows (at most kCsrEmptyRunRows): zeros, unless the output
    // holds them already or the launch accumulates
    if (ACC || a.skip_empty) return;
    for (uint32_t o = tid; o < it.n_rows * kCoils; o += 256) {
      const uint32_t c = o % kCoils;
      if (coil0 + c < a.coils) csr_store<OM, false>(a, glb(a.row_ids)[it.row0 + o / kCoils], coil0 + c, 0.f, 0.f);
    }
    return;
  }
  // the output row of the thread's quad, or of its four quads of a chunk (loaded
  // here: at the end it is another trip to memory before the store)
  const int32_t out_row = glb(a.row_ids)[it.row0 + min(it.n_chunks ? tid >> 4 : quad, it.n_rows - 1u)];
  const uint32_t row_bytes = a.coils * 8;
  const rsrc_t in = make_rsrc(a.in, static_cast<uint64_t>(a.n_cols) * row_bytes);
  const uint32_t lane_off = l * CPL * 8;
  CsrCoils<CPL> acc[SUMS];
#pragma unroll
  for (int k = 0; k < SUMS; ++k)
#pragma unroll
    for (int c = 0; c < CPL; ++c) acc[k].v[c] = float2_t{0.f, 0.f};
  if (tid < kCoils) stage[tid] = float2_t{0.f, 0.f};  // row 0: the column of padding entries
  CsrRound rd = it.first;
  for (uint32_t k = 0;;) {
    // the round's column ids, its first entries, then the rows the ids name
    uint32_t cid[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) cid[i] = glb(a.cols)[rd.col0 + min(i * 64 + quad, rd.n_cols - 1u)];
    uint32_t ent = rd.ent0, ix = rd.idx0;
    for (uint32_t i = 0; i < w; ++i) {
      const uint32_t t = (rd.steps >> (8 * i)) & 0xFFu;
      ent += t;
      ix += (t + 3) / 4;
    }
    CsrStream es;
    es.steps = (rd.steps >> (8 * w)) & 0xFFu;
    es.vals = make_rsrc(a.vals + static_cast<size_t>(ent) * 64, uint64_t{es.steps} * 512);
    es.idx = make_rsrc(a.idx + static_cast<size_t>(ix) * 64, uint64_t{(es.steps + 3) / 4} * 256);
    float2_t val[4];
    uint32_t at = 0;
    if (es.steps) {
#pragma unroll
      for (int i = 0; i < 4; ++i) val[i] = csr_value(es, i, lane);
      at = csr_columns(es, 0, lane);
    }
    // (lanes past the problem's coils read the next row or, past the end,
    // zeros; their sums are never stored)
    u32x4_t g[4][CPL == 4 ? 2 : 1];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const uint32_t o = cid[i] * row_bytes + coil * 8;
      if constexpr (CPL == 1) {
        const u32x2_t v = __builtin_bit_cast(u32x2_t, __builtin_amdgcn_raw_buffer_load_b64(in, o, 0, 0));
        g[i][0] = u32x4_t{v.x, v.y, 0u, 0u};
      } else {
#pragma unroll
        for (int c = 0; c < CPL / 2; ++c) g[i][c] = __builtin_amdgcn_raw_buffer_load_b128(in, o + c * 16, 0, 0);
      }
    }
    if (k) __syncthreads();  // every wave is done with the last round's stage
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const uint32_t r = i * 64 + quad;
      if (r >= rd.n_cols) continue;
      float2_t* to = stage + (r + 1) * kCoils + l * CPL;
      if constexpr (CPL == 1) {
        *to = __builtin_bit_cast(float2_t, u32x2_t{g[i][0].x, g[i][0].y});
      } else {
#pragma unroll
        for (int c = 0; c < CPL / 2; ++c) reinterpret_cast<u32x4_t*>(to)[c] = g[i][c];
      }
    }
    __syncthreads();
    const char* base = reinterpret_cast<const char*>(stage);
    if (it.n_chunks == 0) csr_round<CPL, CONJ, false, SUMS>(es, base, lane, lane_off, val, at, acc);
    else csr_round<CPL, CONJ, true, SUMS>(es, base, lane, lane_off, val, at, acc);
    if (++k == it.n_rounds) break;
    const auto* next = reinterpret_cast<const __attribute__((address_space(4))) CsrRound*>(
        reinterpret_cast<uintptr_t>(a.rounds + it.round0 + k - 1));
    rd = CsrRound{next->col0, next->n_cols, next->ent0, next->idx0, next->steps};
  }
  if (it.n_chunks == 0) {  // quad q is row q
    if (quad >= it.n_rows) return;
#pragma unroll
    for (int c = 0; c < CPL; ++c)
      if (coil + c < a.coils) csr_store<OM, ACC>(a, out_row, coil + c, acc[0].v[c].x, acc[0].v[c].y);
    return;
  }
  // four quads a row: strided sum 4 a + p of quad p, added pairwise over p,
  // then over a
  CsrCoils<CPL> sum;
#pragma unroll
  for (int c = 0; c < CPL; ++c) {
#pragma unroll
    for (int k = 0; k < SUMS; ++k) {
#pragma unroll
      for (int off = 4; off < 16; off <<= 1) {
        acc[k].v[c].x += __shfl_xor(acc[k].v[c].x, off);
        acc[k].v[c].y += __shfl_xor(acc[k].v[c].y, off);
      }
    }
    if constexpr (SUMS == 4) sum.v[c] = (acc[0].v[c] + acc[1].v[c]) + (acc[2].v[c] + acc[3].v[c]);
    else if constexpr (SUMS == 2) sum.v[c] = acc[0].v[c] + acc[1].v[c];
    else sum.v[c] = acc[0].v[c];
  }
  const uint32_t r = tid >> 4;
  const bool owner = (quad & 3u) == 0 && r < it.n_rows;
  if (it.n_chunks == 1) {
    if (!owner) return;
#pragma unroll
    for (int c = 0; c < CPL; ++c)
      if (coil + c < a.coils) csr_store<OM, ACC>(a, out_row, coil + c, sum.v[c].x, sum.v[c].y);
    return;
  }
  // one chunk of the rows: publish, count, and the last arrival adds the
  // chunks' slots in chunk order
  const rsrc_t slots = make_rsrc(a.partials, uint64_t{1} << 32);
  if (owner) {
#pragma unroll
    for (int c = 0; c < CPL; ++c)
      if (coil + c < a.coils)
        __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(u32x2_t, sum.v[c]), slots,
                                              (it.slot0 + it.chunk * it.n_rows + r) * (kMaxCoils * 8) +
                                                  (coil + c) * 8,
                                              0, kCpolDevice);
  }
  __builtin_amdgcn_s_waitcnt(0);  // the wave's slot stores acknowledged
  __syncthreads();
  if (tid == 0)
    last_arrival = __hip_atomic_fetch_add(a.counters + it.counter, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) + 1 ==
                           it.n_chunks * gridDim.y
                       ? 1u
                       : 0u;
  __syncthreads();
  if (!last_arrival) return;
  asm volatile("" ::: "memory");
  if (tid == 0) __hip_atomic_store(a.counters + it.counter, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  for (uint32_t o = tid; o < it.n_rows * kMaxCoils; o += 256) {
    const uint32_t row = o / kMaxCoils, c = o % kMaxCoils;
    if (c >= a.coils) continue;
    float2_t v = float2_t{0.f, 0.f};
    for (uint32_t q0 = 0; q0 < it.n_chunks; q0 += kSlotBatch) {
      float2_t p[kSlotBatch];
#pragma unroll
      for (uint32_t j = 0; j < kSlotBatch; ++j)
        p[j] = __builtin_bit_cast(
            float2_t,
            __builtin_amdgcn_raw_buffer_load_b64(
                slots, (it.slot0 + min(q0 + j, it.n_chunks - 1u) * it.n_rows + row) * (kMaxCoils * 8) + c * 8, 0,
                kCpolDevice));
#pragma unroll
      for (uint32_t j = 0; j < kSlotBatch; ++j)
        if (q0 + j < it.n_chunks) v += p[j];
    }
    csr_store<OM, ACC>(a, glb(a.row_ids)[it.row0 + row], c, v.x, v.y);
  }
}

// hi = RN16(v), res = RN16(v - hi), v = in * scale; in float2 [coil][rows];
// output panel blocks [block][row][16].  Memory bound: a block converts 64
// rows of one coil block, each wave reads 64 consecutive rows of one coil (512
// contiguous bytes), the tile is turned through LDS and each thread writes
// four channels of a row, 8 bytes a panel (a thread per half word: 206 K rows
// of 8 coils 11.3 -> 5.5 us).
constexpr uint32_t kSplitRows = 64;

__global__ __launch_bounds__(256) void split_panel_kernel(const float2* __restrict__ in, uint32_t rows,
                                                          uint32_t coils, float scale, _Float16* __restrict__ hi,
                                                          _Float16* __restrict__ res) {
  typedef _Float16 __attribute__((ext_vector_type(4))) half4_t;
  typedef half4_t __attribute__((aligned(2))) out4_t;  // (the panels need no alignment of their own)
  // [re, im][coil][row]; the pitch keeps the 8 rows x 4 channels that 32 lanes read on banks of their own
  __shared__ float tile[kN][kSplitRows + 2];
  const uint32_t row0 = blockIdx.x * kSplitRows, b = blockIdx.y;
#pragma unroll
  for (uint32_t k = 0; k < kSplitRows * kCoilsPerBlock / 256; ++k) {
    const uint32_t i = threadIdx.x + 256 * k;
    const uint32_t c = i / kSplitRows, r = i % kSplitRows;
    const uint32_t coil = b * kCoilsPerBlock + c, row = row0 + r;
    float2 v = make_float2(0.f, 0.f);
    if (coil < coils && row < rows) {
      const float2 x = in[static_cast<size_t>(coil) * rows + row];
      v = make_float2(x.x * scale, x.y * scale);
    }
    tile[c][r] = v.x;
    tile[c + 8][r] = v.y;
  }
  __syncthreads();
  const uint32_t r = threadIdx.x / 4, n0 = threadIdx.x % 4 * 4, row = row0 + r;
  if (row >= rows) return;
  half4_t h, l;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    float v = tile[n0 + i][r];
    asm volatile("" : "+v"(v));  // split the FP32 value (see split_word)
    h[i] = static_cast<_Float16>(v);
    l[i] = static_cast<_Float16>(v - static_cast<float>(h[i]));
  }
  const size_t e = (static_cast<size_t>(b) * rows + row) * kN + n0;
  *reinterpret_cast<out4_t*>(hi + e) = h;
  *reinterpret_cast<out4_t*>(res + e) = l;
}

// Interleaved variant for the plan: one uint32 = hi | res << 16 per channel,
// FP16 (RN) or, with BF16, bfloat16 (RNE) halves; the same tiles, and the
// panel rows go out as 64 contiguous bytes per row.

template <bool BF16>
__global__ __launch_bounds__(256) void split_panel_il_kernel(const float2* __restrict__ in, uint32_t rows,
                                                             uint32_t coils, float scale, uint32_t row_words,
                                                             uint64_t block_words, uint32_t* __restrict__ out) {
  __shared__ float2 tile[kSplitRows][kCoilsPerBlock + 1];
  const uint32_t row0 = blockIdx.x * kSplitRows, b = blockIdx.y;
#pragma unroll
  for (uint32_t k = 0; k < kSplitRows * kCoilsPerBlock / 256; ++k) {
    const uint32_t i = threadIdx.x + 256 * k;
    const uint32_t c = i / kSplitRows, r = i % kSplitRows;
    const uint32_t coil = b * kCoilsPerBlock + c, row = row0 + r;
    tile[r][c] = (coil < coils && row < rows) ? in[static_cast<size_t>(coil) * rows + row] : make_float2(0.f, 0.f);
  }
  __syncthreads();
#pragma unroll
  for (uint32_t k = 0; k < kSplitRows * kN / 256; ++k) {
    const uint32_t w = threadIdx.x + 256 * k;
    const uint32_t r = w / kN, n = w % kN, row = row0 + r;
    if (row >= rows) continue;
    const float2 x = tile[r][n & 7];
    out[b * block_words + static_cast<size_t>(row) * row_words + n] = split_word<BF16>((n < 8 ? x.x : x.y) * scale);
  }
}

// Materialized data consistency: out = split((pred - scale * y) * w) with
// pred float2 [rows][coils] (a row-major interpolation output) and y read
// through the same strides as the fused epilogue.  One thread per panel word.
template <bool BF16>
__global__ __launch_bounds__(256) void dc_residual_kernel(const float* __restrict__ pred, const float* __restrict__ y,
                                                          const float* __restrict__ density, uint32_t rows,
                                                          uint32_t coils, uint32_t blocks, float scale,
                                                          uint32_t row_stride, uint32_t coil_stride,
                                                          uint32_t* __restrict__ out) {
  const uint64_t gtid = static_cast<uint64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  const uint64_t total = static_cast<uint64_t>(blocks) * rows * kN;
  if (gtid >= total) return;
  const int n = static_cast<int>(gtid & 15);
  const uint64_t br = gtid >> 4;
  const uint32_t row = static_cast<uint32_t>(br % rows);
  const uint32_t b = static_cast<uint32_t>(br / rows);
  const uint32_t coil = b * kCoilsPerBlock + (n & 7);
  const int part = n >> 3;
  float p = 0.0f, m = 0.0f;
  if (coil < coils) {
    p = pred[(static_cast<size_t>(row) * coils + coil) * 2 + part];
    m = y[static_cast<size_t>(row) * row_stride + static_cast<size_t>(coil) * coil_stride + part];
  }
  const float w = density ? density[row] : 1.0f;
  out[gtid] = split_word<BF16>(dc_residual(p, m, scale, w));
}

// ------------------------------------------------------------- dispatch

// Pipeline depths the autotuner may pick besides PipeDepth: for the launches
// plans and batches make with interleaved panels (forward into a split
// panel, adjoint into float2 rows), one wave per entry: 1 or 3 tiles ahead
// for one coil block, 2 for two.
template <int KIND, int NB, int IL, int OM, bool CONJ, bool ACC, int WB>
struct AltDepths {
  static constexpr bool kPlanLaunch = (IL != kHalves) && KIND != kDenseSplit && !ACC && WB == 1 &&
                                      ((OM == kOutRowMajor && CONJ) ||
                                       ((OM == kOutSplit16IL || OM == kOutSplitBF16IL) && !CONJ));
};

template <int KIND, int NB, int IL, int OM, bool CONJ, bool ACC, int WB>
static void launch_both(const InterpArgs& a, hipStream_t s) {
  const uint32_t blocks = a.n_chunks + a.n_items;
  if (!blocks) return;
  using Alt = AltDepths<KIND, NB, IL, OM, CONJ, ACC, WB>;
  if constexpr (Alt::kPlanLaunch) {
    if constexpr (NB == 1) {
      if (a.depth == 1) {
        hipLaunchKernelGGL((interp_tiles_depth_kernel<KIND, NB, IL, OM, CONJ, ACC, WB, 1>), dim3(blocks),
                           dim3(64 * WB), 0, s, a);
        return;
      }
      if (a.depth == 3) {
        hipLaunchKernelGGL((interp_tiles_depth_kernel<KIND, NB, IL, OM, CONJ, ACC, WB, 3>), dim3(blocks),
                           dim3(64 * WB), 0, s, a);
        return;
      }
    } else {
      if (a.depth == 2) {
        hipLaunchKernelGGL((interp_tiles_depth_kernel<KIND, NB, IL, OM, CONJ, ACC, WB, 2>), dim3(blocks),
                           dim3(64 * WB), 0, s, a);
        return;
      }
    }
  }
  hipLaunchKernelGGL((interp_tiles_kernel<KIND, NB, IL, OM, CONJ, ACC, WB>), dim3(blocks), dim3(64 * WB), 0, s, a);
}

template <int KIND, int NB, int IL, int OM, int WB = 1>
static void launch_tiles_om(const InterpArgs& a, bool conj, bool acc, hipStream_t s) {
  constexpr bool kAccOk = OM != kOutSplit16IL && OM != kOutSplitBF16IL;
  if (conj) {
    if (kAccOk && acc) launch_both<KIND, NB, IL, OM, true, kAccOk, WB>(a, s);
    else launch_both<KIND, NB, IL, OM, true, false, WB>(a, s);
  } else {
    if (kAccOk && acc) launch_both<KIND, NB, IL, OM, false, kAccOk, WB>(a, s);
    else launch_both<KIND, NB, IL, OM, false, false, WB>(a, s);
  }
}

// Interleaved panels (plan-internal) pair with FP32 or interleaved split
// output; separate panels with FP32 or separate split output (checked by
// launch_interp).  WB = 2: two coil blocks, one wave each (NB = 1).
template <int KIND, int NB, int IL, int WB = 1>
static void launch_tiles_nb(const InterpArgs& a, int om, bool conj, bool acc, hipStream_t s) {
  if constexpr (IL != kHalves) {
    if (om == kOutCoilMajor) launch_tiles_om<KIND, NB, IL, kOutCoilMajor, WB>(a, conj, acc, s);
    else if (om == kOutRowMajor) launch_tiles_om<KIND, NB, IL, kOutRowMajor, WB>(a, conj, acc, s);
    else if (KIND == kSparseSplitBF16) launch_tiles_om<KIND, NB, IL, kOutSplitBF16IL, WB>(a, conj, false, s);
    else launch_tiles_om<KIND, NB, IL, kOutSplit16IL, WB>(a, conj, false, s);
  } else {
    if (om == kOutCoilMajor) launch_tiles_om<KIND, NB, IL, kOutCoilMajor>(a, conj, acc, s);
    else launch_tiles_om<KIND, NB, IL, kOutRowMajor>(a, conj, acc, s);
  }
}

// Line-row panels (plans and batches of 9..16 coils), one wave for both coil
// blocks: the launches those make (forward into a split panel or, for a plan's
// forward operator, coil-major float2; adjoint into float2 rows).
template <int KIND>
static int launch_lines(const InterpArgs& a, int om, bool conj, bool acc, hipStream_t s) {
  constexpr int kSplitOut = KIND == kSparseSplitBF16 ? kOutSplitBF16IL : kOutSplit16IL;
  if (acc) return fail(TSN_ERR_ARGUMENT, "line-row panels do not accumulate");
  if (om == kOutSplit16IL && !conj) launch_both<KIND, 2, kLines, kSplitOut, false, false, 1>(a, s);
  else if (om == kOutRowMajor && conj) launch_both<KIND, 2, kLines, kOutRowMajor, true, false, 1>(a, s);
  else if (om == kOutCoilMajor && !conj) launch_both<KIND, 2, kLines, kOutCoilMajor, false, false, 1>(a, s);
  else return fail(TSN_ERR_ARGUMENT, "line-row panels do not write output mode %d here", om);
  return TSN_OK;
}

// Two coil blocks of interleaved panels: one wave for both (coil_waves 1) or
// one wave per block (coil_waves 2, either panel layout).
template <int KIND>
static int launch_tiles(const InterpArgs& a, int panels, int om, bool conj, bool acc, uint32_t coil_waves,
                        hipStream_t s) {
  const bool two = a.coils > kCoilsPerBlock;
  if (panels == kHalves) {
    if constexpr (KIND != kSparseSplitBF16) {  // BF16 tiles take interleaved panels (checked by launch_interp)
      if (two) launch_tiles_nb<KIND, 2, kHalves>(a, om, conj, acc, s);
      else launch_tiles_nb<KIND, 1, kHalves>(a, om, conj, acc, s);
    }
    return TSN_OK;
  }
  if (!two) launch_tiles_nb<KIND, 1, kBlocks>(a, om, conj, acc, s);
  else if (coil_waves == 2) launch_tiles_nb<KIND, 1, kBlocks, 2>(a, om, conj, acc, s);
  else if (panels == kLines) return launch_lines<KIND>(a, om, conj, acc, s);
  else launch_tiles_nb<KIND, 2, kBlocks>(a, om, conj, acc, s);
  return TSN_OK;
}

static int launch_interp_impl(const tsn_direction* d, int kind, const void* hi, const void* res, uint32_t coils,
                              int out_mode, bool conj, bool accumulate, float scale, float* out_f32,
                              hipStream_t stream, int panels,
                              uint32_t* out_il, const DcTerms* dc, const ChunkScratch* scratch) {
  const bool interleaved = panels != kHalves;
  if (!d || d->csr) return fail(TSN_ERR_ARGUMENT, "interpolation needs a packed (non-CSR) direction");
  if (coils == 0 || coils > static_cast<uint32_t>(kMaxCoils))
    return fail(TSN_ERR_ARGUMENT, "coils must be in 1..16 (got %u)", coils);
  if (!hi || (!interleaved && kind != kSparseHi && !res))
    return fail(TSN_ERR_ARGUMENT, "missing input panel");
  const bool block_rows = out_mode == kOutBlockRows;
  if (block_rows) out_mode = kOutRowMajor;
  const bool split_out = out_mode == kOutSplit16IL;
  if (split_out ? !out_il : !out_f32)
    return fail(TSN_ERR_ARGUMENT, "missing output");
  if (split_out && !interleaved)
    return fail(TSN_ERR_ARGUMENT, "output mode %d does not match the panel layout", out_mode);
  if (kind == kDenseSplit && !d->tile_dense)
    return fail(TSN_ERR_ARGUMENT, "direction has no dense-control tiles");
  if ((kind == kSparseSplitBF16) != (d->values == TSN_VALUES_BF16))
    return fail(TSN_ERR_ARGUMENT, "tile value format of the direction does not match the interpolation variant");
  if (kind == kSparseSplitBF16 && !interleaved)
    return fail(TSN_ERR_ARGUMENT, "BF16 tiles take an interleaved split panel");
  const bool lines = panels == kLines && coils > static_cast<uint32_t>(kCoilsPerBlock);
  if (lines && d->h.n_cols > kMaxLineCols)
    return fail(TSN_ERR_ARGUMENT, "line-row panels hold at most %u columns (got %u)", kMaxLineCols, d->h.n_cols);
  InterpArgs a{};
  const TileSchedule& schedule = lines ? d->line_rows : d->block_rows;
  a.items = schedule.items;
  a.n_items = schedule.n_items;
  a.chunks = d->chunks;
  a.n_chunks = d->n_chunks;
  a.order = schedule.order;
  a.partials = scratch ? scratch->partials : d->partials;
  a.counters = scratch ? scratch->counters : d->counters;
  if (d->n_chunks && (!a.partials || !a.counters)) return fail(TSN_ERR_ARGUMENT, "missing chunk scratch");
  a.group_rows = d->group_rows;
  a.group_offsets = d->group_offsets;
  a.tile_cols = d->tile_cols;
  a.n_tiles = d->h.tiles;
  a.n_groups = d->h.groups;
  a.tile_a = d->tile_a;
  a.tile_idx = d->tile_idx;
  a.tile_dense = d->tile_dense;
  a.panel_hi = static_cast<const _Float16*>(hi);
  a.panel_res = static_cast<const _Float16*>(res);
  a.panel_il = static_cast<const uint32_t*>(hi);
  a.coils = coils;
  a.n_out = d->h.output_size;
  a.panel_stride = static_cast<uint64_t>(d->h.n_cols) * kN;
  a.lines = lines ? 1u : 0u;
  a.scale = scale;
  a.out_f32 = out_f32;
  a.out_il = out_il;
  a.out_rs = block_rows ? kCoilsPerBlock : coils;
  a.out_bs = block_rows ? static_cast<uint64_t>(a.n_out) * kCoilsPerBlock : kCoilsPerBlock;
  if (dc) {
    a.dc_meas = dc->y;
    a.dc_density = dc->density;
    a.dc_scale = dc->scale;
    a.dc_row_stride = dc->row_stride;
    a.dc_coil_stride = dc->coil_stride;
  }
  a.depth = schedule.pipe_depth;
  const uint32_t cw = schedule.coil_waves;
  if (kind == kSparseSplit) TSN_CHECK(launch_tiles<kSparseSplit>(a, panels, out_mode, conj, accumulate, cw, stream));
  else if (kind == kDenseSplit)
    TSN_CHECK(launch_tiles<kDenseSplit>(a, panels, out_mode, conj, accumulate, cw, stream));
  else if (kind == kSparseSplitBF16)
    TSN_CHECK(launch_tiles<kSparseSplitBF16>(a, panels, out_mode, conj, accumulate, cw, stream));
  else TSN_CHECK(launch_tiles<kSparseHi>(a, panels, out_mode, conj, accumulate, cw, stream));
  TSN_HIP(hipGetLastError());
  return TSN_OK;
}

// Internal entry used by the plan and the C ABI.  All pointers are device
// pointers sized by the caller; panels hold ceil(coils/8) blocks.
int launch_interp(const tsn_direction* d, int kind, const void* hi, const void* res, uint32_t coils,
                  int out_mode, bool conj, bool accumulate, float scale, float* out_f32,
                  hipStream_t stream, int panels, uint32_t* out_il, const ChunkScratch* scratch) {
  return launch_interp_impl(d, kind, hi, res, coils, out_mode, conj, accumulate, scale, out_f32, stream, panels,
                            out_il, nullptr, scratch);
}

int launch_interp_dc(const tsn_direction* d, int kind, const uint32_t* panel, uint32_t coils, float scale,
                     const DcTerms& dc, uint32_t* out_il, hipStream_t s, const ChunkScratch* scratch, int panels) {
  if (!dc.y) return fail(TSN_ERR_ARGUMENT, "missing measurements");
  return launch_interp_impl(d, kind, panel, nullptr, coils, kOutSplit16IL, false, false, scale, nullptr, s, panels,
                            out_il, &dc, scratch);
}

int launch_dc_residual(const float2* pred, uint32_t rows, uint32_t coils, const DcTerms& dc, bool bf16,
                       uint32_t* out_il, hipStream_t s) {
  if (!pred || !dc.y || !out_il) return fail(TSN_ERR_ARGUMENT, "null argument");
  if (coils == 0 || coils > static_cast<uint32_t>(kMaxCoils)) return fail(TSN_ERR_ARGUMENT, "coils must be in 1..16");
  const uint32_t blocks = div_up(coils, kCoilsPerBlock);
  const uint64_t total = static_cast<uint64_t>(blocks) * rows * kN;
  if (total == 0) return TSN_OK;
  const dim3 grid(static_cast<uint32_t>(div_up(total, 256)));
  const float* p = reinterpret_cast<const float*>(pred);
  if (bf16)
    hipLaunchKernelGGL(dc_residual_kernel<true>, grid, dim3(256), 0, s, p, dc.y, dc.density, rows, coils, blocks,
                       dc.scale, dc.row_stride, dc.coil_stride, out_il);
  else
    hipLaunchKernelGGL(dc_residual_kernel<false>, grid, dim3(256), 0, s, p, dc.y, dc.density, rows, coils, blocks,
                       dc.scale, dc.row_stride, dc.coil_stride, out_il);
  TSN_HIP(hipGetLastError());
  return TSN_OK;
}

// FP32 rows float2 [rows][coils] in place: v <- (v - scale * y) * w.
__global__ __launch_bounds__(256) void dc_residual_rows_kernel(float* __restrict__ io, const float* __restrict__ y,
                                                               const float* __restrict__ density, uint32_t rows,
                                                               uint32_t coils, float scale, uint32_t row_stride,
                                                               uint32_t coil_stride) {
  const uint64_t gtid = static_cast<uint64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  const uint64_t per_row = 2ull * coils;
  if (gtid >= per_row * rows) return;
  const uint32_t row = static_cast<uint32_t>(gtid / per_row);
  const uint32_t rem = static_cast<uint32_t>(gtid % per_row);
  const uint32_t coil = rem >> 1, part = rem & 1u;
  const float w = density ? density[row] : 1.0f;
  io[gtid] = dc_residual(io[gtid], y[static_cast<size_t>(row) * row_stride + static_cast<size_t>(coil) * coil_stride + part],
                         scale, w);
}

int launch_dc_residual_rows(float2* rows_io, uint32_t rows, uint32_t coils, const DcTerms& dc, hipStream_t s) {
  if (!rows_io || !dc.y) return fail(TSN_ERR_ARGUMENT, "null argument");
  const uint64_t total = 2ull * coils * rows;
  if (total == 0) return TSN_OK;
  hipLaunchKernelGGL(dc_residual_rows_kernel, dim3(static_cast<uint32_t>(div_up(total, 256))), dim3(256), 0, s,
                     reinterpret_cast<float*>(rows_io), dc.y, dc.density, rows, coils, dc.scale, dc.row_stride,
                     dc.coil_stride);
  TSN_HIP(hipGetLastError());
  return TSN_OK;
}

template <int CPL, int SUMS, int OM>
static void launch_csr_om(const CsrArgs& a, bool conj, bool acc, hipStream_t s) {
#define TSN_CSR(C, A)                                                                                              \
  hipLaunchKernelGGL((interp_csr_kernel<CPL, SUMS, OM, C, A>), dim3(a.n_blocks, div_up(a.coils, 4u * CPL)), dim3(256), \
                     0, s, a)
  if (conj) {
    if (acc) TSN_CSR(true, true); else TSN_CSR(true, false);
  } else {
    if (acc) TSN_CSR(false, true); else TSN_CSR(false, false);
  }
#undef TSN_CSR
}

template <int CPL, int SUMS>
static void launch_csr_cpl(const CsrArgs& a, int om, bool conj, bool acc, hipStream_t s) {
  if (om == kOutCoilMajor) launch_csr_om<CPL, SUMS, kOutCoilMajor>(a, conj, acc, s);
  else launch_csr_om<CPL, SUMS, kOutRowMajor>(a, conj, acc, s);
}

int launch_interp_csr(const tsn_direction* d, const float2* in, uint32_t coils, int out_mode,
                      bool conj, bool accumulate, float scale, float2* out, hipStream_t stream,
                      const ChunkScratch* scratch, bool out_prezeroed) {
  if (!d || !d->csr) return fail(TSN_ERR_ARGUMENT, "FP32 interpolation needs a CSR direction");
  if (coils == 0 || coils > static_cast<uint32_t>(kMaxCoils))
    return fail(TSN_ERR_ARGUMENT, "coils must be in 1..16 (got %u)", coils);
  if (!in || !out) return fail(TSN_ERR_ARGUMENT, "null input/output");
  if (out_mode != kOutCoilMajor && out_mode != kOutRowMajor)
    return fail(TSN_ERR_ARGUMENT, "unsupported FP32 output layout %d", out_mode);
  // gathers address input rows with 32-bit byte offsets
  if (static_cast<uint64_t>(d->h.n_cols) * coils * 8 >= (uint64_t{1} << 32))
    return fail(TSN_ERR_ARGUMENT, "FP32 input of %u rows x %u coils exceeds 4 GiB", d->h.n_cols, coils);
  CsrArgs a{};
  a.blocks = d->csr_blocks;
  a.n_blocks = d->n_csr_blocks;
  a.n_active = d->n_csr_active_blocks;
  a.row_ids = d->row_ids;
  a.cols = d->csr_cols;
  a.vals = d->vals;
  a.idx = d->csr_idx;
  a.rounds = d->csr_rounds;
  a.partials = reinterpret_cast<float2*>(scratch ? scratch->partials : d->partials);
  a.counters = scratch ? scratch->counters : d->counters;
  if (d->n_slots && (!a.partials || !a.counters)) return fail(TSN_ERR_ARGUMENT, "missing chunk scratch");
  a.in = in;
  a.n_cols = d->h.n_cols;
  a.coils = coils;
  a.n_out = d->h.output_size;
  a.scale = scale;
  a.out = out;
  a.skip_empty = out_prezeroed ? 1u : 0u;
  if (out_prezeroed || accumulate) a.n_blocks = a.n_active;  // the trailing empty runs write nothing
  if (a.n_blocks == 0) return TSN_OK;
  const bool few = a.n_active <= kCsrFewBlocks;
  if (coils <= 4) launch_csr_cpl<1, 4>(a, out_mode, conj, accumulate, stream);
  else if (coils <= 8 && few) launch_csr_cpl<1, 2>(a, out_mode, conj, accumulate, stream);
  else if (coils <= 8) launch_csr_cpl<2, 2>(a, out_mode, conj, accumulate, stream);
  else if (few) launch_csr_cpl<1, 1>(a, out_mode, conj, accumulate, stream);
  else launch_csr_cpl<4, 1>(a, out_mode, conj, accumulate, stream);
  TSN_HIP(hipGetLastError());
  return TSN_OK;
}

int launch_split_panel(const float2* in, uint32_t rows, uint32_t coils, float scale, _Float16* hi,
                       _Float16* res, hipStream_t stream) {
  if (!in || !hi || !res || rows == 0) return fail(TSN_ERR_ARGUMENT, "bad split arguments");
  if (coils == 0 || coils > static_cast<uint32_t>(kMaxCoils))
    return fail(TSN_ERR_ARGUMENT, "coils must be in 1..16 (got %u)", coils);
  const uint32_t blocks = div_up(coils, kCoilsPerBlock);
  hipLaunchKernelGGL(split_panel_kernel, dim3(div_up(rows, kSplitRows), blocks), dim3(256), 0, stream, in, rows,
                     coils, scale, hi, res);
  TSN_HIP(hipGetLastError());
  return TSN_OK;
}

int launch_split_panel_il(const float2* in, uint32_t rows, uint32_t coils, float scale, uint32_t* out,
                          hipStream_t stream, int values, bool lines) {
  if (!in || !out || rows == 0) return fail(TSN_ERR_ARGUMENT, "bad split arguments");
  if (coils == 0 || coils > static_cast<uint32_t>(kMaxCoils))
    return fail(TSN_ERR_ARGUMENT, "coils must be in 1..16 (got %u)", coils);
  if (values != TSN_VALUES_FP16 && values != TSN_VALUES_BF16)
    return fail(TSN_ERR_ARGUMENT, "unknown value format %d", values);
  const uint32_t blocks = div_up(coils, kCoilsPerBlock);
  const dim3 grid(div_up(rows, kSplitRows), blocks);
  lines = lines && blocks == 2;
  const uint32_t rw = lines ? 2 * kN : kN;
  const uint64_t bw = lines ? static_cast<uint64_t>(kN) : static_cast<uint64_t>(rows) * kN;
  if (values == TSN_VALUES_BF16)
    hipLaunchKernelGGL(split_panel_il_kernel<true>, grid, dim3(256), 0, stream, in, rows, coils, scale, rw, bw, out);
  else
    hipLaunchKernelGGL(split_panel_il_kernel<false>, grid, dim3(256), 0, stream, in, rows, coils, scale, rw, bw, out);
  TSN_HIP(hipGetLastError());
  return TSN_OK;
}

// ------------------------------------------------------------- upload

template <typename T>
static int device_copy(const T* host, size_t count, T** out, size_t* bytes) {
  *out = nullptr;
  if (count == 0) return TSN_OK;
  TSN_HIP(hipMalloc(reinterpret_cast<void**>(out), count * sizeof(T)));
  TSN_HIP(hipMemcpy(*out, host, count * sizeof(T), hipMemcpyHostToDevice));
  *bytes += count * sizeof(T);
  return TSN_OK;
}

static void release(tsn_direction* d) {
  if (!d) return;
  void* ptrs[] = {d->group_offsets, d->group_rows, d->tile_cols, d->tile_a, d->tile_idx,
                  d->tile_dense, d->chunks, d->partials, d->counters, d->csr_data};
  for (void* p : ptrs)
    if (p) (void)hipFree(p);
  for (void* p : d->schedules) (void)hipFree(p);
  delete d;
}

// Longest entries first within each XCD's contiguous range of a launch order
// (block b runs on XCD b mod 8 and takes entry xcd_remap(b)), in windows of
// kLptWindow entries, about what one XCD holds resident: the waves dispatched
// last are then the shortest.  The sort is stable, so entries of equal length
// keep pack order.  Measured at 205,824 samples / 512^2 grid / 8 coils: G 18.5
// -> 17.9 us, G^T 19.7 -> 18.3 us.
constexpr uint32_t kLptWindow = 512;

template <typename F>
static void lpt_order(std::vector<uint32_t>& order, F tiles_of) {
  const uint32_t nb = static_cast<uint32_t>(order.size());
  for (uint32_t x = 0; x < 8; ++x) {
    const uint32_t lo = xcd_remap(x, nb), hi = x == 7 ? nb : xcd_remap(x + 1, nb);
    for (uint32_t b = lo; b < hi; b += kLptWindow)
      std::stable_sort(order.begin() + b, order.begin() + std::min(hi, b + kLptWindow),
                       [&](uint32_t p, uint32_t q) { return tiles_of(p) > tiles_of(q); });
  }
}

// Work schedule of a packed direction: the groups of at most
// kSplitAboveTiles tiles are cut, in pack order, into contiguous runs of whole
// groups holding at most unit_tiles tiles (a single group is never cut); an
// empty group is a unit of its own (zero epilogue).  Longer groups are
// chunks, fixed at upload.  unit_tiles 0 picks the default: the regular tiles
// over 12 waves per CU, clamped to 4..14 tiles.  The launch order then runs
// the longest entries of each XCD first (lpt_order).  Measured at 205,824
// samples / 512^2 grid / 8 coils: G 17.9 us with 14-tile units against 18.0
// (16) and 18.1 (12); G^T 18.3 us against 18.4 (16) and 20.1 (12); smaller
// units start more waves than the CUs hold at once.
static int schedule_units(tsn_direction* d, uint32_t unit_tiles, std::initializer_list<TileSchedule*> into) {
  const std::vector<uint32_t>& off = d->host_offsets;
  const uint32_t groups = d->h.groups;
  uint64_t regular_tiles = 0;
  for (uint32_t g = 0; g < groups; ++g) {
    const uint32_t n = off[g + 1] - off[g];
    if (n <= static_cast<uint32_t>(kSplitAboveTiles)) regular_tiles += n;
  }
  int64_t target = unit_tiles;
  if (target == 0) {
    int cus = 0;
    if (hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, d->device) != hipSuccess || cus <= 0)
      cus = 256;
    const uint64_t waves = static_cast<uint64_t>(cus) * 12;
    target = std::clamp<int64_t>(static_cast<int64_t>((regular_tiles + waves - 1) / waves), 4, 14);
  }
  // a unit's column words are staged in the wave's LDS slice: at most 16 tiles
  target = std::min<int64_t>(target, kSplitAboveTiles);
  std::vector<WorkItem> items;
  std::vector<uint32_t> order;
  uint32_t chunk = 0;  // chunks are numbered in group order (long_chunks)
  std::vector<int32_t> chunk_tiles;
  WorkItem cur{-1, -1, 0, 0};
  auto flush = [&]() {
    if (cur.group >= 0) {
      order.push_back(static_cast<uint32_t>(items.size()));
      items.push_back(cur);
    }
    cur = {-1, -1, 0, 0};
  };
  for (uint32_t g = 0; g < groups; ++g) {
    const int32_t b = static_cast<int32_t>(off[g]);
    const int32_t e = static_cast<int32_t>(off[g + 1]);
    const int32_t gi = static_cast<int32_t>(g);
    if (e - b > kSplitAboveTiles) {  // a chunked long group
      flush();
      const uint32_t n = static_cast<uint32_t>(e - b + kSplitAboveTiles - 1) / kSplitAboveTiles;
      for (uint32_t c = 0; c < n; ++c) {
        order.push_back(kChunkTag | chunk++);
        // a chunk ranks as if longer by its finishing chain, so chunks start first
        chunk_tiles.push_back(static_cast<int32_t>(chunk_begin(b, e, n, c + 1) - chunk_begin(b, e, n, c)) +
                              kChunkFinishTiles);
      }
      continue;
    }
    if (e == b) {
      flush();
      order.push_back(static_cast<uint32_t>(items.size()));
      items.push_back({gi, gi + 1, b, e});
      continue;
    }
    if (cur.group >= 0 && cur.tile_end - cur.tile_begin + (e - b) > target) flush();
    if (cur.group < 0) {
      cur = {gi, gi + 1, b, e};
    } else {
      cur.group_end = gi + 1;
      cur.tile_end = e;
    }
  }
  flush();
  lpt_order(order, [&](uint32_t e) {
    return (e & kChunkTag) ? chunk_tiles[e & ~kChunkTag] : items[e].tile_end - items[e].tile_begin;
  });
  WorkItem* new_items = nullptr;
  uint32_t* new_order = nullptr;
  size_t bytes = 0;
  int rc = device_copy(items.data(), items.size(), &new_items, &bytes);
  if (rc == TSN_OK) rc = device_copy(order.data(), order.size(), &new_order, &bytes);
  if (rc != TSN_OK) {
    if (new_items) (void)hipFree(new_items);
    return rc;
  }
  // Earlier schedules stay allocated until the direction is freed: a captured
  // graph may still hold their addresses in its kernel arguments.
  for (void* p : {static_cast<void*>(new_items), static_cast<void*>(new_order)})
    if (p) d->schedules.push_back(p);
  for (TileSchedule* to : into) {
    to->items = new_items;
    to->order = new_order;
    to->n_items = static_cast<uint32_t>(items.size());
    to->unit_tiles = static_cast<uint32_t>(target);
    to->host_items = items;
    to->host_order = order;
  }
  d->bytes += bytes;
  return TSN_OK;
}

}  // namespace tsn

namespace {

// The entries of an FP32 direction's rows, ascending columns: G as the matrix
// holds them, or its transpose.  (Plain pointers: loops copy a view, so that
// their stores cannot alias it.)
struct CsrForward {
  uint32_t width;
  const int32_t* cols;
  const float *re, *im;
  uint32_t begin(uint32_t t) const { return t * width; }
  uint32_t column(uint32_t e) const { return static_cast<uint32_t>(cols[e]); }
  float2 value(uint32_t e) const { return make_float2(re[e], im[e]); }
};
struct CsrTranspose {
  struct Entry {
    uint32_t sample, at;  // column, and the entry's place in the matrix
  };
  const uint32_t* ptr;
  const Entry* entries;
  const float *re, *im;
  uint32_t begin(uint32_t t) const { return ptr[t]; }
  uint32_t column(uint32_t e) const { return entries[e].sample; }
  float2 value(uint32_t e) const { return make_float2(re[entries[e].at], im[entries[e].at]); }
};

// One lane quad of an FP32 block: entries base + stride i, i < count, whose
// columns' numbers in uniq are at local + stride i of the block's list.
struct CsrQuad {
  uint32_t base, stride, count, local;
};

// Builds the blocks of one range of a direction's rows (csr_build).
template <typename View>
struct CsrBuilder {
  // the group that last named a column, and its number there
  struct Slot {
    uint32_t group, place;
  };
  const View view;
  const std::vector<int32_t>& rows;
  uint32_t short_rows, long_rows;  // rows of a block of either kind, at most
  Slot* slots;                     // [n_cols]
  uint32_t group = 1;
  tsn::CsrHost h;
  // the group's entries and their columns' numbers, its columns as first named
  // (one place more: name() writes before it knows), their place in ascending order
  static constexpr uint32_t kEntries = 65 * tsn::kCsrShortEntries;
  static_assert(16 * tsn::kCsrChunkEntries <= kEntries, "entries of a group of long rows");
  uint32_t n_local = 0, n_uniq = 0;
  std::vector<uint16_t> local = std::vector<uint16_t>(kEntries), rank = std::vector<uint16_t>(kEntries);
  std::vector<uint32_t> uniq = std::vector<uint32_t>(kEntries + 1);

  uint32_t length(uint32_t t) const { return view.begin(t + 1) - view.begin(t); }

  // Names entries [b, e) in the group; where their first is in local.  (Without
  // a branch: whether a column is new is a coin toss.)
  uint32_t name(uint32_t b, uint32_t e) {
    const View v = view;
    const uint32_t at = n_local, g = group;
    Slot* const table = slots;
    uint16_t* to = local.data() + at;
    uint32_t* const named = uniq.data();
    uint32_t n = n_uniq;
    for (uint32_t k = b; k < e; ++k) {
      const uint32_t c = v.column(k);
      const Slot s = table[c];
      const bool fresh = s.group != g;
      const uint32_t place = fresh ? n : s.place;
      table[c] = {g, place};
      named[n] = c;
      n += fresh;
      *to++ = static_cast<uint16_t>(place);
    }
    n_uniq = n;
    n_local = at + (e - b);
    return at;
  }

  // One block of the quads (16 to a wave), whose entries name the columns uniq.
  void emit(tsn::CsrBlock b, const CsrQuad* quads, uint32_t n_quads) {
    b.n_rounds = tsn::div_up(n_uniq, tsn::kCsrCols);
    b.round0 = static_cast<uint32_t>(h.rounds.size());
    if (b.n_rounds == 1) b.first = one_round(quads, n_quads);
    else if (b.n_rounds > 1) b.first = rounds(b.n_rounds, quads, n_quads);
    h.blocks.push_back(b);
    n_uniq = n_local = 0;
    ++group;
  }

  // The wave's n steps, entry i of a quad at step i / 4 and lane i mod 4 of it.
  struct Wave {
    float2* vals;
    uint8_t* idx;  // one byte a step
    float2& value(uint32_t q, uint32_t i) { return vals[(i / 4) * 64 + q * 4 + (i & 3u)]; }
    uint8_t& column(uint32_t q, uint32_t i) { return idx[((i / 16) * 64 + q * 4 + (i & 3u)) * 4 + (i / 4 & 3u)]; }
  };
  Wave wave(uint32_t n) {
    const size_t words = static_cast<size_t>(tsn::div_up(n, 4)) * 64;
    const Wave w{h.vals.grow(static_cast<size_t>(n) * 64), reinterpret_cast<uint8_t*>(h.idx.grow(words))};
    std::memset(w.idx, 0, words * 4);
    return w;
  }
  tsn::CsrRound round_at(uint32_t u0, uint32_t u1) {
    tsn::CsrRound rd{};
    rd.col0 = static_cast<uint32_t>(h.cols.size());
    rd.n_cols = u1 - u0;
    rd.ent0 = static_cast<uint32_t>(h.vals.size() / 64);
    rd.idx0 = static_cast<uint32_t>(h.idx.size() / 64);
    h.cols.insert(h.cols.end(), uniq.begin() + u0, uniq.begin() + u1);
    return rd;
  }

  // All columns in one round, in the order in which they were named.
  tsn::CsrRound one_round(const CsrQuad* quads, uint32_t n_quads) {
    const View v = view;
    tsn::CsrRound rd = round_at(0, n_uniq);
    for (uint32_t q0 = 0; q0 < n_quads; q0 += 16) {
      const uint32_t in_wave = std::min(n_quads - q0, 16u);
      uint32_t n = 0;
      for (uint32_t q = 0; q < in_wave; ++q) n = std::max(n, tsn::div_up(quads[q0 + q].count, 4));
      if (n == 0) continue;
      rd.steps |= n << (q0 / 2);  // byte q0 / 16
      Wave w = wave(n);
      for (uint32_t q = 0; q < 16; ++q) {
        const CsrQuad qd = q < in_wave ? quads[q0 + q] : CsrQuad{};
        const uint16_t* from = local.data() + qd.local;
        uint32_t e = qd.base, i = 0;
        auto put = [&, v, stride = qd.stride](float2* value, uint8_t* column) {
          *value = v.value(e);
          *column = static_cast<uint8_t>(*from + 1);
          e += stride;
          from += stride;
        };
        for (; i + 4 <= qd.count; i += 4)
          for (uint32_t l = 0; l < 4; ++l) put(&w.value(q, i) + l, &w.column(q, i) + 4 * l);
        for (; i < qd.count; ++i) put(&w.value(q, i), &w.column(q, i));
        for (; i < 4 * n; ++i) w.value(q, i) = make_float2(0.f, 0.f);  // (and local column 0)
      }
    }
    return rd;
  }

  // The columns in ascending order cut into n_rounds rounds: a quad's entries
  // (ascending too) follow the rounds.  The first round; the rest in h.rounds.
  tsn::CsrRound rounds(uint32_t n_rounds, const CsrQuad* quads, uint32_t n_quads) {
    const uint32_t u = n_uniq;
    std::sort(uniq.begin(), uniq.begin() + u);
    for (uint32_t i = 0; i < u; ++i) rank[slots[uniq[i]].place] = static_cast<uint16_t>(i);
    tsn::CsrRound head{};
    uint32_t at[64] = {};
    for (uint32_t k = 0; k < n_rounds; ++k) {
      const uint32_t u0 = static_cast<uint32_t>(static_cast<uint64_t>(u) * k / n_rounds);
      const uint32_t u1 = static_cast<uint32_t>(static_cast<uint64_t>(u) * (k + 1) / n_rounds);
      tsn::CsrRound rd = round_at(u0, u1);
      for (uint32_t q0 = 0; q0 < n_quads; q0 += 16) {
        const uint32_t in_wave = std::min(n_quads - q0, 16u);
        // a quad's entries at .. end of this round, from step 0 on (lane i mod 4)
        uint32_t end[16] = {}, n = 0;
        for (uint32_t q = 0; q < in_wave; ++q) {
          const CsrQuad& qd = quads[q0 + q];
          uint32_t i = at[q0 + q];
          while (i < qd.count && rank[local[qd.local + qd.stride * i]] < u1) ++i;
          end[q] = i;
          if (i > at[q0 + q]) n = std::max(n, (i - 1) / 4 - at[q0 + q] / 4 + 1);
        }
        if (n == 0) continue;
        rd.steps |= n << (q0 / 2);
        Wave w = wave(n);
        std::fill_n(w.vals, static_cast<size_t>(n) * 64, make_float2(0.f, 0.f));
        for (uint32_t q = 0; q < in_wave; ++q) {
          const CsrQuad& qd = quads[q0 + q];
          const uint32_t s0 = at[q0 + q] & ~3u;
          for (uint32_t i = at[q0 + q]; i < end[q]; ++i) {
            w.value(q, i - s0) = view.value(qd.base + qd.stride * i);
            w.column(q, i - s0) = static_cast<uint8_t>(rank[local[qd.local + qd.stride * i]] - u0 + 1);
          }
          at[q0 + q] = end[q];
        }
      }
      if (k == 0) head = rd;
      else h.rounds.push_back(rd);
    }
    return head;
  }

  // The rows of perm[lo .. hi): long rows and short rows each form groups of
  // consecutive rows, the long ones (blocks of several rounds) first.
  void build(const std::vector<uint32_t>& perm, uint32_t lo, uint32_t hi) {
    struct Row {
      uint32_t row, length, local;
    };
    std::vector<Row> small;
    std::vector<uint32_t> large;
    CsrQuad quads[64];
    // (about a fifth of the steps' lanes hold no entry)
    size_t entries = 0;
    for (uint32_t i = lo; i < hi; ++i) entries += length(perm[i]);
    h.vals.reserve(entries + entries / 4);
    h.idx.reserve(entries / 4 + entries / 16);
    auto flush_small = [&]() {
      if (small.empty()) return;
      // longest first, so that the 16 rows of a wave are of similar length
      // (stable, by counting)
      uint32_t first[tsn::kCsrShortEntries + 2] = {};
      for (const Row& r : small) ++first[tsn::kCsrShortEntries - r.length + 1];
      for (uint32_t i = 1; i < tsn::kCsrShortEntries + 2; ++i) first[i] += first[i - 1];
      tsn::CsrBlock b{};
      b.row0 = static_cast<uint32_t>(h.row_ids.size());
      b.n_rows = static_cast<uint32_t>(small.size());
      h.row_ids.resize(b.row0 + b.n_rows);
      for (const Row& r : small) {
        const uint32_t q = first[tsn::kCsrShortEntries - r.length]++;
        h.row_ids[b.row0 + q] = rows[r.row];
        quads[q] = {view.begin(r.row), 1, r.length, r.local};
      }
      emit(b, quads, b.n_rows);
      small.clear();
    };
    auto flush_large = [&]() {
      if (large.empty()) return;
      tsn::CsrBlock b{};
      b.row0 = static_cast<uint32_t>(h.row_ids.size());
      b.n_rows = static_cast<uint32_t>(large.size());
      b.n_chunks = tsn::div_up(length(large[0]), tsn::kCsrChunkEntries);
      if (b.n_chunks > 1) {
        b.slot0 = h.slots;
        b.counter = h.counters;
        h.slots += b.n_chunks * b.n_rows;
        h.counters += 1;
      }
      for (uint32_t t : large) h.row_ids.push_back(rows[t]);
      for (uint32_t c = 0; c < b.n_chunks; ++c) {
        b.chunk = c;
        for (uint32_t r = 0; r < b.n_rows; ++r) {
          const uint32_t n = length(large[r]), t = view.begin(large[r]);
          const uint32_t e0 = t + static_cast<uint32_t>(static_cast<uint64_t>(n) * c / b.n_chunks);
          const uint32_t e1 = t + static_cast<uint32_t>(static_cast<uint64_t>(n) * (c + 1) / b.n_chunks);
          const uint32_t at = name(e0, e1);
          for (uint32_t p = 0; p < 4; ++p) quads[4 * r + p] = {e0 + p, 4, (e1 - e0 + 3 - p) / 4, at + p};
        }
        emit(b, quads, 4 * b.n_rows);
      }
      large.clear();
    };
    for (uint32_t i = lo; i < hi; ++i) {
      const uint32_t t = perm[i], n = length(t);
      if (n <= tsn::kCsrShortEntries) continue;
      if (large.size() == long_rows || (!large.empty() && tsn::div_up(n, tsn::kCsrChunkEntries) !=
                                                       tsn::div_up(length(large[0]), tsn::kCsrChunkEntries)))
        flush_large();
      large.push_back(t);
    }
    flush_large();
    for (uint32_t i = lo; i < hi; ++i) {
      const uint32_t t = perm[i], n = length(t);
      if (n > tsn::kCsrShortEntries) continue;
      if (small.size() == short_rows) flush_small();
      const uint32_t named = n_uniq;
      uint32_t at = name(view.begin(t), view.begin(t) + n);
      if (n_uniq > tsn::kCsrCols && !small.empty()) {  // the row starts the next block
        n_uniq = named;
        flush_small();  // (and with it the row's names)
        at = name(view.begin(t), view.begin(t) + n);
      }
      small.push_back({t, n, at});
    }
    flush_small();
  }
};

}  // namespace

// Launch order of an FP32 direction's blocks: XCD x runs the x-th of eight equal
// ranges (xcd_remap), so the blocks are cut into eight contiguous runs of equal
// work (steps, and a round's start counted as kCsrRoundSteps), each run's long
// rows go first (blocks of several rounds last the longest), and shorter runs
// are filled up with blocks of no rows.  512^2 / 8 coils adjoint: 30.1 -> 27.6 us
// against equal block counts.
static void csr_balance(std::vector<tsn::CsrBlock>* blocks, const std::vector<tsn::CsrRound>& rounds) {
  constexpr uint32_t kCsrRoundSteps = 6;
  auto longest = [](const tsn::CsrRound& r) {
    uint32_t n = 0;
    for (uint32_t w = 0; w < 4; ++w) n = std::max(n, (r.steps >> (8 * w)) & 0xFFu);
    return n + kCsrRoundSteps;
  };
  auto work = [&](const tsn::CsrBlock& b) {
    uint64_t n = longest(b.first);
    for (uint32_t k = 1; k < b.n_rounds; ++k) n += longest(rounds[b.round0 + k - 1]);
    return n;
  };
  uint64_t total = 0, done = 0;
  for (const tsn::CsrBlock& b : *blocks) total += work(b);
  std::vector<tsn::CsrBlock> runs[8];
  for (const tsn::CsrBlock& b : *blocks) {
    const uint64_t w = work(b);
    runs[std::min<uint64_t>(7, (2 * done + w) * 4 / std::max<uint64_t>(total, 1))].push_back(b);
    done += w;
  }
  size_t most = 0;
  for (auto& r : runs) {
    std::stable_partition(r.begin(), r.end(), [](const tsn::CsrBlock& b) { return b.n_chunks != 0; });
    most = std::max(most, r.size());
  }
  blocks->clear();
  for (auto& r : runs) {
    r.resize(most, tsn::CsrBlock{});
    blocks->insert(blocks->end(), r.begin(), r.end());
  }
}

// Blocks of an FP32 direction: the rows of the view in the order `perm` (row t
// is output row rows[t]), cut into up to kCsrParts ranges of equally many
// entries (to within a row) built side by side (false: out of memory).  In a
// range, short rows form groups of up to 64 rows naming at most kCsrCols
// distinct columns (one round), long rows groups of up to 16 rows of equally
// many chunks, one block per chunk.
template <typename View>
static bool csr_build(const View& view, const std::vector<int32_t>& rows, const std::vector<uint32_t>& perm,
                      uint32_t entries, uint32_t n_cols, std::vector<tsn::CsrHost>* out) {
  const uint32_t n = static_cast<uint32_t>(perm.size());
  // ranges of fewer than kCsrPartEntries entries cost more in groups cut short
  // at their ends and in threads than they save; ranges of equally many rows
  // left the dense centre's rows to a few threads (205,824 samples, transpose:
  // 11-12 -> 8.3 ms for the blocks)
  const uint32_t parts = std::clamp(entries / tsn::kCsrPartEntries, 1u, tsn::kCsrParts);
  out->clear();
  out->resize(parts);
  std::vector<uint32_t> cut(parts + 1, n);
  cut[0] = 0;
  uint64_t before = 0;
  for (uint32_t i = 0, k = 1; i < n && k < parts; ++i) {
    before += view.begin(perm[i] + 1) - view.begin(perm[i]);
    for (; k < parts && before * parts >= static_cast<uint64_t>(entries) * k; ++k) cut[k] = i + 1;
  }
  // blocks hold fewer rows where full ones would not give every compute unit
  // one, down to one wave's quads (24 x 64 samples, 32^2 image, 8 coils: a solve
  // of 6 steps 190 -> 187 us)
  uint32_t n_long = 0;
  for (uint32_t t = 0; t < n; ++t) n_long += view.begin(t + 1) - view.begin(t) > tsn::kCsrShortEntries;
  const uint32_t short_rows = std::clamp((n - n_long) / tsn::kCsrUnits / 16 * 16, 16u, 64u);
  const uint32_t long_rows = std::clamp(n_long / tsn::kCsrUnits / 4 * 4, 4u, 16u);
  std::atomic<uint32_t> next{0};
  std::atomic<bool> done{true};
  using Builder = CsrBuilder<View>;
  auto work = [&]() {
    try {
      // (zeros from calloc: only the pages that the thread's rows name are ever touched)
      std::unique_ptr<typename Builder::Slot, decltype(&std::free)> slots(
          static_cast<typename Builder::Slot*>(std::calloc(n_cols, sizeof(typename Builder::Slot))), &std::free);
      if (!slots) throw std::bad_alloc();
      uint32_t group = 1;
      for (uint32_t k; (k = next++) < parts;) {
        Builder b{view, rows, short_rows, long_rows, slots.get(), group};
        b.build(perm, cut[k], cut[k + 1]);
        (*out)[k] = std::move(b.h);
        group = b.group;
      }
    } catch (const std::bad_alloc&) {
      done = false;
    }
  };
  const uint32_t threads = std::clamp(std::thread::hardware_concurrency(), 1u, parts);
  std::vector<std::thread> pool;
  pool.reserve(threads);  // nothing may throw past a running helper
  try {
    for (uint32_t i = 1; i < threads; ++i) pool.emplace_back(work);
  } catch (const std::system_error&) {  // fewer helpers
  } catch (const std::bad_alloc&) {
  }
  work();
  for (std::thread& t : pool) t.join();
  return done;
}

std::vector<tsn::ChunkItem> tsn::long_chunks(const std::vector<uint32_t>& off, uint32_t problem, uint32_t slot_base,
                                             uint32_t counter_base, uint32_t* slots, uint32_t* counters) {
  std::vector<ChunkItem> out;
  uint32_t slot = slot_base, counter = counter_base;
  for (size_t g = 0; g + 1 < off.size(); ++g) {
    const uint32_t b = off[g], e = off[g + 1];
    if (e - b <= static_cast<uint32_t>(kSplitAboveTiles)) continue;
    const uint32_t n = (e - b + kSplitAboveTiles - 1) / kSplitAboveTiles;
    for (uint32_t c = 0; c < n; ++c)
      out.push_back({static_cast<int32_t>(g), static_cast<int32_t>(chunk_begin(b, e, n, c)),
                     static_cast<int32_t>(chunk_begin(b, e, n, c + 1)), c, n, slot, counter, problem});
    slot += n;
    ++counter;
  }
  *slots = slot - slot_base;
  *counters = counter - counter_base;
  return out;
}

namespace tsn {

// Dense-control tiles from the sparse operands, one thread per (tile, lane):
// lane r + 16q holds compressed row r, slots 4q .. 4q+3, i.e. the two kept
// values of column chunks 2q and 2q+1; the index byte holds each chunk's
// 4-bit code (positions lo = code & 3, hi = code >> 2 of its two values in
// the chunk).  Out: expanded row r, columns 8q .. 8q+7 as {re 8 x f16},
// {im 8 x f16}, zeros elsewhere (the kept value written second wins if a
// code repeats a position, as in the reference's expansion).
__global__ __launch_bounds__(256) void expand_dense_kernel(const uint4* __restrict__ a,
                                                           const uint16_t* __restrict__ idx, uint64_t lanes,
                                                           uint4* __restrict__ dense) {
  const uint64_t e = static_cast<uint64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  if (e >= lanes) return;
  const uint4 v = a[e];
  const uint32_t code = idx[e];
  const uint32_t vals[2][4] = {{v.x & 0xFFFFu, v.x >> 16, v.y & 0xFFFFu, v.y >> 16},
                               {v.z & 0xFFFFu, v.z >> 16, v.w & 0xFFFFu, v.w >> 16}};
  uint4 out[2];
#pragma unroll
  for (int part = 0; part < 2; ++part) {  // re, im
    uint16_t d[8] = {0, 0, 0, 0, 0, 0, 0, 0};
    const uint32_t byte = (code >> (8 * part)) & 0xFFu;
#pragma unroll
    for (int cc = 0; cc < 2; ++cc) {
      const uint32_t nib = (byte >> (4 * cc)) & 0xFu;
      d[4 * cc + (nib & 3u)] = static_cast<uint16_t>(vals[part][2 * cc]);
      d[4 * cc + (nib >> 2)] = static_cast<uint16_t>(vals[part][2 * cc + 1]);
    }
    out[part] = make_uint4(d[0] | (static_cast<uint32_t>(d[1]) << 16), d[2] | (static_cast<uint32_t>(d[3]) << 16),
                           d[4] | (static_cast<uint32_t>(d[5]) << 16), d[6] | (static_cast<uint32_t>(d[7]) << 16));
  }
  dense[2 * e] = out[0];
  dense[2 * e + 1] = out[1];
}

int ensure_dense_tiles(const tsn_direction* cd) {
  if (!cd || cd->csr) return fail(TSN_ERR_ARGUMENT, "dense tiles need a packed (non-CSR) direction");
  if (cd->tile_dense) return TSN_OK;
  if (cd->h.tiles > kMaxDenseTiles)
    return fail(TSN_ERR_ARGUMENT, "pack has %u tiles, dense-control tiles hold at most %u", cd->h.tiles,
                kMaxDenseTiles);
  // the dense tiles are a cache of the direction's own operands
  auto* d = const_cast<tsn_direction*>(cd);
  const uint64_t lanes = static_cast<uint64_t>(d->h.tiles) * 64;
  if (lanes == 0) return TSN_OK;
  uint4* dense = nullptr;
  TSN_HIP(hipMalloc(reinterpret_cast<void**>(&dense), lanes * 2 * sizeof(uint4)));
  hipLaunchKernelGGL(expand_dense_kernel, dim3(div_up(lanes, 256)), dim3(256), 0, 0, d->tile_a, d->tile_idx, lanes,
                     dense);
  hipError_t e = hipGetLastError();
  if (e == hipSuccess) e = hipDeviceSynchronize();
  if (e != hipSuccess) {
    (void)hipFree(dense);
    return fail(TSN_ERR_RUNTIME, "dense tile expansion: %s", hipGetErrorString(e));
  }
  d->tile_dense = dense;
  d->bytes += lanes * 2 * sizeof(uint4);
  return TSN_OK;
}

// Chunk table, partial slots and zeroed arrival counters of a direction's
// long groups (fixed by the pack; rescheduling keeps them).
static int upload_chunks(tsn_direction* d) {
  uint32_t slots = 0, counters = 0;
  const std::vector<ChunkItem> chunks = long_chunks(d->host_offsets, 0, 0, 0, &slots, &counters);
  if (chunks.empty()) return TSN_OK;
  if (slots > kMaxSlots) return fail(TSN_ERR_ARGUMENT, "%u long-group chunks (at most %u)", slots, kMaxSlots);
  size_t bytes = 0;
  TSN_CHECK(device_copy(chunks.data(), chunks.size(), &d->chunks, &bytes));
  d->n_chunks = static_cast<uint32_t>(chunks.size());
  d->n_slots = slots;
  d->n_counters = counters;
  TSN_HIP(hipMalloc(reinterpret_cast<void**>(&d->partials), static_cast<size_t>(slots) * kSlotFloats * 4));
  TSN_HIP(hipMalloc(reinterpret_cast<void**>(&d->counters), counters * sizeof(uint32_t)));
  TSN_HIP(hipMemset(d->counters, 0, counters * sizeof(uint32_t)));
  d->bytes += bytes + static_cast<size_t>(slots) * kSlotFloats * 4 + counters * sizeof(uint32_t);
  return TSN_OK;
}

static int upload_pack(const HostPack& p, tsn_direction** out) {
  const tsn_pack_header& h = p.h;
  if (h.tiles > kMaxDeviceTiles)
    return fail(TSN_ERR_ARGUMENT, "pack has %u tiles, the device format holds at most %u", h.tiles, kMaxDeviceTiles);
  TSN_CHECK(validate_pack(p));
  const size_t tiles = h.tiles;
  std::vector<uint4> tile_a(tiles * 64);
  std::vector<uint16_t> tile_idx(tiles * 64);
  for (size_t t = 0; t < tiles; ++t) {
    uint32_t rm_re[16], rm_im[16];
    decode_row_meta(p.real_meta.data() + t * 16, rm_re);
    decode_row_meta(p.imag_meta.data() + t * 16, rm_im);
    const uint16_t* cre = p.real_comp.data() + t * 256;
    const uint16_t* cim = p.imag_comp.data() + t * 256;
    for (int lane = 0; lane < 64; ++lane) {
      const int r = lane & 15, q = lane >> 4;
      const uint16_t* re4 = cre + r * 16 + 4 * q;
      const uint16_t* im4 = cim + r * 16 + 4 * q;
      uint4 v;
      v.x = re4[0] | (static_cast<uint32_t>(re4[1]) << 16);
      v.y = re4[2] | (static_cast<uint32_t>(re4[3]) << 16);
      v.z = im4[0] | (static_cast<uint32_t>(im4[1]) << 16);
      v.w = im4[2] | (static_cast<uint32_t>(im4[3]) << 16);
      tile_a[t * 64 + lane] = v;
      tile_idx[t * 64 + lane] = static_cast<uint16_t>(((rm_re[r] >> (8 * q)) & 0xFF) |
                                                      (((rm_im[r] >> (8 * q)) & 0xFF) << 8));
    }
  }
  // Device column words (see TileCols): byte offset of the column's row in a
  // half panel, bit 31 of word 2 of each lane segment = last tile of a group.
  if (h.n_cols > kMaxDeviceCols)
    return fail(TSN_ERR_ARGUMENT, "pack has %u columns, the device format holds at most %u", h.n_cols,
                kMaxDeviceCols);
  std::vector<uint32_t> dev_cols(p.tile_col_ids.size());
  for (size_t i = 0; i < dev_cols.size(); ++i) dev_cols[i] = static_cast<uint32_t>(p.tile_col_ids[i]) * 32u;
  for (uint32_t g = 0; g < h.groups; ++g) {
    if (p.group_offsets[g + 1] == p.group_offsets[g]) continue;
    const size_t t = p.group_offsets[g + 1] - 1;
    for (int q = 0; q < 4; ++q) dev_cols[t * kK + q * 8 + 2] |= 0x80000000u;
  }
  auto* d = new tsn_direction();
  d->h = h;
  d->values = p.values;
  (void)hipGetDevice(&d->device);
  d->host_offsets = p.group_offsets;
  size_t bytes = 0;
  int rc = TSN_OK;
  if (rc == TSN_OK) rc = device_copy(p.group_offsets.data(), p.group_offsets.size(), &d->group_offsets, &bytes);
  if (rc == TSN_OK) rc = device_copy(p.group_row_ids.data(), p.group_row_ids.size(), &d->group_rows, &bytes);
  if (rc == TSN_OK) rc = device_copy(dev_cols.data(), dev_cols.size(), &d->tile_cols, &bytes);
  if (rc == TSN_OK) rc = device_copy(tile_a.data(), tile_a.size(), &d->tile_a, &bytes);
  if (rc == TSN_OK) rc = device_copy(tile_idx.data(), tile_idx.size(), &d->tile_idx, &bytes);
  d->bytes = bytes;
  if (rc == TSN_OK) rc = schedule_units(d, 0, {&d->line_rows, &d->block_rows});
  if (rc == TSN_OK) rc = upload_chunks(d);
  if (rc != TSN_OK) {
    release(d);
    return rc;
  }
  *out = d;
  return TSN_OK;
}

constexpr uint32_t kMemberGroup = 8;  // default member group (batch autotuner candidate)

int interp_batch_build(const std::vector<InterpBatchPart>& parts, InterpBatch* out, bool lines,
                       uint32_t member_group, uint32_t coil_waves, uint32_t depth) {
  *out = InterpBatch{};
  if (depth > 3) return fail(TSN_ERR_ARGUMENT, "pipeline depth must be 0 (default) or 1..3");
  if (member_group == 0) member_group = kMemberGroup;
  if (coil_waves != 1 && coil_waves != 2) return fail(TSN_ERR_ARGUMENT, "coil_waves must be 1 or 2");
  if (parts.empty()) return fail(TSN_ERR_ARGUMENT, "empty interpolation batch");
  const int values = parts[0].dir->values;
  const uint32_t blocks = parts[0].blocks;
  if (blocks != 1 && blocks != 2) return fail(TSN_ERR_ARGUMENT, "a batch part covers 1 or 2 coil blocks");
  lines = lines && blocks == 2;
  std::vector<InterpProblem> probs;
  for (const InterpBatchPart& p : parts) {
    const tsn_direction* d = p.dir;
    if (!d || d->csr) return fail(TSN_ERR_ARGUMENT, "batched interpolation needs packed directions");
    if (d->values != values) return fail(TSN_ERR_ARGUMENT, "a batch mixes tile value formats");
    if (p.blocks != blocks) return fail(TSN_ERR_ARGUMENT, "a batch mixes parts of 1 and 2 coil blocks");
    InterpProblem q{};
    q.group_rows = d->group_rows;
    q.tile_cols = d->tile_cols;
    q.tile_a = d->tile_a;
    q.tile_idx = d->tile_idx;
    q.tile_dense = d->tile_dense;
    q.n_tiles = d->h.tiles;
    q.n_groups = d->h.groups;
    q.n_out = d->h.output_size;
    q.n_cols = d->h.n_cols;
    q.lines = lines ? 1u : 0u;
    if (lines && q.n_cols > kMaxLineCols)
      return fail(TSN_ERR_ARGUMENT, "line-row panels hold at most %u columns (got %u)", kMaxLineCols, q.n_cols);
    q.coils = p.coils;
    q.coil_base = p.coil_base;
    q.panel_il = p.panel_il;
    q.out_f32 = p.out_f32;
    q.out_il = p.out_il;
    // row-major output: compact rows of the problem's coils (one block), or
    // 64-byte rows in blocks of 8 coils (two blocks)
    q.out_rs = blocks == 2 ? kCoilsPerBlock : p.coils;
    q.out_bs = blocks == 2 ? static_cast<uint64_t>(q.n_out) * kCoilsPerBlock : kCoilsPerBlock;
    probs.push_back(q);
  }
  // Parts are grouped by direction, in order of first appearance.  Each
  // direction's own launch order (cut into one range per XCD, longest first)
  // is split at its XCD boundaries, and XCD x of the batch runs piece x of
  // every direction, one after the other: as in a launch of its own, each
  // XCD's L2 holds one eighth of a panel's columns at a time.  Within a
  // piece, groups of kMemberGroup members of a direction (frames sharing a
  // pack) follow each entry, so they reuse its tile operands from L2 while
  // only that many panels are gathered from at once (24 frames of 768^2 / 16
  // coils: 243 ms with all members per entry, 231 ms in groups of 8).
  std::vector<const tsn_direction*> dirs;
  for (const InterpBatchPart& p : parts)
    if (std::find(dirs.begin(), dirs.end(), p.dir) == dirs.end()) dirs.push_back(p.dir);
  std::vector<WorkItem> items;
  std::vector<uint32_t> item_problem;
  std::vector<ChunkItem> chunks;
  std::vector<uint32_t> xcd_entries[8];
  uint32_t slots = 0, counters = 0;
  for (const tsn_direction* d : dirs) {
    std::vector<uint32_t> members;
    for (uint32_t i = 0; i < parts.size(); ++i)
      if (parts[i].dir == d) members.push_back(i);
    // every part has its own slots and counters
    uint32_t ns = 0, nc = 0;
    const std::vector<ChunkItem> dc = long_chunks(d->host_offsets, 0, 0, 0, &ns, &nc);
    const TileSchedule& schedule = lines ? d->line_rows : d->block_rows;
    const uint32_t nd = static_cast<uint32_t>(schedule.host_order.size());
    for (uint32_t x = 0; x < 8; ++x) {
      const uint32_t lo = xcd_remap(x, nd), hi = x == 7 ? nd : xcd_remap(x + 1, nd);
      const uint32_t nm = static_cast<uint32_t>(members.size());
      for (uint32_t k0 = 0; k0 < nm; k0 += member_group)
      for (uint32_t i = lo; i < hi; ++i) {
        const uint32_t e = schedule.host_order[i];
        for (uint32_t k = k0; k < std::min(nm, k0 + member_group); ++k) {
          if (e & kChunkTag) {
            ChunkItem c = dc[e & ~kChunkTag];
            c.slot0 += slots + k * ns;
            c.counter += counters + k * nc;
            c.problem = members[k];
            xcd_entries[x].push_back(kChunkTag | static_cast<uint32_t>(chunks.size()));
            chunks.push_back(c);
          } else {
            xcd_entries[x].push_back(static_cast<uint32_t>(items.size()));
            items.push_back(schedule.host_items[e]);
            item_problem.push_back(members[k]);
          }
        }
      }
    }
    slots += static_cast<uint32_t>(members.size()) * ns;
    counters += static_cast<uint32_t>(members.size()) * nc;
  }
  // The launch takes XCD ranges of equal length (xcd_remap), so a few entries
  // at each boundary run on the neighbouring XCD.
  std::vector<uint32_t> order;
  for (const std::vector<uint32_t>& v : xcd_entries) order.insert(order.end(), v.begin(), v.end());
  InterpBatch b;
  b.blocks = blocks;
  b.lines = lines;
  b.coil_waves = coil_waves;
  b.depth = depth;
  b.member_group = member_group;
  b.values = values;
  b.dense = std::all_of(parts.begin(), parts.end(), [](const InterpBatchPart& p) { return p.dir->tile_dense; });
  b.n_problems = static_cast<uint32_t>(probs.size());
  b.n_items = static_cast<uint32_t>(items.size());
  b.n_chunks = static_cast<uint32_t>(chunks.size());
  size_t bytes = 0;
  InterpProblem* dprobs = nullptr;
  int rc = device_copy(probs.data(), probs.size(), &dprobs, &bytes);
  b.problems = dprobs;
  if (rc == TSN_OK) rc = device_copy(items.data(), items.size(), &b.items, &bytes);
  if (rc == TSN_OK) rc = device_copy(item_problem.data(), item_problem.size(), &b.item_problem, &bytes);
  if (rc == TSN_OK) rc = device_copy(chunks.data(), chunks.size(), &b.chunks, &bytes);
  if (rc == TSN_OK) rc = device_copy(order.data(), order.size(), &b.order, &bytes);
  if (rc == TSN_OK && slots > kMaxSlots)
    rc = fail(TSN_ERR_ARGUMENT, "%u long-group chunks in the batch (at most %u)", slots, kMaxSlots);
  if (rc == TSN_OK && slots) {
    const hipError_t e1 = hipMalloc(reinterpret_cast<void**>(&b.partials), static_cast<size_t>(slots) * kSlotFloats * 4);
    const hipError_t e2 = e1 == hipSuccess ? hipMalloc(reinterpret_cast<void**>(&b.counters), counters * 4) : e1;
    const hipError_t e3 = e2 == hipSuccess ? hipMemset(b.counters, 0, counters * 4) : e2;
    if (e3 != hipSuccess) rc = fail(TSN_ERR_RUNTIME, "batch chunk buffers: %s", hipGetErrorString(e3));
  }
  if (rc != TSN_OK) {
    interp_batch_free(&b);
    return rc;
  }
  *out = b;
  return TSN_OK;
}

void interp_batch_free(InterpBatch* b) {
  if (!b) return;
  void* ptrs[] = {b->problems, b->items, b->item_problem, b->chunks, b->partials, b->counters, b->order};
  for (void* p : ptrs)
    if (p) (void)hipFree(p);
  *b = InterpBatch{};
}

// One wave per entry, or (two coil blocks) one per block; entries of two
// blocks in separate panels always take the latter.
template <int KIND>
static void launch_batch_kind(const InterpArgs& a, const InterpBatch& b, int out_mode, bool conj, hipStream_t s) {
  constexpr int kSplitOut = KIND == kSparseSplitBF16 ? kOutSplitBF16IL : kOutSplit16IL;
  if (b.blocks == 2 && (b.coil_waves == 2 || !b.lines)) {
    if (conj) launch_both<KIND, 1, kBlocks, kOutRowMajor, true, false, 2>(a, s);
    else launch_both<KIND, 1, kBlocks, kSplitOut, false, false, 2>(a, s);
  } else if (b.blocks == 2) {
    if (conj) launch_both<KIND, 2, kLines, kOutRowMajor, true, false, 1>(a, s);
    else launch_both<KIND, 2, kLines, kSplitOut, false, false, 1>(a, s);
  } else {
    if (conj) launch_both<KIND, 1, kBlocks, kOutRowMajor, true, false, 1>(a, s);
    else launch_both<KIND, 1, kBlocks, kSplitOut, false, false, 1>(a, s);
  }
}

int launch_interp_batch(const InterpBatch& b, int kind, int out_mode, bool conj, float scale, hipStream_t s) {
  if (!b.problems) return fail(TSN_ERR_ARGUMENT, "empty interpolation batch");
  if (out_mode != (conj ? kOutRowMajor : kOutSplit16IL))
    return fail(TSN_ERR_ARGUMENT, "batched interpolation writes split panels (forward) or row-major float2 (adjoint)");
  if ((kind == kSparseSplitBF16) != (b.values == TSN_VALUES_BF16))
    return fail(TSN_ERR_ARGUMENT, "tile value format of the batch does not match the interpolation variant");
  if (kind == kDenseSplit && !b.dense) return fail(TSN_ERR_ARGUMENT, "batch has no dense-control tiles");
  InterpArgs a{};
  a.items = b.items;
  a.n_items = b.n_items;
  a.chunks = b.chunks;
  a.n_chunks = b.n_chunks;
  a.order = b.order;
  a.partials = b.partials;
  a.counters = b.counters;
  a.scale = scale;
  a.problems = static_cast<const InterpProblem*>(b.problems);
  a.item_problem = b.item_problem;
  a.coils = kCoilsPerBlock;  // replaced per problem
  a.depth = b.depth;
  switch (kind) {
    case kSparseSplit: launch_batch_kind<kSparseSplit>(a, b, out_mode, conj, s); break;
    case kDenseSplit: launch_batch_kind<kDenseSplit>(a, b, out_mode, conj, s); break;
    case kSparseHi: launch_batch_kind<kSparseHi>(a, b, out_mode, conj, s); break;
    case kSparseSplitBF16:
      launch_batch_kind<kSparseSplitBF16>(a, b, out_mode, conj, s);
      break;
    default: return fail(TSN_ERR_ARGUMENT, "unknown interpolation kind %d", kind);
  }
  TSN_HIP(hipGetLastError());
  return TSN_OK;
}

// ------------------------------------------------- no-allocation entry point
// tsn_interp_noalloc takes the long-group chunk scratch from this file-scope
// array instead of the direction's: kStaticSlots partial slots (4 KiB each)
// followed by kStaticCounters arrival counters, 6 MiB + 16 KiB in all.  Every
// device the library runs on holds its own copy until the process ends.  On
// the host `scratch` names a host-side stand-in, never the device memory: the
// device address comes from hipGetSymbolAddress, once per device, and only
// that address is handed to kernels.
constexpr uint32_t kStaticSlots = 1536;
constexpr uint32_t kStaticCounters = 4096;
constexpr size_t kStaticScratchWords = static_cast<size_t>(kStaticSlots) * kSlotFloats + kStaticCounters;
static __device__ __align__(256) uint32_t scratch[kStaticScratchWords];
constexpr int kMaxStaticDevices = 64;

// Device address of `scratch` on the current device (looked up on the first
// call per device).
static int static_scratch(uint32_t** out) {
  static std::mutex lock;
  static uint32_t* address[kMaxStaticDevices] = {};
  int device = 0;
  TSN_HIP(hipGetDevice(&device));
  if (device < 0 || device >= kMaxStaticDevices)
    return fail(TSN_ERR_ARGUMENT, "device %d is beyond the %d devices of the static scratch table", device,
                kMaxStaticDevices);
  std::lock_guard<std::mutex> guard(lock);
  if (!address[device]) {
    void* ptr = nullptr;
    TSN_HIP(hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch)));
    if (!ptr) return fail(TSN_ERR_RUNTIME, "no device address for the static scratch on device %d", device);
    address[device] = static_cast<uint32_t*>(ptr);
  }
  *out = address[device];
  return TSN_OK;
}

__global__ __launch_bounds__(256) void clear_words_kernel(uint4* __restrict__ p, uint32_t n4) {
  const uint32_t e = blockIdx.x * blockDim.x + threadIdx.x;
  if (e < n4) p[e] = make_uint4(0u, 0u, 0u, 0u);
}

}  // namespace tsn

extern "C" {

int tsn_interp_noalloc(const tsn_direction* d, const void* hi, const void* res, void* out, uint32_t coils,
                       int conjugate, int accumulate, float scale, int out_layout, void* stream) {
  if (out_layout != TSN_OUT_COIL_MAJOR && out_layout != TSN_OUT_ROW_MAJOR)
    return fail(TSN_ERR_ARGUMENT, "unknown output layout %d", out_layout);
  if (!d || d->csr) return fail(TSN_ERR_ARGUMENT, "interpolation needs a packed (non-CSR) direction");
  if (d->n_slots > kStaticSlots || d->n_counters > kStaticCounters)
    return fail(TSN_ERR_ARGUMENT,
                "direction needs %u chunk slots and %u counters; the static scratch holds %u and %u",
                d->n_slots, d->n_counters, kStaticSlots, kStaticCounters);
  int device = 0;
  TSN_HIP(hipGetDevice(&device));
  if (device != d->device)
    return fail(TSN_ERR_ARGUMENT, "direction lives on device %d, the current device is %d", d->device, device);
  ChunkScratch chunk;
  hipStream_t s = static_cast<hipStream_t>(stream);
  if (d->n_chunks) {
    uint32_t* base = nullptr;
    TSN_CHECK(static_scratch(&base));
    chunk.partials = reinterpret_cast<float*>(base);
    chunk.counters = base + static_cast<size_t>(kStaticSlots) * kSlotFloats;
    // the counters this launch uses start at zero whatever the last call left
    const uint32_t n4 = div_up(d->n_counters, 4);
    hipLaunchKernelGGL(clear_words_kernel, dim3(div_up(n4, 256)), dim3(256), 0, s,
                       reinterpret_cast<uint4*>(chunk.counters), n4);
    TSN_HIP(hipGetLastError());
  }
  return launch_interp(d, res ? kSparseSplit : kSparseHi, hi, res, coils, out_layout, conjugate != 0,
                       accumulate != 0, scale, static_cast<float*>(out), s, kHalves, nullptr,
                       d->n_chunks ? &chunk : nullptr);
}

int tsn_direction_upload(const tsn_host_pack* pack, tsn_direction** out) {
  if (!pack || !out) return fail(TSN_ERR_ARGUMENT, "null argument");
  *out = nullptr;
  return upload_pack(*pack, out);
}

int tsn_direction_schedule(tsn_direction* d, uint32_t unit_tiles) {
  if (!d) return fail(TSN_ERR_ARGUMENT, "null direction");
  if (d->csr) return fail(TSN_ERR_ARGUMENT, "a CSR direction has no tile schedule");
  if (unit_tiles > (1u << 20)) return fail(TSN_ERR_ARGUMENT, "unit_tiles %u is out of range", unit_tiles);
  TSN_HIP(hipSetDevice(d->device));
  TSN_HIP(hipDeviceSynchronize());
  return schedule_units(d, unit_tiles, {&d->line_rows, &d->block_rows});
}

uint32_t tsn_direction_unit_tiles(const tsn_direction* d) { return d ? d->line_rows.unit_tiles : 0; }

int tsn_direction_set_coil_waves(tsn_direction* d, uint32_t waves) {
  if (!d) return fail(TSN_ERR_ARGUMENT, "null direction");
  if (waves != 1 && waves != 2) return fail(TSN_ERR_ARGUMENT, "coil waves must be 1 or 2 (got %u)", waves);
  d->line_rows.coil_waves = d->block_rows.coil_waves = waves;
  return TSN_OK;
}

uint32_t tsn_direction_coil_waves(const tsn_direction* d) { return d ? d->line_rows.coil_waves : 0; }

int tsn_direction_set_pipe_depth(tsn_direction* d, uint32_t depth) {
  if (!d) return fail(TSN_ERR_ARGUMENT, "null direction");
  if (depth > 3) return fail(TSN_ERR_ARGUMENT, "pipeline depth must be 0 (default) or 1..3");
  d->line_rows.pipe_depth = d->block_rows.pipe_depth = depth;
  return TSN_OK;
}

uint32_t tsn_direction_pipe_depth(const tsn_direction* d) { return d ? d->line_rows.pipe_depth : 0; }

int tsn_direction_autotune(tsn_direction* d, uint32_t coils, void* stream, uint32_t* best_unit_tiles,
                           float* best_us) {
  if (!d) return fail(TSN_ERR_ARGUMENT, "null direction");
  if (d->csr) return fail(TSN_ERR_ARGUMENT, "a CSR direction has no tile schedule");
  if (coils == 0 || coils > static_cast<uint32_t>(kMaxCoils)) return fail(TSN_ERR_ARGUMENT, "coils must be in 1..16");
  hipStream_t s = static_cast<hipStream_t>(stream);
  TSN_HIP(hipSetDevice(d->device));
  const uint32_t blocks = div_up(coils, kCoilsPerBlock);
  const size_t panel_words = static_cast<size_t>(blocks) * d->h.n_cols * kN;
  // timed with the interleaved split output (64-byte rows per coil block, as
  // plans write both directions' outputs: split panels forward, float2 rows
  // adjoint); a coil-major output's scattered writes rank the units differently
  const size_t out_words = static_cast<size_t>(blocks) * d->h.output_size * kN;
  uint32_t* panel = nullptr;
  uint32_t* out = nullptr;
  hipEvent_t e0 = nullptr, e1 = nullptr;
  int rc = TSN_OK;
  auto hip = [&](hipError_t e, const char* what) {
    if (rc == TSN_OK && e != hipSuccess) rc = fail(TSN_ERR_RUNTIME, "autotune %s: %s", what, hipGetErrorString(e));
  };
  hip(hipMalloc(reinterpret_cast<void**>(&panel), panel_words * 4), "alloc");
  hip(hipMalloc(reinterpret_cast<void**>(&out), out_words * 4), "alloc");
  if (rc == TSN_OK) hip(hipMemsetAsync(panel, 0, panel_words * 4, s), "clear");
  hip(hipEventCreate(&e0), "event");
  hip(hipEventCreate(&e1), "event");
  const int kind = d->values == TSN_VALUES_BF16 ? kSparseSplitBF16 : kSparseSplit;
  // candidates: unit sizes x, for 9..16 coils, one wave for both coil blocks
  // or one per block x pipeline depths (the default and the alternatives of
  // the launch: 1 or 3 tiles ahead for one block per wave, 2 for two); for
  // 9..16 coils each on line rows (plans, batches) and on separate blocks
  // (tsn_interp_il), whose best schedules differ: 512^2 / 11 coils adjoint on
  // blocks 33 us, 37 us with the one that is best on line rows
  struct Candidate {
    TileSchedule* of;
    uint32_t waves, unit, depth;
  };
  const bool two = coils > static_cast<uint32_t>(kCoilsPerBlock);
  const bool line_rows = two && d->h.n_cols <= kMaxLineCols;
  std::vector<Candidate> cands;
  for (uint32_t u : {2u, 3u, 4u, 5u, 6u, 8u, 10u, 12u, 14u, 16u})
    for (TileSchedule* of : line_rows ? std::vector<TileSchedule*>{&d->line_rows, &d->block_rows}
                                      : std::vector<TileSchedule*>{&d->block_rows})
      for (uint32_t cw : two ? std::vector<uint32_t>{1u, 2u} : std::vector<uint32_t>{of->coil_waves}) {
        std::vector<uint32_t> depths = {0u};
        if (two && cw == 1) depths.push_back(2u);
        if (!two) depths.insert(depths.end(), {1u, 3u});
        for (uint32_t dp : depths) cands.push_back({of, cw, u, dp});
      }
  // two passes, the second over the candidates within 5% of their layout's best
  // (neighbouring unit sizes differ by a few percent, about the spread of one
  // timing); each candidate's faster pass counts
  struct Best {
    Candidate c;
    float ms;
  };
  Best best_lines{{&d->line_rows, d->line_rows.coil_waves, 0, d->line_rows.pipe_depth}, 0.0f};
  Best best_blocks{{&d->block_rows, d->block_rows.coil_waves, 0, d->block_rows.pipe_depth}, 0.0f};
  std::vector<float> times(cands.size(), 0.0f);
  uint32_t unit = 0;
  for (int pass = 0; pass < 2; ++pass)
  for (size_t ci = 0; ci < cands.size(); ++ci) {
    if (rc != TSN_OK) break;
    const Candidate& c = cands[ci];
    Best& best = c.of == &d->line_rows ? best_lines : best_blocks;
    if (pass == 1 && times[ci] > 1.05f * best.ms) continue;
    if (c.unit != unit) rc = schedule_units(d, c.unit, {&d->line_rows, &d->block_rows});
    unit = c.unit;
    c.of->coil_waves = c.waves;
    c.of->pipe_depth = c.depth;
    auto launch = [&]() {
      return launch_interp(d, kind, panel, nullptr, coils, kOutSplit16IL, false, false, 1.0f, nullptr, s,
                           c.of == &d->line_rows ? kLines : kBlocks, out);
    };
    for (int i = 0; rc == TSN_OK && i < 3; ++i) rc = launch();
    if (rc != TSN_OK) break;
    hip(hipEventRecord(e0, s), "event");
    constexpr int kReps = 20;
    for (int i = 0; rc == TSN_OK && i < kReps; ++i) rc = launch();
    hip(hipEventRecord(e1, s), "event");
    hip(hipEventSynchronize(e1), "event");
    float ms = 0.0f;
    hip(hipEventElapsedTime(&ms, e0, e1), "event");
    ms /= kReps;
    if (rc != TSN_OK) break;
    if (pass == 1) ms = std::min(ms, times[ci]);
    times[ci] = ms;
    if (best.c.unit == 0 || ms < best.ms) best = {c, ms};
  }
  if (!line_rows) {
    best_lines = best_blocks;
    best_lines.c.of = &d->line_rows;
    if (!two) best_lines.c.waves = d->line_rows.coil_waves;
  }
  (void)hipStreamSynchronize(s);
  if (e0) (void)hipEventDestroy(e0);
  if (e1) (void)hipEventDestroy(e1);
  if (panel) (void)hipFree(panel);
  if (out) (void)hipFree(out);
  for (const Best& best : {best_lines, best_blocks}) {
    best.c.of->coil_waves = best.c.waves;
    best.c.of->pipe_depth = best.c.depth;
  }
  // (first both at the one, then the blocks at theirs)
  if (rc == TSN_OK) rc = schedule_units(d, best_lines.c.unit, {&d->line_rows, &d->block_rows});
  if (rc == TSN_OK && best_blocks.c.unit != best_lines.c.unit)
    rc = schedule_units(d, best_blocks.c.unit, {&d->block_rows});
  if (rc != TSN_OK) return rc;
  if (best_unit_tiles) *best_unit_tiles = best_lines.c.unit;
  if (best_us) *best_us = best_lines.ms * 1000.0f;
  return TSN_OK;
}

int tsn_direction_load(const char* real_dir, const char* imag_dir, tsn_direction** out) {
  if (!out) return fail(TSN_ERR_ARGUMENT, "null argument");
  *out = nullptr;
  tsn_host_pack* p = nullptr;
  TSN_CHECK(tsn_host_pack_read(real_dir, imag_dir, &p));
  const int rc = upload_pack(*p, out);
  tsn_host_pack_free(p);
  return rc;
}

// The indices of the keys in ascending order, equal keys in order of index
// (by counting, 11 bits at a time).
static std::vector<uint32_t> stable_order(const std::vector<uint32_t>& key) {
  std::vector<uint32_t> order(key.size()), next(key.size());
  std::iota(order.begin(), order.end(), 0u);
  const uint32_t most = key.empty() ? 0 : *std::max_element(key.begin(), key.end());
  for (uint32_t shift = 0; shift < 32 && most >> shift; shift += 11) {
    uint32_t first[2049] = {};
    for (uint32_t k : key) ++first[(k >> shift & 2047u) + 1];
    for (uint32_t d = 1; d < 2049; ++d) first[d] += first[d - 1];
    for (uint32_t i : order) next[first[key[i] >> shift & 2047u]++] = i;
    order.swap(next);
  }
  return order;
}

static int upload_csr(const tsn_kb_matrix* kb, int view, tsn_direction** out) {
  const uint32_t m = kb->rows, w = kb->width;
  const uint32_t grid = kb->grid0 * kb->grid1;
  std::vector<uint32_t> ptr;
  std::vector<int32_t> rows;
  std::vector<CsrTranspose::Entry> entries;
  tsn_pack_header h{};
  h.magic = kMagic;
  h.version = kVersion;
  h.n_channels = kN;
  h.m_tile = kM;
  h.k_tile = kK;
  h.nnz = m * w;
  if (view == 0) {
    rows.resize(m);
    std::iota(rows.begin(), rows.end(), 0);
    h.output_size = m;
    h.n_cols = grid;
    h.active_rows = m;
  } else {
    // exact transpose: rows = active grid points ascending, entries by sample ascending
    std::vector<uint32_t> count(grid + 1, 0);
    for (int32_t c : kb->cols) ++count[c + 1];
    std::vector<uint32_t> start(grid + 1, 0);
    for (uint32_t g = 0; g < grid; ++g) start[g + 1] = start[g] + count[g + 1];
    entries.resize(static_cast<size_t>(m) * w);
    std::vector<uint32_t> fill(start.begin(), start.end() - 1);
    for (uint32_t i = 0, k = 0; i < m; ++i)
      for (uint32_t j = 0; j < w; ++j, ++k) entries[fill[kb->cols[k]]++] = {i, k};
    ptr.push_back(0);
    for (uint32_t g = 0; g < grid; ++g) {
      if (count[g + 1] == 0) continue;
      rows.push_back(static_cast<int32_t>(g));
      ptr.push_back(start[g + 1]);
    }
    h.output_size = grid;
    h.n_cols = m;
    h.active_rows = static_cast<uint32_t>(rows.size());
  }
  // Rows in Morton order of their k-space position (samples: the rounded grid
  // coordinate; grid points: their own): a block's rows share columns, and the
  // contiguous range of blocks each XCD runs covers a compact k-space region
  // whose input rows stay in that XCD's L2.
  const uint32_t n = static_cast<uint32_t>(rows.size());
  std::vector<uint32_t> key(n);
  for (uint32_t t = 0; t < n; ++t) {
    if (view == 0) {
      const double c0 = std::nearbyint(kb->coord0[t]), c1 = std::nearbyint(kb->coord1[t]);
      key[t] = morton_key(static_cast<uint32_t>(std::max(0.0, c0)), static_cast<uint32_t>(std::max(0.0, c1)));
    } else {
      const uint32_t g = static_cast<uint32_t>(rows[t]);
      key[t] = morton_key(g % kb->grid1, g / kb->grid1);
    }
  }
  const std::vector<uint32_t> perm = stable_order(key);
  std::vector<CsrHost> parts;
  const CsrForward forward{w, kb->cols.data(), kb->re.data(), kb->im.data()};
  const CsrTranspose transpose{ptr.data(), entries.data(), kb->re.data(), kb->im.data()};
  if (!(view == 0 ? csr_build(forward, rows, perm, h.nnz, h.n_cols, &parts)
                  : csr_build(transpose, rows, perm, h.nnz, h.n_cols, &parts)))
    return fail(TSN_ERR_RUNTIME, "out of host memory");
  // the parts one after the other: every block's offsets move by what precedes it
  CsrHost host;  // blocks, rounds, row ids and columns of all parts; values and local columns stay in parts
  uint32_t steps = 0, words = 0;
  for (const CsrHost& q : parts) {
    auto moved = [&](CsrRound r) {
      r.col0 += static_cast<uint32_t>(host.cols.size());
      r.ent0 += steps;
      r.idx0 += words;
      return r;
    };
    std::vector<CsrRound> more;
    for (const CsrRound& r : q.rounds) more.push_back(moved(r));
    for (CsrBlock b : q.blocks) {
      b.first = moved(b.first);
      b.round0 += static_cast<uint32_t>(host.rounds.size());
      b.row0 += static_cast<uint32_t>(host.row_ids.size());
      b.slot0 += host.slots;
      b.counter += host.counters;
      host.blocks.push_back(b);
    }
    host.rounds.insert(host.rounds.end(), more.begin(), more.end());
    host.cols.insert(host.cols.end(), q.cols.begin(), q.cols.end());
    host.row_ids.insert(host.row_ids.end(), q.row_ids.begin(), q.row_ids.end());
    steps += static_cast<uint32_t>(q.vals.size() / 64);
    words += static_cast<uint32_t>(q.idx.size() / 64);
    host.slots += q.slots;
    host.counters += q.counters;
  }
  csr_balance(&host.blocks, host.rounds);
  const uint32_t active_blocks = static_cast<uint32_t>(host.blocks.size());
  // Output rows no entry reaches (grid points of the transpose no sample
  // touches) follow as runs of empty rows in ascending order, so a launch that
  // does not accumulate writes zeros there too; a launch into an output
  // already zero leaves them out.
  if (rows.size() < h.output_size) {
    std::vector<uint8_t> hit(h.output_size, 0);
    for (int32_t r : rows) hit[r] = 1;
    for (uint32_t r = 0; r < h.output_size; ++r) {
      if (hit[r]) continue;
      if (host.blocks.size() == active_blocks || host.blocks.back().n_rows == kCsrEmptyRunRows) {
        CsrBlock b{};
        b.row0 = static_cast<uint32_t>(host.row_ids.size());
        host.blocks.push_back(b);
      }
      host.blocks.back().n_rows += 1;
      host.row_ids.push_back(static_cast<int32_t>(r));
    }
  }
  if (host.slots > kMaxCsrSlots)
    return fail(TSN_ERR_ARGUMENT, "%u long-row chunks (at most %u)", host.slots, kMaxCsrSlots);
  std::unique_ptr<tsn_direction, void (*)(tsn_direction*)> owner(new tsn_direction(), release);
  tsn_direction* d = owner.get();
  d->h = h;
  d->csr = true;
  (void)hipGetDevice(&d->device);
  d->n_csr_blocks = static_cast<uint32_t>(host.blocks.size());
  d->n_csr_active_blocks = active_blocks;
  d->n_slots = host.slots;
  d->n_counters = host.counters;
  // one allocation for all arrays, each array's parts one after the other
  struct Piece {
    const void* data;
    size_t bytes, at;
  };
  std::vector<Piece> pieces;
  size_t total = 0;
  auto add = [&](const auto& v) {
    const size_t bytes = v.size() * sizeof(*v.data());
    if (bytes) pieces.push_back({v.data(), bytes, total});
    total += bytes;
  };
  auto begin = [&] { return total = (total + 255) / 256 * 256; };
  const size_t vals_at = begin();
  for (const CsrHost& q : parts) add(q.vals);
  const size_t idx_at = begin();
  for (const CsrHost& q : parts) add(q.idx);
  const size_t rows_at = begin();
  add(host.row_ids);
  const size_t cols_at = begin();
  add(host.cols);
  const size_t blocks_at = begin();
  add(host.blocks);
  const size_t rounds_at = begin();
  add(host.rounds);
  TSN_HIP(hipMalloc(reinterpret_cast<void**>(&d->csr_data), std::max<size_t>(total, 1)));
  std::vector<unsigned char> stage(total <= kCsrStagedBytes ? total : 0);
  if (!stage.empty()) {
    for (const Piece& p : pieces) std::memcpy(stage.data() + p.at, p.data, p.bytes);
    pieces = {Piece{stage.data(), total, 0}};
  }
  hipError_t copied = hipSuccess;
  for (const Piece& p : pieces)
    if (copied == hipSuccess)
      copied = hipMemcpyAsync(d->csr_data + p.at, p.data, p.bytes, hipMemcpyHostToDevice, nullptr);
  const hipError_t done = hipStreamSynchronize(nullptr);  // (also after a failure: the copies read this call's memory)
  TSN_HIP(copied);
  TSN_HIP(done);
  d->vals = reinterpret_cast<float2*>(d->csr_data + vals_at);
  d->csr_idx = reinterpret_cast<uint32_t*>(d->csr_data + idx_at);
  d->row_ids = reinterpret_cast<int32_t*>(d->csr_data + rows_at);
  d->csr_cols = reinterpret_cast<uint32_t*>(d->csr_data + cols_at);
  d->csr_blocks = reinterpret_cast<CsrBlock*>(d->csr_data + blocks_at);
  d->csr_rounds = reinterpret_cast<CsrRound*>(d->csr_data + rounds_at);
  d->bytes = total;
  if (host.slots) {
    const std::vector<uint32_t> zeros(round_up(host.counters, 4u), 0u);
    const size_t slot_bytes = static_cast<size_t>(host.slots) * kMaxCoils * sizeof(float2);
    TSN_HIP(hipMalloc(reinterpret_cast<void**>(&d->partials), slot_bytes));
    TSN_CHECK(device_copy(zeros.data(), zeros.size(), &d->counters, &d->bytes));
    d->bytes += slot_bytes;
  }
  *out = owner.release();
  return TSN_OK;
}

int tsn_direction_upload_csr(const tsn_kb_matrix* kb, int view, tsn_direction** out) {
  if (!kb || !out || (view != 0 && view != 1)) return fail(TSN_ERR_ARGUMENT, "bad argument");
  *out = nullptr;
  try {
    return upload_csr(kb, view, out);
  } catch (const std::bad_alloc&) {
    return fail(TSN_ERR_RUNTIME, "out of host memory");
  }
}

int tsn_direction_header(const tsn_direction* d, tsn_pack_header* out) {
  if (!d || !out) return fail(TSN_ERR_ARGUMENT, "null argument");
  *out = d->h;
  return TSN_OK;
}

size_t tsn_direction_bytes(const tsn_direction* d) { return d ? d->bytes : 0; }

int tsn_direction_expand_dense(tsn_direction* d) { return ensure_dense_tiles(d); }

void tsn_direction_free(tsn_direction* d) { release(d); }

int tsn_interp(const tsn_direction* d, const void* hi, const void* res, void* out, uint32_t coils,
               int conjugate, int accumulate, float scale, int out_layout, void* stream) {
  if (out_layout != TSN_OUT_COIL_MAJOR && out_layout != TSN_OUT_ROW_MAJOR)
    return fail(TSN_ERR_ARGUMENT, "unknown output layout %d", out_layout);
  return launch_interp(d, res ? kSparseSplit : kSparseHi, hi, res, coils, out_layout, conjugate != 0,
                       accumulate != 0, scale, static_cast<float*>(out), static_cast<hipStream_t>(stream), kHalves, nullptr);
}

int tsn_interp_dense(const tsn_direction* d, const void* hi, const void* res, void* out,
                     uint32_t coils, int conjugate, int accumulate, float scale, int out_layout,
                     void* stream) {
  if (out_layout != TSN_OUT_COIL_MAJOR && out_layout != TSN_OUT_ROW_MAJOR)
    return fail(TSN_ERR_ARGUMENT, "unknown output layout %d", out_layout);
  if (!res) return fail(TSN_ERR_ARGUMENT, "dense control needs hi and residual panels");
  TSN_CHECK(ensure_dense_tiles(d));
  return launch_interp(d, kDenseSplit, hi, res, coils, out_layout, conjugate != 0, accumulate != 0,
                       scale, static_cast<float*>(out), static_cast<hipStream_t>(stream), kHalves, nullptr);
}

int tsn_interp_f32(const tsn_direction* d, const void* in, void* out, uint32_t coils, int conjugate,
                   int accumulate, float scale, int out_layout, void* stream) {
  return launch_interp_csr(d, static_cast<const float2*>(in), coils, out_layout, conjugate != 0,
                           accumulate != 0, scale, static_cast<float2*>(out),
                           static_cast<hipStream_t>(stream));
}

int tsn_interp_il(const tsn_direction* d, const void* panel, void* out, uint32_t coils, int conjugate,
                  int accumulate, float scale, int out_layout, void* stream) {
  if (out_layout != TSN_OUT_COIL_MAJOR && out_layout != TSN_OUT_ROW_MAJOR && out_layout != TSN_OUT_SPLIT_IL)
    return fail(TSN_ERR_ARGUMENT, "unknown output layout %d", out_layout);
  if (!d) return fail(TSN_ERR_ARGUMENT, "null direction");
  const int kind = d->values == TSN_VALUES_BF16 ? kSparseSplitBF16 : kSparseSplit;
  if (out_layout == TSN_OUT_SPLIT_IL) {
    if (accumulate) return fail(TSN_ERR_ARGUMENT, "a split-panel output cannot accumulate");
    return launch_interp(d, kind, panel, nullptr, coils, kOutSplit16IL, conjugate != 0, false, scale, nullptr,
                         static_cast<hipStream_t>(stream), kBlocks, static_cast<uint32_t*>(out));
  }
  return launch_interp(d, kind, panel, nullptr, coils, out_layout, conjugate != 0, accumulate != 0, scale,
                       static_cast<float*>(out), static_cast<hipStream_t>(stream), kBlocks, nullptr);
}

int tsn_interp_dc(const tsn_direction* d, const void* panel, const void* measurements, int measurement_layout,
                  const float* density, uint32_t coils, float scale, float measurement_scale, int mode,
                  void* workspace, void* out_panel, void* stream) {
  if (!d || !panel || !measurements || !out_panel) return fail(TSN_ERR_ARGUMENT, "null argument");
  if (d->csr) return fail(TSN_ERR_ARGUMENT, "data consistency needs a packed (non-CSR) direction");
  if (coils == 0 || coils > static_cast<uint32_t>(kMaxCoils)) return fail(TSN_ERR_ARGUMENT, "coils must be in 1..16");
  if (measurement_layout != TSN_OUT_COIL_MAJOR && measurement_layout != TSN_OUT_ROW_MAJOR)
    return fail(TSN_ERR_ARGUMENT, "unknown measurement layout %d", measurement_layout);
  if (mode != TSN_DC_MATERIALIZED && mode != TSN_DC_FUSED)
    return fail(TSN_ERR_ARGUMENT, "data-consistency mode must be 1 (materialized) or 2 (fused), got %d", mode);
  if (mode == TSN_DC_MATERIALIZED && !workspace) return fail(TSN_ERR_ARGUMENT, "materialized mode needs a workspace");
  const uint32_t rows = d->h.output_size;
  DcTerms dc;
  dc.y = static_cast<const float*>(measurements);
  dc.density = density;
  dc.scale = measurement_scale;
  dc.row_stride = measurement_layout == TSN_OUT_ROW_MAJOR ? 2 * coils : 2;
  dc.coil_stride = measurement_layout == TSN_OUT_ROW_MAJOR ? 2 : 2 * rows;
  const bool bf16 = d->values == TSN_VALUES_BF16;
  const int kind = bf16 ? kSparseSplitBF16 : kSparseSplit;
  hipStream_t s = static_cast<hipStream_t>(stream);
  auto* out = static_cast<uint32_t*>(out_panel);
  if (mode == TSN_DC_FUSED) return launch_interp_dc(d, kind, static_cast<const uint32_t*>(panel), coils, scale, dc, out, s);
  TSN_CHECK(launch_interp(d, kind, panel, nullptr, coils, kOutRowMajor, false, false, scale,
                          static_cast<float*>(workspace), s, kBlocks, nullptr));
  return launch_dc_residual(static_cast<const float2*>(workspace), rows, coils, dc, bf16, out, s);
}

int tsn_split_panel_il(const void* in, uint32_t rows, uint32_t coils, float scale, int values, void* panel,
                       void* stream) {
  return launch_split_panel_il(static_cast<const float2*>(in), rows, coils, scale,
                               static_cast<uint32_t*>(panel), static_cast<hipStream_t>(stream), values, false);
}

int tsn_split_panel(const void* in, uint32_t rows, uint32_t coils, float scale, void* hi, void* res,
                    void* stream) {
  return launch_split_panel(static_cast<const float2*>(in), rows, coils, scale,
                            static_cast<_Float16*>(hi), static_cast<_Float16*>(res),
                            static_cast<hipStream_t>(stream));
}

}  // extern "C"

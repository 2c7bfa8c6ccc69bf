// Internal declarations shared by the host side of the C-ABI and the gfx950
// kernels.  Not installed; the public interface is include/moe_abi.h.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "../../include/moe_abi.h"

namespace moe {

// Records the text of a failure for moe_last_error() on the calling thread and
// returns `code` (defined with the C-ABI's host side).
int set_error(int code, const char *fmt, ...) __attribute__((format(printf, 2, 3)));

// float -> bf16 bits, round to nearest even; a NaN stays a NaN
// (/opt/rocm/include/hip/amd_detail/amd_hip_bfloat16.h:96-131).
__device__ __forceinline__ uint16_t f32_to_bf16_rne(float f) {
  uint32_t u = __float_as_uint(f);
  if (~u & 0x7f800000u) {
    u += 0x7fffu + ((u >> 16) & 1u);
  } else if (u & 0xffffu) {
    u |= 0x10000u;
  }
  return (uint16_t)(u >> 16);
}

constexpr int kTopK = 4;        // EXPERT_PER_TOKEN, common/defines.h:27
constexpr int kRowBlock = 32;   // rows of one MFMA fragment (v_mfma_f32_32x32x16_bf16)
constexpr int kFragK = 16;      // reduction depth of one fragment
constexpr int kFragBytes = 1024;  // 64 lanes x 8 bf16
constexpr int kTileRows = 256;  // tallest row tile of the grouped GEMMs
constexpr int kHalfTileRows = 128;  // ... where two workgroups share a CU (MXFP4 weights, half_tiles)
constexpr int kTileGran = 32;   // an expert's segment of padded rows is a multiple of one row block
constexpr float kAlpha = 1.702f;  // run.cpp:709

// Work split of the grouped GEMMs over the 8 XCDs (each has an L2 of its own).
// Tiles are numbered (expert, group of row tiles, column tile, row tile of the
// group), row tile fastest; XCD x takes the tiles [bounds[x], bounds[x+1]), a
// range of about an eighth of the estimated cost.  (Cutting the last tiles of a range into smaller pieces, so
// that its CUs run dry together, was measured and does not pay: the pieces are
// less efficient than what they save.)
constexpr int kGemmTileNb = 8;  // column blocks (of 32) per tile of the grouped GEMMs (tile_width: wider plans)
constexpr int kRowTileGroup = 4;  // row tiles of one expert that run side by side (see write_expert_tiles)
constexpr int kXcds = 8;
// Estimated cost of a tile: a fixed part (plan_tile_cost) + kCostPerRowBlock * row blocks.
constexpr int kCostPerRowBlock = 8;
// layout of DispatchBuffers::totals
constexpr int kTotRows = 0;                                  // padded rows
constexpr int kTotBoundsGateUp = 1;                          // 9 ints
constexpr int kTotBoundsDown = kTotBoundsGateUp + kXcds + 1;  // 9 ints
constexpr int kTotInts = kTotBoundsDown + kXcds + 1;

// Most tiles one XCD can be given out of `total`: the balancing never moves a
// boundary further than this, so that the launch grid can be sized on the host.
__host__ __device__ inline int xcd_tile_cap(int total) { return (total + 7) / 8 + (total + 15) / 16 + 1; }

// One tile of a grouped GEMM, looked up by its number in the tile sequence.
// Written by the scan kernel for both GEMMs, so that a GEMM workgroup finds its
// work with one load instead of a binary search over the experts (a chain of
// dependent global loads in front of every tile).
struct TileDesc {
  int e;    // expert
  int rb0;  // first row block of the tile in the padded row space
  uint16_t rbt, nbt;  // its row blocks (1..8) and column blocks (1..10)
  int nb0;  // its first column block
};
// Column blocks of a tile of so many row blocks.  wide: see bf16_wide_tiles.
constexpr int kWideTileRb = 6, kWideTileNb = 10;
__host__ __device__ inline int tile_width(int height, bool wide) {
  return wide && height <= kWideTileRb ? kWideTileNb : kGemmTileNb;
}

struct LayerWeights {
  uint16_t *wr = nullptr;  // router weight, bf16 in the operand order of v_mfma_f32_16x16x32_bf16
  float *br = nullptr;     // router bias [E_pad] (padded experts = -inf), then the two floats of rstat
  uint16_t *w1 = nullptr;  // gate_up weight, bf16 MFMA fragments, gate/up blocks paired
  float *b1g = nullptr;    // gate bias [E, IM]
  float *b1u = nullptr;    // up bias   [E, IM]
  uint16_t *w2 = nullptr;  // down weight, bf16 MFMA fragments
  float *b2 = nullptr;     // down bias [E, H]
  // Expert matrices kept as MXFP4 instead (moe_upload_layer_mxfp4): 16-byte
  // chunks of nibbles and two scale bytes per row, pair of row blocks and 32 k
  // (see pack_fp4_kernel); w1/w2 are then not allocated.
  uint8_t *w1q = nullptr, *w2q = nullptr;
  uint16_t *w1s = nullptr, *w2s = nullptr;
  float *rms_w = nullptr;  // weight of the RMS norm in front of the layer [H] (bf16 values), optional
  bool uploaded = false;
};

// ---- kernel launchers (defined in the .hip files) ----

hipError_t launch_pack_router(const float *w_src, const float *b_src, uint16_t *wr, float *br,
                              int E, int E_pad, int H, hipStream_t s);
// The grouped GEMMs work on matrices whose sides are multiples of 64 (a double
// step of the reduction, a pair of column blocks).  Sizes that are multiples of
// 32 only are padded to that inside the library: zero weights and biases at
// upload, zero columns of the routed rows per call (launch_pad_rows).  The
// reference pads its packed weights likewise (utility/utility.cpp:558-622).
constexpr int kDimGran = 64;
inline int padded_dim(int n) { return (n + kDimGran - 1) / kDimGran * kDimGran; }
// rows x cols (source) -> rows_p x cols_p (packed, zero outside the source)
hipError_t launch_pack_weight(const float *src, uint16_t *dst, int rows, int cols, int rows_p, int cols_p,
                              bool gate_up, hipStream_t s);
hipError_t launch_pack_fp4(const uint8_t *blocks, const uint8_t *scales, uint8_t *wq, uint16_t *ws,
                           int rows, int cols, int rows_p, int cols_p, bool gate_up, hipStream_t s);
// n_rows rows of len values -> rows of len_p (each half len_p / 2 when de-interleaving)
hipError_t launch_pack_bias(const float *src, float *dst_a, float *dst_b, int n_rows, int len, int len_p,
                            bool deinterleave, hipStream_t s);
hipError_t launch_pad_rows(const uint16_t *x, uint16_t *xp, int T, int H, int Hp, hipStream_t s);

// rstat: two floats written by launch_router_stats at upload (largest 2-norm of
// an expert's router weights, largest bias magnitude), the inputs of the error
// bound that decides which tokens need exact fp64 logits.
hipError_t launch_router_stats(const float *w_src, const float *b_src, int E, int H, float *rstat,
                               hipStream_t s);
// first: scratch for T * (E_pad + 4) floats that no other call uses meanwhile, or nullptr.  With it, batches of up to
// split_router_tokens at more than 64 experts run the first pass on E_pad / 16 times as many
// workgroups and a launch of their own; the results are the same bits.  That pays where one workgroup
// would take long over the router matrix: the more the longer its rows, and the less the more workgroups
// there are anyway.  Time of a layer call (MXFP4 experts) with the launch over that without:
//   128 experts   tokens 1   40    200   400   600   1024
//     256 columns    1.03  1.05  1.01  1.01  1.05  1.03
//     512            1.01  1.00  1.00  0.98  1.01  1.01
//     768            0.97  0.99  0.99  0.99  1.01  1.01
//     1024           0.93  0.98  0.98  0.98  1.02  0.99
//     1440           0.92  0.97  0.97  0.98  0.99  0.99
//     2880           0.84  0.97  0.98  0.98  0.99  0.99   (4096 tokens 1.01)
//   256 experts
//     128            0.95  0.98  0.97  1.01  1.03  1.05
//     256            0.92  0.96  0.96  0.99  1.01  1.04
//     384            0.89  0.92  0.94  0.96  0.99  1.01
//     2880           0.67  0.95  0.97  0.98  0.98  0.99
inline int split_router_tokens(int E_pad, int H) {
  if (E_pad < 128) return 0;
  if (H > 1024) return 1024;
  if (E_pad == 128) return H >= 768 ? 400 : 0;
  return H >= 256 ? 400 : 200;
}
hipError_t launch_router(const uint16_t *x, const int *pos, const uint16_t *wr, const float *br,
                         const float *rstat, int T, int H, int E, int E_pad, float *score, int *topk_i,
                         float *topk_v, float *first, hipStream_t s);

struct DispatchBuffers {
  int *blk_counts;    // [n_blk, E]
  int *offsets;       // [E+1]   exclusive scan of valid rows
  int *perm;          // [A]     position -> assignment id
  int *rowmap;        // [A_pad] padded position -> assignment id, -1 = padding
  int *inv;           // [A]     assignment id -> padded position, -1 = inactive
  int *blk_expert;    // [A_pad / 32] row block of the padded rows -> expert (nullptr: not wanted)
  int *totals;        // [kTotInts]: padded rows; XCD bounds of both GEMMs
  int a_pad_cap;      // capacity of rowmap in rows
  TileDesc *tiles_gate_up;  // [tile_cap_gate_up] tile sequence of the gate_up GEMM
  TileDesc *tiles_down;     // [tile_cap_down]    ... of the down GEMM
  int tile_cap_gate_up, tile_cap_down;
};
// How the XCDs' ranges of tiles are cut (plan_tile_cost): the fixed part of a tile's estimated cost, and another
// (0: none) that a GEMM of up to `rounds` rounds of tiles on the CUs is cut by instead, where with it the slowest XCD's
// time, estimated with fixed part `slow`, is below `gain` of what it is otherwise.
struct TileCost {
  int fixed, few, rounds, slow;
  float gain;
};
// tile_rows: tallest row tile of the plan (kTileRows or kHalfTileRows); wide: tile_width; nb_*: column blocks of an
// expert's matrices (0: no tile tables)
hipError_t launch_dispatch(const int *topk_i, const int *pos, int T, int E, int nb_gate_up, int nb_down,
                           int tile_rows, bool wide, TileCost tile_cost, const DispatchBuffers &d, hipStream_t s);

// Batches of at most kDirectTokens tokens run without a dispatch pass: the 256
// threads of a workgroup hold one assignment each, so every workgroup of the
// GEMMs reads the batch's expert ids itself and finds its rows with a ballot; the
// first GEMM leaves inv for the combine.  Expert e owns the padded rows [e * kDirectSlotRows,
// (e + 1) * kDirectSlotRows); inside them its assignments stand in ascending
// order, as the dispatch kernels place them.  Requires that no expert is given
// more than kDirectSlotRows assignments.  topk_i == nullptr: not in use, the
// plan of launch_dispatch is.
constexpr int kDirectTokens = 64;
constexpr int kDirectSlotRows = 64;
struct DirectIds {
  const int *topk_i;  // [T, 4]
  const int *pos;     // [T] or nullptr
  int T, E;
};
// expert of assignment a by the rule of the dispatch kernels: -1 past the batch,
// for a row with pos < 0 and for an id outside [0, E)
__device__ __forceinline__ int direct_expert_of(const DirectIds &d, int a) {
  if (a >= d.T * kTopK) return -1;
  const int id = d.topk_i[a];                      // both loads go out together
  const int ps = d.pos ? d.pos[a / kTopK] : 0;
  return ps >= 0 && id >= 0 && id < d.E ? id : -1;
}
inline bool direct_plan_fits(int T, int max_rows, int E, int a_pad_cap) {
  return T <= kDirectTokens && max_rows <= kDirectSlotRows && kDirectSlotRows * E <= a_pad_cap;
}
// Batches in which the weights are a stream run the kernels of stream.hip: up to
// kDirectTokens tokens, and up to kStreamMeanRows rows per active expert on
// average when every expert is active.  Those kernels take 32 rows per tile, so an
// expert with more is multiplied (and, with MXFP4, decoded) once per tile, by
// workgroups that read its weights side by side (share_of in stream.hip).  On
// either side of the line, us per moe_experts call at 2880 x 2880 with the kernels
// of stream.hip / of gemm.hip, even routing and Zipf's (exponent 1.2):
//   32 experts, MXFP4:  96 tokens 98 / 113, 103 / 121;  128: 103 / 113, 109 / 141;  192: 113 / 114, 117 / 138
//   32 experts, bf16:   96 tokens 263 / 277, 261 / 285;  128: 272 / 278, 270 / 291;  192: 288 / 282, 305 / 321
//   128 experts, MXFP4: 384 tokens 342 / 367, 314 / 356;  512: 364 / 370, 372 / 424;  768: 391 / 379, 436 / 451
//   128 experts, bf16:  384 tokens 993 / 1087, 942 / 988;  512: 1027 / 1087, 1088 / 1122;  768: 1111 / 1098, 1210 / 1168
//   8 experts, 96 tokens: MXFP4 48 / 52, 49 / 60;  bf16 117 / 96, 101 / 106;  128 tokens, bf16: 135 / 106, 132 / 111
// Up to the line neither format loses under either routing; past it bf16 does.
// The rule knows nothing of the weights' format: both formats give the same bits.
constexpr int kCus = 256;
constexpr int kStreamMeanRows = 16;
inline bool stream_batch(int T, int E) { return T <= kDirectTokens || T * kTopK <= kStreamMeanRows * E; }
// row tiles of the grouped GEMMs in all, at most: row blocks of 32 (stream.hip) or tiles of tile_rows (gemm.hip)
inline int stream_tile_cap(int T, int E) {
  const int A = T * kTopK;
  return A < E ? A : (A / kRowBlock + E < A ? A / kRowBlock + E : A);
}
// ... of stream.hip without a plan: experts that can have rows, and those that can have more than kRowBlock
inline int stream_direct_tile_cap(int T, int E) {
  const int A = T * kTopK;
  return (A < E ? A : E) + A / (kRowBlock + 1);
}
inline int gemm_tile_cap(int T, int E, int tile_rows) { return T * kTopK / tile_rows + E; }
// MXFP4 weights: whether the kernels of gemm_fp4.hip (tiles of 128 rows, products of 16 x 16
// x 32) run rather than those of gemm.hip (128 or 256 rows, 32 x 32 x 16).  They do where
// the products are the time: many rows per expert on average, of all experts.  us per layer call at 2880
// x 2880, gemm.hip / gemm_fp4.hip: 32 experts, 150 tokens (19 rows) 120 / 125, 256 (32) 136 / 138,
// 512 (64) 174 / 162; 16 experts, 300 (75) 107 / 105, 450 (112) 135 / 122; 128 experts, 600 (19) 385 /
// 397, 3072 (96) 688 / 655.  With a workgroup on every CU or fewer, a wave has its SIMD to
// itself and the smaller products' instructions show until experts have more than one tile:
// 8 experts, 150 tokens (75 rows) 70 / 76, 256 (128) 93 / 99, 300 (150) 105 / 100, 400 128 / 115; 4
// experts, 100 (100) 78 / 86, 150 (150) 88 / 75.  Over 500 batches of 4 to 128 experts, sides of 512 to 2880, even
// and Zipf's routing, from 64 rows on, the time is 0.7 to 1.02 of that with gemm.hip, but for: 32 experts,
// 1024 x 2048 and 512 x 2048 (two workgroups per CU exactly), 64 to 80 rows 1.03 to 1.04; 4 experts, 2880 x
// 2880, 260 to 380 rows (276 tiles on 256 CUs) 1.00 to 1.10.  w1_rows: rows of an expert's gate_up matrix.
constexpr int kFp4ManyRows = 64;
inline bool fp4_many_rows(int T, int E, int w1_rows) {
  const int n_ct = (w1_rows / kRowBlock + kGemmTileNb - 1) / kGemmTileNb;
  return T * kTopK > kHalfTileRows * E || (T * kTopK >= kFp4ManyRows * E && E * n_ct > kCus);
}
// Height of the row tiles of a batch on MXFP4 weights: half where the kernels of gemm_fp4.hip run,
// and where it gives the GPU two workgroups per CU (CfgHalf in gemm.hip has the reason).  With
// fewer tiles than that the full height keeps more columns' worth of work in each.
inline bool half_tiles(int T, int E, int w1_rows) {
  const int n_ct = (w1_rows / kRowBlock + kGemmTileNb - 1) / kGemmTileNb;
  const int row_tiles = T * kTopK / kHalfTileRows > E ? T * kTopK / kHalfTileRows : E;
  return fp4_many_rows(T, E, w1_rows) || (long long)row_tiles * n_ct >= 2 * kCus;
}
// bf16 weights: whether row tiles of 128 rows in place of 256 are expected to be quicker.  They stream an
// expert's weights more often, so they pay only where the tall tiles leave CUs without work, in either
// GEMM, and where the weights come out of the memory-side cache (cached: kCachedWeightBytes).  The estimate: an
// expert has half a tile more than its rows fill on average; a tile takes the time of 4 + (its row blocks)
// steps of its reduction; the CUs take tiles in rounds.  us per layer call, 256 rows / 128: 4
// experts, 2880 x 2880, 145 tokens 88 / 70, 256 124 / 81; 1024 x 1024, 8 experts, 1800 tokens 96 / 79; 256 x
// 1440, 8 experts, 1000 tokens 63 / 51, 32 experts, 1440 tokens, Zipf's routing 74 / 61; 512 x 512, 32 experts,
// 1000 tokens 57 / 49.  Where the estimate says 256 rows: 8 experts, 512 x 512, 7000 tokens 92 / 96 (3000, a
// close call, 59 / 56).  128 rows have to be a tenth quicker by the estimate.
// From HBM a round more or less, which the host cannot foresee, costs more than the rule gains: where it
// says 128, at 2880 x 2880, even / Zipf's routing: 8 experts, 520 tokens 0.94 / 1.00 of the time with 256, 221
// 1.00 / 1.13, 1200 1.05 / 0.97; 10 experts, 450 1.10 / 0.96; 12 experts, 360 0.96 / 0.95, 480 1.18 /
// 0.95; 14 experts, 460 1.26 / 1.10; 24 experts, 640 0.98 / 1.12.
inline bool bf16_half_tiles(int T, int E, int H, int IM, bool cached) {
  if (!cached) return false;
  const int A = T * kTopK;
  const float blocks = (float)A / kRowBlock + 0.5f * E;
  auto time = [&](int tile_rows) {
    float tiles = (float)A / tile_rows + 0.5f * E;
    if (tiles < E) tiles = (float)E;
    auto rounds = [&](int cols) {
      const int n = (int)(tiles * ((cols / kRowBlock + kGemmTileNb - 1) / kGemmTileNb));
      return (float)((n + kCus - 1) / kCus);
    };
    return (4.f + blocks / tiles) * (H * rounds(2 * IM) + IM * rounds(H));
  };
  return time(kHalfTileRows) < 0.9f * time(kTileRows);
}
// Whether the expert matrices are read past the caches (non-temporal loads): while
// most experts have one row tile their weights are read by one workgroup, and
// lines that nobody reads again push the rows and the code out of L2.  us per
// layer call, cached / past the caches: bf16 (tiles of 256 rows), 32 experts, 256
// tokens 330 / 305, 512: 364 / 351, 1024: 392 / 374, 1536 (192 rows per expert): 433 / 414, 2048
// (256): 525 / 512, 2560: 603 / 607, 4096: 831 / 845; 128 experts, 1024: 1234 / 1173, 6144 (192): 1631 /
// 1632; 8 experts, 400 (200): 159 / 153, 600 (300): 191 / 195, 1000: 242 / 244.  MXFP4 in tiles of 128 rows,
// 32 experts, 256 tokens 143 / 135, 512: 172 / 163, 1024 (128 rows): 242 / 245, 4096: 725 / 750; 128 experts, 3072
// (96 rows): 676 / 668.  MXFP4 in tiles of 256 rows gains nothing (8 experts, 256 tokens 93 / 95), and
// bf16 has tiles of 128 rows only where the caches hold the matrices.  cached: kCachedWeightBytes.
constexpr int kStreamRowsBf16 = 256, kStreamRowsFp4 = 96;  // mean rows of an expert, at most
inline bool gemm_streams_weights(int T, int E, bool mxfp4, int tile_rows, bool cached) {
  if (cached || tile_rows != (mxfp4 ? kHalfTileRows : kTileRows)) return false;
  return T * kTopK <= (mxfp4 ? kStreamRowsFp4 : kStreamRowsBf16) * E;
}
// bf16 weights past the caches: whether tiles of up to 6 row blocks take 10 column blocks instead of 8 (the
// registers and the LDS of a workgroup hold 60 as well as 64).  A tile streams its weights for its
// whole life but for a fill and an epilogue, and reads its rows once per tile: fewer tiles, less of either.  But a
// wider tile makes the CUs' last round of tiles longer, so there have to be rounds enough that it is small beside the
// others whatever the routing, which the host does not know.  us per moe_experts call, 8 / 10 column blocks, means of two
// to four routings, even or Zipf's (exponent in brackets): 128 experts (9 rounds in gate_up, 4.5 in down at 6144 tokens),
// 6144, even, 1555 / 1457 per layer call, 4000 1206 / 1164, (0.6) 1393 / 1360, (1.2) 1530 / 1500, 2000, even, 1102 / 1095,
// (1.2) 1185 / 1188, 600, even, 1000 / 1012, (1.2) 861 / 842.  32 experts (2.3 rounds, 1.1), where either may win: even, 256
// 277 / 308, 512 281 / 320, 1000 313 / 351, 1400 350 / 387, but (1.2) 450 337 / 310, 512 331 / 322, 600 339 / 345, (0.6) 1400
// 417 / 403; 1800 405 / 399, (0.6) 460 / 441.  8 experts, 250, even, 116 / 130, 500 167 / 143.
inline bool bf16_wide_tiles(int T, int E, int H, int IM, bool past_caches) {
  const int cols = (H < 2 * IM ? H : 2 * IM) / kRowBlock;
  const int row_tiles = T * kTopK / kTileRows > E ? T * kTopK / kTileRows : E;
  return past_caches && (long long)row_tiles * ((cols + kWideTileNb - 1) / kWideTileNb) >= 4 * kCus;
}
// bf16 weights past the caches: whether the rows that a GEMM stores go past them as well (store_output has what that
// gains).  Not where few rows are stored and the GEMM is over after a round or two: its end then waits for them and the
// kernel behind would have found them in the caches.  us per moe_experts call, even routing, past / through, gate_up: 16
// experts, 2880 x 2880 (368 tiles), 100 tokens (25 rows) 148.5 / 145.1, 150 155.4 / 153.0, 200 155.0 / 154.2, 300 (75)
// 162 / 171; 20 experts (460 tiles), 90 (18) 164 / 162, 150 (30) 168.9 / 167.6, 200 (40) 169.8 / 172.1; 32 experts, 2048 x 1440 (384 tiles), 150 (19) 111.7 / 108.7, 300 (37) 130.2 / 128.4, 500 (62) 135 / 138; 2880 x
// 2880 (736 tiles), 150 265.5 / 266.3, 400 273 / 293; 8 experts (184 tiles), 70 to 500 within 0.5 %.  Down: 16 experts
// (192 tiles), 150 155.4 / 151.6, 200 155.0 / 152.0, 600 188.0 / 188.0; 32 experts of 2048 x 1440 (256 tiles), 300
// 130.2 / 128.7, 500 135.0 / 135.6; 2880 x 2880 (384 tiles), 150 265.5 / 267.8, 400 273 / 278.
inline bool bf16_stores_past(bool gate_up, int tiles, int T, int E) {
  return gate_up ? tiles >= 2 * kCus || T * kTopK > 36 * E : tiles > kCus || T * kTopK > 64 * E;
}
// Row tiles of a plan, and what runs on it.
inline int plan_tile_rows(int T, int E, int H, int IM, bool mxfp4, bool cached) {
  return (mxfp4 ? half_tiles(T, E, 2 * IM) : bf16_half_tiles(T, E, H, IM, cached)) ? kHalfTileRows : kTileRows;
}
// Fixed part of a tile's estimated cost, by which the XCDs' ranges are cut.  It stands for the column
// operand, which a tile streams in full however few rows it has: 8 row blocks' worth with bf16 weights, one
// and a half with MXFP4, which are a quarter of the bytes, and four in the kernels of many rows.  us per moe_experts
// call, means of two to four routings, even or Zipf's (exponent in brackets), 2880 x 2880 unless stated.  bf16, 32 / 64:
// 128 experts, 600 tokens (1.2) 895 / 842, 1000 (0.6) 1075 / 1053, 2000 (1.2) 1270 / 1188, 4000 (1.2) 1598 / 1500, even
// 1164 / 1164; 32 experts, 200 (0.6) 297 / 276, 600 (1.2) 362 / 339, 1000 412 / 394, 1400 457 / 431, even, 256 289 /
// 277, 1000 321 / 313; 8 experts, 400 (1.2) 161 / 153.  Matrices that the caches hold: 512 x 512, 32 experts, 1000
// (1.2; tiles of 128 rows) 34.8 / 33.8, 3000, even, 55.5 / 52.6, (1.2) 54.9 / 55.8; 1024 x 1024, 3000, even, 124 / 119;
// 4 experts, 600 (128 rows) 134 / 134.  MXFP4, 12 / 32: tiles of 256 rows, 8 experts, 128 (1.2) 68.3 / 69.1, 250 104.4 /
// 104.6, even 81.3 / 81.6; gemm.hip with 128, 32 experts, 200 (1.2) 128 / 147, 300 (0.6) 124 / 147, even 124.8 / 125.5;
// 128 experts, 1000 (1.2) 411 / 462, 2000 575 / 629, even, 600 326 / 324, 1000 383 / 378, 2000 491 / 497.
// gemm_fp4.hip, 12 / 20 / 32: 32 experts, 512 (1.2) 183 / 184 / 184, 2000 (0.6) 390 / 389 / 390, 7168 (1.2) 1162 /
// 1156 / 1165, even, 1000 252 / 245 / 246.
//
// Few rounds, bf16: an XCD that gets one tile more than its CUs take at a time begins another
// round, which a cut by cost does not see.  With 64 an XCD of tall tiles had 35 to 40 of the down GEMM's at 32 experts,
// 350 to 500 tokens (1.2), with 32 no more than its 32, and the others 60 of low ones.  So a GEMM of few rounds of
// tiles is cut by 32 where the slowest XCD's time (its rounds times its tiles' mean cost) is expected to be lower.
// Past the caches, up to two rounds, a fixed part of 96 and 2 % predict the measured times best: us per call, 64
// throughout / this: 32 experts, 256 (1.2) 307 / 298, 350 317 / 305, 400 325 / 311, 450 337 / 315, 480 338 / 319, 560 (0.6)
// 326 / 318; 16 experts, 200 (1.2) 175 / 167; 32 experts of 2048 x 1440, 400 (1.2) 143 / 136; over 396 batches of 8 to 128
// experts, 100 to 7000 tokens, no GEMM that this cuts by 32 was slower by more than 1 %; without the 2 % or with more
// rounds some were, by 2 to 10.  Through the caches, where a tile's columns cost it less, up to three rounds, 64 and
// 5 %: 128 experts of 512 x 512, 4000 tokens (1.2) 93.8 / 89.7, 4500 102.6 / 96.2, 5000 107.4 / 100.8, of 800 x 320, 1500,
// even, 67.5 / 62.7; 32 experts of 1024 x 1024, 1000 (0.6) 70.5 / 67.2; over 1356 batches 0.874 to 1.031 of the time with
// 64 throughout.  (32 throughout is as quick on average there, 0.82 to 1.18 from batch to batch: what the last rounds do
// beyond their number is not foreseen.)
inline TileCost plan_tile_cost(int T, int E, int w1_rows, bool mxfp4, bool past_caches) {
  if (mxfp4) return {fp4_many_rows(T, E, w1_rows) ? 32 : 12, 0, 0, 0, 0.f};
  return past_caches ? TileCost{64, 32, 2, 96, 0.98f} : TileCost{64, 32, 3, 64, 0.95f};
}
enum TileKernel { kBf16Tiles /* gemm_bf16.hip */, kFp4Tiles /* gemm.hip */, kFp4ManyTiles /* gemm_fp4.hip */ };
struct TileRoute {
  TileKernel kernel;
  bool past_caches;
};
inline TileRoute tile_route(int T, int E, int w1_rows, bool mxfp4, int tile_rows, bool cached) {
  const bool past_caches = gemm_streams_weights(T, E, mxfp4, tile_rows, cached);
  if (!mxfp4) return {kBf16Tiles, past_caches};
  return {tile_rows == kHalfTileRows && fp4_many_rows(T, E, w1_rows) ? kFp4ManyTiles : kFp4Tiles, past_caches};
}
// Expert matrices up to this many bytes, over all layers of a handle, are read through
// the caches whatever the batch: they then stay in the 256 MB memory-side cache from
// one call to the next, which loads past the caches do not use.  us per moe_experts
// call through / past the caches, 2880 x 2880: MXFP4, 64 tokens, 20 experts (265 MB)
// 56.2 / 61.3, 22 (291 MB) 61.5 / 62.2, 24 (318 MB) 74.1 / 70.1, 32 (423 MB) 90.1 /
// 81.4; bf16, 96 tokens, 4 experts (199 MB) 63.2 / 93.8, 6 (299 MB) 101.7 / 98.2, 8
// 107.1 / 96.2.  Eight layers of 8 experts, 1440 x 1440, called in turn, 24 tokens:
// MXFP4 (211 MB together) 18.7 / 20.7, bf16 (796 MB) 32.3 / 31.2.
constexpr size_t kCachedWeightBytes = (size_t)256 << 20;
// The first GEMM reads the routed token rows of x itself, through rowmap; there is
// no gathered copy.  act holds the activation in the order the second GEMM of the
// same file reads it: MFMA fragments (gemm.hip), quads or rows (stream.hip).
hipError_t launch_gate_up(const uint16_t *x, const void *w1, const uint16_t *w1_scale, const float *b1g,
                          const float *b1u, const DispatchBuffers &d, uint16_t *act, int H, int IM,
                          float limit, int T, int E, int tile_rows, bool wide, bool cached, hipStream_t s);
hipError_t launch_down(const uint16_t *act, const void *w2, const uint16_t *w2_scale, const float *b2,
                       const DispatchBuffers &d, float *y, int H, int IM, int T, int E, int tile_rows,
                       bool wide, bool cached, hipStream_t s);
// bf16 weights (gemm_bf16.hip; launch_gate_up and launch_down call them), a plan of either height.
// stream: weights past the caches.
hipError_t launch_bf16_gate_up(const uint16_t *x, const void *w1, const float *b1g, const float *b1u,
                               const DispatchBuffers &d, uint16_t *act, int H, int IM, float limit, int T, int E,
                               int tile_rows, bool wide, bool stream, hipStream_t s);
hipError_t launch_bf16_down(const uint16_t *act, const void *w2, const float *b2, const DispatchBuffers &d, float *y,
                            int H, int IM, int T, int E, int tile_rows, bool wide, bool stream, hipStream_t s);
// MXFP4 weights with many rows per expert (gemm_fp4.hip; likewise), a plan of kHalfTileRows, which is never a wide one.
hipError_t launch_fp4_gate_up(const uint16_t *x, const void *w1, const uint16_t *w1_scale, const float *b1g,
                              const float *b1u, const DispatchBuffers &d, uint16_t *act, int H, int IM, float limit,
                              int T, int E, bool stream, hipStream_t s);
hipError_t launch_fp4_down(const uint16_t *act, const void *w2, const uint16_t *w2_scale, const float *b2,
                           const DispatchBuffers &d, float *y, int H, int IM, int T, int E, bool stream, hipStream_t s);
// tiles: row tiles, at most (stream_direct_tile_cap with ids.topk_i, otherwise stream_tile_cap).
// T, E: tokens and experts of the batch, the same for both (the order of act between them follows from these).
// cached: kCachedWeightBytes.
hipError_t launch_stream_gate_up(const uint16_t *x, const void *w1, const uint16_t *w1_scale, const float *b1g,
                                 const float *b1u, const DispatchBuffers &d, uint16_t *act, int H, int IM,
                                 float limit, int tiles, int T, int E, bool cached, const DirectIds &ids, hipStream_t s);
hipError_t launch_stream_down(const uint16_t *act, const void *w2, const uint16_t *w2_scale, const float *b2,
                              const DispatchBuffers &d, float *y, int H, int IM, int tiles, int T, int E,
                              bool cached, const DirectIds &ids, hipStream_t s);
// ldy: floats per row of y (the padded hidden size)
hipError_t launch_combine(const float *y, int ldy, const int *inv, const float *topk_v, const int *pos, float *out,
                          int T, int H, int accumulate, hipStream_t s);
hipError_t launch_combine_residual(const float *y, int ldy, const int *inv, const float *topk_v, const int *pos,
                                   uint16_t *x, int T, int H, hipStream_t s);
// Whether the norm takes a wave per token instead of a workgroup: rows that a wave's registers
// hold, and of those beyond one piece per thread only with tokens enough for a workgroup on every
// CU.  moe_block_forward, wave / workgroup: 7168 tokens, 64 columns 46.5 / 51.5 us, 256 0.93, 512 0.95, 1024
// 0.98 of the time; 768 to 1024 columns, 2000 tokens 0.98, 1000 0.99, 8 to 64 tokens 1.02 to 1.03.
constexpr int kNormHeld = 2;  // 16-byte pieces of the row per thread
inline bool norm_wave_per_token(int T, int H) { return H <= 64 * 8 || (H <= 64 * 8 * kNormHeld && T >= 4 * kCus); }
hipError_t launch_rmsnorm(const uint16_t *x, const float *weight, const int *pos, uint16_t *t_out,
                          int T, int H, hipStream_t s);

}  // namespace moe

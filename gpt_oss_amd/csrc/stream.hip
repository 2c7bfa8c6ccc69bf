// Grouped expert GEMMs of the batches in which the weights are a stream: few rows
// per expert, so the time is that of reading the weights once.  Same contract as
// the kernels of gemm.hip, gemm_bf16.hip and gemm_fp4.hip (matmul/matmul.cpp:1023-1914, SwiGLU of run.cpp:709-726).
//
// A wave owns a pair of column blocks (64 columns) of one expert and a slice of
// the reduction, and shares nothing with other waves until its slice is done: the
// weights and the token rows go straight into registers, D steps of 32 k ahead,
// there is no barrier and no DMA in the loop.  The KW waves of a
// workgroup take the KW slices of the same columns and add their sums through
// LDS at the end, in a fixed order.  Compared with one workgroup per 256 columns
// whose waves walk the whole reduction in lock step (gemm_tile), a wave's chain
// of dependent steps is KW times shorter, there are KW times as many streams,
// and a late load holds up one wave instead of four.
//
// The products are v_mfma_f32_16x16x32_bf16: 16 token rows at a time, which is
// what an expert has in such a batch.  The weights are the first operand, so a
// lane ends with four consecutive weight rows of one token.  Lane l = 16 q + r of
// either operand holds row r and the 8 k of piece (q >> 1) + 2 (q & 1) of the
// step's four: that is the order in which one v_permlane16_swap turns a pair of
// 32-row weight fragments (pack.hip) into two 16-row ones.
//
// Bound by HBM with bf16 weights; with MXFP4 weights the rows' loads through L1 (64 tokens, 32 experts: 92 us
// per call, 87 without them), the scales' (88) and the few microseconds in which a launch fills and drains
// show as well; the conversions do not (91.6).  Measured at 2880 x 2880 and 32 experts, against the kernels this
// replaced (us, gate_up + down): 24 tokens bf16, 30 experts named, 147 + 79 (6.8 and
// 6.3 TB/s of weights; were 194 + 102), 64 tokens MXFP4 52 + 28 (were 59 + 39), 1
// token MXFP4 10 + 6 (were 23 + 14).  What that rests on, by leaving it out, measured on a
// batch that named all 32 experts (157 + 81; MXFP4 50 + 29): the weights' non-temporal
// loads (bf16 174 + 90 with plain ones), two pairs of columns per wave that share the
// rows they load (MXFP4 55 + 32 with one; kStreamTwoPairs), no refill loads past the slice's end
// (MXFP4 57 + 32 with them).  The number of slices (1, 2 or 4) matters to the
// small launches only.
//
// Every path a batch can take at its size (whole layer, caller's routing, stage
// by stage; bf16 and MXFP4 weights) runs these kernels with the same slices, so
// they all give the same bits.
#include <type_traits>

#include "moe_internal.h"
#include "swiglu.h"

namespace moe {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

constexpr int kStreamKw = 4;     // waves of a workgroup = slices of the reduction
constexpr int kStreamCols = 64;  // columns of a pair of column blocks
constexpr int kStreamRows = 32;  // rows of a tile, at most
// MXFP4: with this many column tiles of one pair or more, and more than this many
// tokens, a wave takes two pairs.  What they save are loads of rows, which are few in a
// batch of a few tokens, and with half as many workgroups the last ones leave more CUs
// idle.  us per moe_experts call, one pair / two, even routing: 128 experts, 6 tokens
// 54.9 / 60.1, 24: 136.4 / 140.8, 64: 219 / 218, 128: 277.6 / 268.5; Zipf's (exponent
// 1.2) 6: 39.3 / 42.4, 24: 89 / 89, 32: 95.6 / 91.8, 64: 164.6 / 156.8; 32 experts, 6
// tokens 45.6 / 47.5, 24: 73.2 / 73.5, 48: 78.9 / 77.2, 128: 114.4 / 100.6; 16 experts, 24
// tokens 41.1 / 43.5, 64: 47.6 / 48.7.  Few column tiles, eight layers of 8 experts: 24
// tokens (900 in gate_up) 33.9 / 34.2, 32 (990) 37.3 / 37.7, 48 (1170) 42.6 / 41.3.
constexpr int kStreamTwoPairs = 1024, kStreamTwoPairsTokens = 24;
// Order of act between the two GEMMs: in quads (act_place) from this many rows per
// expert on; with fewer in rows, whose pieces then stand in fewer cache lines.  us per
// moe_experts call, rows / quads, MXFP4: 128 experts, 24 tokens (0.75 rows per expert)
// 140.8 / 143.1, 64 (2): 220 / 222, 256 (8): 305 / 302; 32 experts, 48 (6): 77.1 /
// 76.6, 128 (16): 103.8 / 100.8; 8 experts, 32 (16): 39.0 / 36.7, 64 (32): 48.6 / 42.9.
// bf16 gains less: 8 experts, 64 tokens 92.6 / 87.8.
constexpr int kStreamQuadRows = 6;

// Orders LDS traffic only: the loads in flight stay in flight.
__device__ __forceinline__ void stream_barrier() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }

// 16 bytes of weights: past the caches where one workgroup reads them and they are not
// there from the call before (measured, see above), through them where several do at
// about the same time (share_of) or all weights fit (kCachedWeightBytes).
template <bool CACHED>
__device__ __forceinline__ u32x4 load_weights(const char *g) {
  const u32x4 *v = reinterpret_cast<const u32x4 *>(g);
  if constexpr (CACHED) return *v;
  return __builtin_nontemporal_load(v);
}

// Place of workgroup l of an expert with nb tiles of rows and wgs tiles of columns:
// eight column tiles at a time, their first row tiles, then their second ones, and
// so on.  Workgroup ids are dealt round-robin to the XCDs, so the row tiles that
// read the same weights run at about the same time on one XCD and the weights come
// from HBM once.  With a row tile's workgroups wgs ids apart and every load past the
// caches each tile fetched them for itself: 128 experts, bf16, Zipf routing (exponent
// 1.2), us per moe_experts call at 256 tokens 958, with this order 888, at 512 tokens
// 1294 and 1130; MXFP4 301 and 279, 415 and 380; even routing within 1 %.
__device__ __forceinline__ void share_of(int l, int wgs, int nb, int &col, int &blk) {
  col = l;
  blk = 0;
  if (nb == 1) return;
  const int g = l / (kXcds * nb), r = l - g * kXcds * nb;
  const int width = min(kXcds, wgs - g * kXcds);
  blk = r / width;
  col = g * kXcds + r - blk * width;
}

// The L1 serves four adjacent lanes at a time, 64 contiguous bytes in one access.  In
// operand order adjacent lanes hold different rows, and a load of 16 rows of 64 bytes
// takes 52 accesses (counted) instead of 16.  So, where there are more than a few rows,
//   * token rows are loaded with four adjacent lanes to a row and put in operand order
//     through a kilobyte of LDS that only the wave touches (STAGED; tiles of more than
//     16 rows: below, the weights' loads are the more).  8 experts, 64 tokens, us per
//     moe_experts call without / with: bf16 90.7 / 87.9, MXFP4 43.5 / 42.6;
//   * gate_up leaves the activation in "quads" for the down GEMM (kStreamQuadRows):
//     per 16 rows and step of 32 k a kilobyte, in it the pieces of 8 k of four rows side
//     by side.  The byte of piece `piece` of row r:
__device__ __forceinline__ uint32_t act_place(int r, int piece) { return (r >> 2) * 256u + piece * 64u + (r & 3) * 16u; }

// One wave's share of a tile: RG groups of 16 rows times NP pairs of column
// blocks over the steps [ks0, ks0 + n) of 32 k.  a_rows: rows of lda 16-byte
// pieces; row[g]: the row this lane loads in group g.  np_valid: pairs inside
// the matrix; one past it repeats the first, and its sums are not used.
// stage: RG KB of LDS that only this wave touches (STAGED).  QUADS: a_rows is an
// activation in quads.
template <int NP, int RG, int D, bool FP4, bool CACHED, bool STAGED, bool QUADS>
__device__ __forceinline__ void stream_slice(const uint4 *__restrict__ a_rows, int lda, const int (&row)[RG],
                                             const uint4 *__restrict__ w, const uint16_t *__restrict__ ws, int KB,
                                             int np_valid, int ks0, int n, int lane, f32x4 *stage,
                                             f32x4 (&acc)[NP][4][RG]) {
  constexpr int WR = FP4 ? 1 : 4;  // 16-byte registers of weights per pair and step
  const int r = lane & 15, q = lane >> 4;
  const int piece = (q >> 1) + 2 * (q & 1);
  // STAGED: lane 4 r + c loads piece (c - r / 4) % 4 of row r and writes it at its own
  // place; the reads of one piece of 16 rows then fall on 16 different slots of 256 bytes.
  const int own = ((lane & 3) - q) & 3, staged_at = 4 * r + ((piece + (r >> 2)) & 3);
  // addresses: a base that is the same for the whole wave and moves with the step,
  // plus an offset per lane that does not.  The rows' is 64 bits wide: the fixed
  // slots of 256 experts reach 4 GiB from an intermediate size of 131 600 on.
  size_t a_off[RG];
#pragma unroll
  for (int g = 0; g < RG; g++)
    a_off[g] = QUADS ? (size_t)(row[g] >> 4) * lda * 256 + act_place(row[g] & 15, piece)
                     : ((size_t)row[g] * lda + (STAGED ? own : piece)) * 16;
  // bf16: fragment (block b, k block kb) is 64 pieces; this lane's piece of half hh is
  // kb = q & 1, (q >> 1) * 32 + 16 hh + r.  FP4: one chunk of 64 pieces per step.
  const uint32_t w_off = FP4 ? lane * 16u : ((q & 1) * 64 + (q >> 1) * 32 + r) * 16u;
  // scale bytes of a step: 16 bits per row; loaded as the 32 bits of two rows, of which the lane shifts its own down
  const uint32_t s_off = (lane & 30) * 2u, s_shift = (lane & 1) * 16u;
  u32x4 wq[D][NP][WR], xa[D][RG];
  uint32_t sc[D][NP];
  auto load = [&](int d, int s) {
    const size_t k = ks0 + s;
#pragma unroll
    for (int p = 0; p < NP; p++) {
      const size_t pair = p < np_valid ? p : 0;
      if (FP4) {
        const char *wb = reinterpret_cast<const char *>(w) + pair * KB * 512 + k * 1024;
        const char *sb = reinterpret_cast<const char *>(ws) + pair * KB * 32 + k * 64;
        wq[d][p][0] = load_weights<CACHED>(wb + w_off);
        sc[d][p] = *reinterpret_cast<const uint32_t *>(sb + s_off);
      } else {
        const char *wb = reinterpret_cast<const char *>(w) + pair * KB * 2048 + k * 2048;
#pragma unroll
        for (int i = 0; i < 4; i++)
          wq[d][p][i] = load_weights<CACHED>(wb + (size_t)(i >> 1) * KB * 1024 + (i & 1) * 256 + w_off);
      }
    }
    const char *ab = reinterpret_cast<const char *>(a_rows) + k * (QUADS ? 1024 : 64);
#pragma unroll
    for (int g = 0; g < RG; g++) xa[d][g] = *reinterpret_cast<const u32x4 *>(ab + a_off[g]);
  };
#pragma unroll
  for (int p = 0; p < NP; p++)
#pragma unroll
    for (int i = 0; i < 4; i++)
#pragma unroll
      for (int g = 0; g < RG; g++) acc[p][i][g] = f32x4{0.f, 0.f, 0.f, 0.f};
  auto compute = [&](int d) {
    u32x4 xf[RG];
    if constexpr (STAGED) {
      // (the LDS instructions of a wave are carried out in their order)
#pragma unroll
      for (int g = 0; g < RG; g++) stage[g * 64 + lane] = __builtin_bit_cast(f32x4, xa[d][g]);
      __builtin_amdgcn_wave_barrier();
#pragma unroll
      for (int g = 0; g < RG; g++) xf[g] = __builtin_bit_cast(u32x4, stage[g * 64 + staged_at]);
      __builtin_amdgcn_wave_barrier();
    } else {
#pragma unroll
      for (int g = 0; g < RG; g++) xf[g] = xa[d][g];
    }
#pragma unroll
    for (int p = 0; p < NP; p++) {
      bf16x8 wf[4];  // 16 weight rows each: [2 * block + half]
      if constexpr (FP4) {
        const uint32_t own = sc[d][p] >> s_shift;
        const u32x2 ss = __builtin_amdgcn_permlane16_swap(own, own, false, false);
#pragma unroll
        for (int b = 0; b < 2; b++) {
          const u32x2 nn = __builtin_amdgcn_permlane16_swap(wq[d][p][0][2 * b], wq[d][p][0][2 * b + 1], false, false);
#pragma unroll
          for (int hh = 0; hh < 2; hh++) {
            const float scale = __uint_as_float(((ss[hh] >> (8 * b)) & 0xffu) << 23);  // 2^(s - 127)
            const uint32_t nib = nn[hh];
            const bf16x2 p0 = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp4(nib, scale, 0);
            const bf16x2 p1 = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp4(nib, scale, 1);
            const bf16x2 p2 = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp4(nib, scale, 2);
            const bf16x2 p3 = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp4(nib, scale, 3);
            wf[2 * b + hh] = bf16x8{p0[0], p0[1], p1[0], p1[1], p2[0], p2[1], p3[0], p3[1]};
          }
        }
      } else {
#pragma unroll
        for (int i = 0; i < 4; i++) wf[i] = __builtin_bit_cast(bf16x8, wq[d][p][i]);
      }
#pragma unroll
      for (int i = 0; i < 4; i++)
#pragma unroll
        for (int g = 0; g < RG; g++)
          acc[p][i][g] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wf[i], __builtin_bit_cast(bf16x8, xf[g]),
                                                                 acc[p][i][g], 0, 0, 0);
    }
  };
  if (n <= 0) return;  // a short reduction has fewer steps than slices
  // Rounds of D steps.  The refill of a round is the next round's loads, so the
  // last one has none; the steps that pad it load the slice's last step again (at
  // most D - 1 of them, real traffic: the loads go past the caches) and are not
  // multiplied.
#pragma unroll
  for (int d = 0; d < D; d++) load(d, min(d, n - 1));
  int s = 0;
  for (; s + D < n; s += D) {
#pragma unroll
    for (int d = 0; d < D; d++) {
      compute(d);
      load(d, min(s + d + D, n - 1));
      __builtin_amdgcn_sched_barrier(0);
    }
  }
#pragma unroll
  for (int d = 0; d < D; d++)
    if (s + d < n) compute(d);
}

// Sum of the slices in their order, bias, SwiGLU and the rows out.  A unit is 16
// columns (gate_up: 16 of gate and the same 16 of up) of one group of rows, in
// which a lane holds four consecutive columns of one row; the waves share them.
template <int RG, bool GATE_UP, bool QUADS>
__device__ __forceinline__ void stream_finish(const f32x4 *part, const float *__restrict__ bias_a,
                                              const float *__restrict__ bias_b, int P, int row0, int rows,
                                              void *__restrict__ outp, int ldo, float limit, int w, int lane) {
  const int r = lane & 15, q = lane >> 4;
  auto sum = [&](int i, int g) {
    f32x4 v = part[(i * RG + g) * 64 + lane];
#pragma unroll
    for (int k = 1; k < kStreamKw; k++) v += part[((k * 4 + i) * RG + g) * 64 + lane];
    return v;
  };
  constexpr int UNITS = (GATE_UP ? 2 : 4) * RG;
  for (int u = w; u < UNITS; u += kStreamKw) {
    const int i = u / RG, g = u % RG;
    const int row = 16 * g + r;
    if (GATE_UP) {
      const int j = kRowBlock * P + 16 * i + 4 * q;
      const f32x4 bg = *reinterpret_cast<const f32x4 *>(bias_a + j), bu = *reinterpret_cast<const f32x4 *>(bias_b + j);
      const f32x4 ga = sum(i, g) + bg, up = sum(2 + i, g) + (bu + 1.0f);
      const uint32_t lo = pack_bf16(swiglu_shifted(ga[0], up[0], limit), swiglu_shifted(ga[1], up[1], limit));
      const uint32_t hi = pack_bf16(swiglu_shifted(ga[2], up[2], limit), swiglu_shifted(ga[3], up[3], limit));
      // QUADS: columns [32 P, 32 P + 32) are a step of the down GEMM, these half of its piece 2 i + q / 2
      const int ar = row0 + row;
      const size_t at = QUADS ? ((size_t)(ar >> 4) * (ldo / 32) + P) * 1024 + act_place(ar & 15, 2 * i + (q >> 1)) + 8 * (q & 1)
                              : ((size_t)ar * ldo + j) * 2;
      if (row < rows) *reinterpret_cast<uint2 *>(static_cast<char *>(outp) + at) = make_uint2(lo, hi);
    } else {
      const int j = kStreamCols * P + 16 * i + 4 * q;
      const f32x4 v = sum(i, g) + *reinterpret_cast<const f32x4 *>(bias_a + j);
      if (row < rows) *reinterpret_cast<f32x4 *>(static_cast<float *>(outp) + (size_t)(row0 + row) * ldo + j) = v;
    }
  }
}

// The ti-th expert that has rows (-1: there are fewer).  mine: the expert of the
// assignment of thread tid, -1: none.  some: LDS.
__device__ __forceinline__ void find_expert(unsigned long long *some, int mine, int ti, int E, int tid, int &e,
                                            int &first, int &nb) {
  uint32_t *mask = reinterpret_cast<uint32_t *>(some);
  if (tid < 2 * kStreamKw) mask[tid] = 0;
  stream_barrier();
  if (mine >= 0) atomicOr(&mask[mine >> 5], 1u << (mine & 31));
  stream_barrier();
  e = -1;
  int left = ti;
  for (int ww = 0; ww < (E + 31) / 32; ww++) {
    uint32_t m = __builtin_amdgcn_readfirstlane(mask[ww]);
    const int c = __builtin_popcount(m);
    if (left < c) {
      for (int i = 0; i < left; i++) m &= m - 1;
      e = ww * 32 + __builtin_ctz(m);
      break;
    }
    left -= c;
  }
  e = __builtin_amdgcn_readfirstlane(e);
  first = ti;
  nb = 1;
}

// The same where an expert with more than 32 rows counts as two tiles: the expert of
// the ti-th tile, its first tile and its tiles.  The tiles follow each other without
// gaps: with two places for every expert the workgroups without work stand between
// the others, and the CUs they are dealt to stay idle (8 experts, 48 tokens, MXFP4:
// 54.1 us per moe_experts call instead of 42.6).
__device__ __forceinline__ void find_tile(int *hist, unsigned long long *some, unsigned long long *more, int mine,
                                          int ti, int tid, int &e, int &first, int &nb) {
  static_assert(kDirectSlotRows <= 2 * kStreamRows, "two tiles per expert, at most");
  const int lane = tid & 63;
  hist[tid] = 0;  // expert -> rows
  stream_barrier();
  if (mine >= 0) atomicAdd(&hist[mine], 1);
  stream_barrier();
  {
    const int rows = hist[tid];
    const unsigned long long s = __ballot(rows > 0), m = __ballot(rows > kStreamRows);
    if (lane == 0) {
      some[tid >> 6] = s;
      more[tid >> 6] = m;
    }
  }
  stream_barrier();
  e = -1;
  first = 0;
  nb = 1;
  const unsigned long long below = (1ull << lane) - 1ull;
#pragma unroll
  for (int ww = 0; ww < kStreamKw; ww++) {
    const unsigned long long s = some[ww], m = more[ww];
    const int tiles = __builtin_amdgcn_readfirstlane(__popcll(s) + __popcll(m));
    if (e < 0 && ti < first + tiles) {
      // lane: expert 64 ww + lane
      const int at = first + __popcll(s & below) + __popcll(m & below);
      const int have = (int)(s >> lane & 1) + (int)(m >> lane & 1);
      const int l = __builtin_ctzll(__ballot(at <= ti && ti < at + have));
      e = ww * 64 + l;
      first = __builtin_amdgcn_readlane(at, l);
      nb = __builtin_amdgcn_readlane(have, l);
    } else if (e < 0) {
      first += tiles;
    }
  }
}

// DIRECT: there is no plan.  The workgroup reads the batch's ids (one per
// thread), finds the expert of its tile and by ballot that expert's rows; workgroup
// i * wgs + c is column tile c of tile i, so that the column tiles of the few experts a
// small batch reaches spread over all XCDs.  Otherwise a tile is a row block of the
// plan's padded rows.  tiles: tiles of rows, at most.  cached: the weights are read
// through the caches (also those that several tiles of rows read).
template <int NP, bool GATE_UP, bool FP4, bool DIRECT, bool QUADS>
__global__ __launch_bounds__(kStreamKw * 64, NP == 1 ? 4 : 3) void stream_gemm_kernel(
    const uint4 *__restrict__ a_rows, const uint4 *__restrict__ w_frag, const uint16_t *__restrict__ w_scale,
    const float *__restrict__ bias_a, const float *__restrict__ bias_b, const int *__restrict__ rowmap,
    const int *__restrict__ blk_expert, const int *__restrict__ totals, int *__restrict__ inv,
    void *__restrict__ outp, int K, int N, float limit, int tiles, bool cached, DirectIds ids) {
  constexpr int RG = kStreamRows / 16;
  __shared__ f32x4 part[kStreamKw * 4 * RG * 64];
  __shared__ int rows_sh[DIRECT ? kDirectSlotRows : kStreamRows];  // row of the tile -> token
  const int tid = threadIdx.x;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int n_cols = GATE_UP ? 2 * N : N;
  const int pairs = n_cols / kStreamCols;
  const int wgs = (pairs + NP - 1) / NP;
  const int KB = K / kFragK, steps = K / 32;
  const int per = (steps + kStreamKw - 1) / kStreamKw;
  const int ks0 = min(w * per, steps), n = min(per, steps - ks0);
  int e, row0, count, col;
  int r0 = 0;  // the tile's first row among those from row0
  if constexpr (DIRECT) {
    static_assert(kStreamKw * 64 == kDirectTokens * kTopK, "one thread per assignment");
    __shared__ int hist[256], cnt[kStreamKw];
    __shared__ unsigned long long some[kStreamKw], more[kStreamKw];
    const int lane = tid & 63;
    const int mine = direct_expert_of(ids, tid);
    const int ti = blockIdx.x / wgs;
    // the first column tile's workgroups also write where each assignment's row is, for the combine
    if (GATE_UP && blockIdx.x == 0 && mine < 0 && tid < ids.T * kTopK) inv[tid] = -1;
    int first, nb;  // the expert's first tile and its tiles
    if (ids.T * kTopK <= kStreamRows) {  // no expert has a second tile, whatever the ids
      find_expert(some, mine, ti, ids.E, tid, e, first, nb);
    } else {
      find_tile(hist, some, more, mine, ti, tid, e, first, nb);
    }
    if (e < 0) return;  // fewer tiles than the grid provides for
    int blk;
    share_of(blockIdx.x - first * wgs, wgs, nb, col, blk);
    cached |= nb > 1;
    r0 = blk * kStreamRows;
    const bool writes_inv = GATE_UP && col == 0 && blk == 0;
    const unsigned long long bal = __ballot(mine == e);
    if (lane == 0) cnt[w] = __popcll(bal);
    stream_barrier();
    int before = 0;
    count = 0;
#pragma unroll
    for (int ww = 0; ww < kStreamKw; ww++) {
      const int c = cnt[ww];
      if (ww < w) before += c;
      count += c;
    }
    count = __builtin_amdgcn_readfirstlane(min(count, kDirectSlotRows));
    row0 = e * kDirectSlotRows;
    if (GATE_UP) {
      const int at = before + __popcll(bal & ((1ull << lane) - 1ull));
      if (mine == e && at < kDirectSlotRows) rows_sh[at] = tid / kTopK;
      if (mine == e && writes_inv) inv[tid] = at < kDirectSlotRows ? row0 + at : -1;
      stream_barrier();
    }
  } else {
    // Row block ti is one of an expert's: its blocks (those among the 64 from `from`)
    // stand in a row and share the wgs workgroups of each (share_of).
    const int ti = blockIdx.x / wgs, from = ti & ~63;
    const int lane = tid & 63;
    const int n_blk = totals[kTotRows] / kRowBlock;
    const int be = blk_expert[min(from + lane, tiles - 1)];
    int a = lane < kStreamRows ? rowmap[ti * kRowBlock + lane] : -1;  // asked for before it is known to be the one
    if (ti >= n_blk) return;  // surplus workgroups of the upper-bound grid
    e = __builtin_amdgcn_readlane(be, ti & 63);
    const unsigned long long own = __ballot(be == e && from + lane < n_blk);
    const int first = from + __builtin_ctzll(own), nb = __popcll(own);
    int blk;
    share_of(blockIdx.x - first * wgs, wgs, nb, col, blk);
    cached |= nb > 1;
    row0 = (first + blk) * kRowBlock;
    if (first + blk != ti) a = lane < kStreamRows ? rowmap[row0 + lane] : -1;
    count = __popcll(__ballot(a >= 0));  // the valid rows of a block come first
    if (GATE_UP) {
      if (w == 0 && lane < count) rows_sh[lane] = a / kTopK;
      stream_barrier();
    }
  }
  const int P = col * NP, np_valid = min(NP, pairs - P);
  const size_t blk0 = (size_t)e * (n_cols / kRowBlock) + 2 * P;
  const uint4 *wp = w_frag + blk0 * (size_t)(KB * (FP4 ? 16 : 64));
  const uint16_t *sp = FP4 ? w_scale + blk0 * KB * 8 : nullptr;
  const float *ba = bias_a + (size_t)e * N;
  const float *bb = GATE_UP ? bias_b + (size_t)e * N : nullptr;
  const int lane = tid & 63, rows = min(count - r0, kStreamRows);
  auto tile = [&](auto g_c, auto d_c, auto cached_c) {
    constexpr int G = decltype(g_c)::value;
    constexpr bool kStaged = GATE_UP && G > 1;
    // lanes past the last row repeat it; their sums are not stored
    int row[G];
#pragma unroll
    for (int g = 0; g < G; g++) {
      const int rr = r0 + min(16 * g + (kStaged ? lane >> 2 : lane & 15), rows - 1);
      row[g] = GATE_UP ? rows_sh[rr] : row0 + rr;
    }
    f32x4 acc[NP][4][G];
    stream_slice<NP, G, decltype(d_c)::value, FP4, decltype(cached_c)::value, kStaged, !GATE_UP && QUADS>(
        a_rows, K / 8, row, wp, sp, KB, np_valid, ks0, n, lane, part + w * (4 * RG * 64), acc);
#pragma unroll
    for (int p = 0; p < NP; p++) {
      if (p >= np_valid) break;
      if (p) stream_barrier();  // the sums before have been read
#pragma unroll
      for (int i = 0; i < 4; i++)
#pragma unroll
        for (int g = 0; g < G; g++) part[((w * 4 + i) * G + g) * 64 + lane] = acc[p][i][g];
      stream_barrier();
      stream_finish<G, GATE_UP, QUADS>(part, ba, bb, P + p, row0 + r0, rows, outp, N, limit, w, lane);
    }
  };
  // steps ahead: as many as the registers of three or four waves per SIMD hold (more gain
  // nothing: at 64 tokens and 32 experts, MXFP4, the same time with 4, 6 and 8; fewer cost:
  // two pairs of columns and up to 32 rows, 16 experts and 64 tokens, 2 steps 56.7 us per
  // moe_experts call, 3 steps 55.3)
  using One = std::integral_constant<int, 1>;
  using Two = std::integral_constant<int, 2>;
  using DeepTwo = std::integral_constant<int, FP4 ? (NP == 1 ? 4 : 3) : 3>;
  using DeepOne = std::integral_constant<int, FP4 ? (NP == 1 ? 6 : 4) : 4>;
  if (rows > 16) {
    if (cached) tile(Two{}, DeepTwo{}, std::true_type{}); else tile(Two{}, DeepTwo{}, std::false_type{});
  } else {
    if (cached) tile(One{}, DeepOne{}, std::true_type{}); else tile(One{}, DeepOne{}, std::false_type{});
  }
}

template <int NP, bool GATE_UP>
static hipError_t launch_stream_np(const uint4 *a, const uint4 *w, const uint16_t *w_scale, const float *ba,
                                   const float *bb, const DispatchBuffers &d, void *out, int K, int N, float limit,
                                   int tiles, int T, int E, bool cached, const DirectIds &ids, hipStream_t s) {
  const int pairs = (GATE_UP ? 2 * N : N) / kStreamCols;
  const int grid = tiles * ((pairs + NP - 1) / NP);
#define MOE_STREAM(FP4, DIRECT)                                                              \
  do {                                                                                       \
    if (T * kTopK >= kStreamQuadRows * E)                                                    \
      stream_gemm_kernel<NP, GATE_UP, FP4, DIRECT, true><<<grid, kStreamKw * 64, 0, s>>>(    \
          a, w, w_scale, ba, bb, d.rowmap, d.blk_expert, d.totals, d.inv, out, K, N, limit,  \
          tiles, cached, ids);                                                               \
    else                                                                                     \
      stream_gemm_kernel<NP, GATE_UP, FP4, DIRECT, false><<<grid, kStreamKw * 64, 0, s>>>(   \
          a, w, w_scale, ba, bb, d.rowmap, d.blk_expert, d.totals, d.inv, out, K, N, limit,  \
          tiles, cached, ids);                                                               \
  } while (0)
  if constexpr (NP == 1) {
    if (!w_scale) {
      if (ids.topk_i) MOE_STREAM(false, true); else MOE_STREAM(false, false);
      return hipGetLastError();
    }
  }
  if (ids.topk_i) MOE_STREAM(true, true); else MOE_STREAM(true, false);
#undef MOE_STREAM
  return hipGetLastError();
}

template <bool GATE_UP>
static hipError_t launch_stream(const void *a, const void *w, const uint16_t *w_scale, const float *ba,
                                const float *bb, const DispatchBuffers &d, void *out, int K, int N, float limit,
                                int tiles, int T, int E, bool cached, const DirectIds &ids, hipStream_t s) {
  const uint4 *af = static_cast<const uint4 *>(a), *wf = static_cast<const uint4 *>(w);
  const int pairs = (GATE_UP ? 2 * N : N) / kStreamCols;
  if (w_scale && tiles * pairs >= kStreamTwoPairs && T > kStreamTwoPairsTokens)
    return launch_stream_np<2, GATE_UP>(af, wf, w_scale, ba, bb, d, out, K, N, limit, tiles, T, E, cached, ids, s);
  return launch_stream_np<1, GATE_UP>(af, wf, w_scale, ba, bb, d, out, K, N, limit, tiles, T, E, cached, ids, s);
}

hipError_t launch_stream_gate_up(const uint16_t *x, const void *w1, const uint16_t *w1_scale, const float *b1g,
                                 const float *b1u, const DispatchBuffers &d, uint16_t *act, int H, int IM,
                                 float limit, int tiles, int T, int E, bool cached, const DirectIds &ids, hipStream_t s) {
  return launch_stream<true>(x, w1, w1_scale, b1g, b1u, d, act, H, IM, limit, tiles, T, E, cached, ids, s);
}

hipError_t launch_stream_down(const uint16_t *act, const void *w2, const uint16_t *w2_scale, const float *b2,
                              const DispatchBuffers &d, float *y, int H, int IM, int tiles, int T, int E,
                              bool cached, const DirectIds &ids, hipStream_t s) {
  return launch_stream<false>(act, w2, w2_scale, b2, nullptr, d, y, IM, H, 0.f, tiles, T, E, cached, ids, s);
}

}  // namespace moe

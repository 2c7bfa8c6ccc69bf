// Grouped expert GEMMs with MXFP4 weights on the bf16 matrix cores
// (v_mfma_f32_32x32x16_bf16, fp32 accumulate).  Replaces mlp1_kernel / mlp1_120b_kernel
// (matmul/matmul.cpp:1023-1465) with the clamped SwiGLU in the epilogue
// (utility/utility.cpp:1108-1125; formula of run.cpp:709-726) and
// mlp2_kernel_noatomic / mlp2_120b_kernel (matmul/matmul.cpp:1470-1914).
//
// Data layout.  The weights and the activation between the two GEMMs are kept
// as ready-made MFMA fragments of 1 KB (64 lanes x 8 bf16, see pack.hip and the
// gate_up epilogue), ordered [row block of 32][k block of 16]: every global load
// is a contiguous 16 bytes per lane and is already in register order.  The row
// operand of gate_up is the token rows themselves, bf16 row-major, found through
// the dispatch's row map: there is no gathered copy (gemm_tile_gl).
//
// Batches with few rows per expert run the kernels of stream.hip instead, bf16 weights
// those of gemm_bf16.hip, and MXFP4 weights with many rows per expert those of gemm_fp4.hip.
//
// Tiling.  A workgroup of NW waves owns a tile of (RBT*32) rows x
// (NW*NBW*32) columns of one expert.  The waves split the columns only: each
// wave keeps RBT x NBW accumulators of 32x32 over all rows of the tile, RBT =
// 1..8 following the expert's row count (see build_plan in dispatch.hip), so a ragged
// segment pads to at most 31 rows and MFMA work follows the real rows.
//
// Feeding the matrix cores.  Many bytes are kept in flight:
//   * the row operand (shared by all waves) goes straight into an R-stage LDS
//     ring by DMA (global_load_lds_dwordx4), R-1 steps ahead of the MFMAs;
//   * the column operand is private to a wave in this layout, so it never
//     touches LDS: it is loaded into an R-slot ring of VGPRs, R-1 steps ahead.
// R is 4 (measured against 3, 5, 6 and 7 on bf16 weights, which these kernels ran as
// well: a deeper ring gains nothing in the main loop and its longer fill costs at the
// start of every tile; with 3 the main loop starves).  These loads
// complete in the order they were issued, so waiting for "all but the newest n"
// (s_waitcnt vmcnt(n)) picks out exactly the step that is needed next and
// leaves the later ones in flight.
//
// Tile order.  Workgroup ids are dealt round-robin to the 8 XCDs, each with
// its own L2.  Logical tile ids are laid out (expert, group of up to four row
// tiles, column tile, row tile) with the row tile fastest, and XCD x takes a
// contiguous range of them (see build_plan and write_expert_tiles: about an
// eighth by estimated cost): the tiles an XCD runs at one time share a few row
// tiles of the expert and a few column slabs of its weights.
#include "gemm_common.h"

namespace moe {
namespace {

typedef float f32x16 __attribute__((ext_vector_type(16)));

// Epilogue of the gate_up GEMM: SwiGLU of the (gate, up) accumulator pairs, bf16,
// stored in the fragment order the down GEMM reads as its row operand.
template <int RBT, int RS, typename C, bool STREAM>
__device__ __forceinline__ void gate_up_epilogue(const f32x16 (&acc)[RBT][C::NBW], void *__restrict__ outp,
                                                 int out_ld, float limit, int rb0, int rbt, int nb0,
                                                 int nb_valid, int cw, int rg, int lane) {
  constexpr int NBW = C::NBW;
  // Column blocks come in (gate, up) pairs (see pack_weight_kernel): blocks 2P
  // and 2P+1 of the product hold gate_j and up_j of j = 32P .. 32P+31 in the
  // same lane and register.  The activation goes out as bf16 in the fragment
  // order the down GEMM reads as its row operand: column j is k block j/16,
  // lane ((j%16)/8)*32 + token, element j % 8.  Registers 4g .. 4g+3 of lane
  // (token t, half h) are j = 8g + 4h .. +3: elements 4h .. 4h+3 of the
  // fragment lane (g % 2)*32 + t of k block g / 2.  One exchange between the
  // lane halves (v_permlane32_swap) per dword completes the 16 bytes of every
  // fragment lane; nothing goes through LDS.
  u32x4 *act = reinterpret_cast<u32x4 *>(outp);
  const int kb2_total = out_ld / kFragK;
  const int P0 = (nb0 + cw * NBW) >> 1;                // first pair of this wave
  const int pairs_valid = (nb_valid - cw * NBW) >> 1;  // >= 1 here
#pragma unroll
  for (int i = 0; i < RBT; i++) {
    const int blk = i * RS + rg;
    if (RS > 1 && blk >= rbt) break;
#pragma unroll
    for (int p = 0; p < NBW / 2; p++) {
      uint32_t pk[4][2];
#pragma unroll
      for (int g = 0; g < 4; g++)
#pragma unroll
        for (int d = 0; d < 2; d++)
          pk[g][d] = pack_bf16(
              swiglu_shifted(acc[i][2 * p][4 * g + 2 * d], acc[i][2 * p + 1][4 * g + 2 * d], limit),
              swiglu_shifted(acc[i][2 * p][4 * g + 2 * d + 1], acc[i][2 * p + 1][4 * g + 2 * d + 1],
                             limit));
      u32x4 *dst = act + ((size_t)(rb0 + blk) * kb2_total + 2 * (P0 + p)) * 64 + lane;
#pragma unroll
      for (int kb = 0; kb < 2; kb++) {
        // upper lane half of registers 8kb .. 8kb+3 <-> lower lane half of 8kb+4 .. 8kb+7
        const u32x2 s0 = __builtin_amdgcn_permlane32_swap(pk[2 * kb][0], pk[2 * kb + 1][0], false, false);
        const u32x2 s1 = __builtin_amdgcn_permlane32_swap(pk[2 * kb][1], pk[2 * kb + 1][1], false, false);
        if (p < pairs_valid) store_output<STREAM>(&dst[kb * 64], u32x4{s0[0], s1[0], s0[1], s1[1]});
      }
    }
  }
}

// The column operand is MXFP4 as packed by pack_fp4_kernel: per pair of
// column blocks and step of 32 k one 16-byte chunk per lane (blocks 2P and 2P+1,
// each [k block 0: 8 nibbles][k block 1: 8 nibbles] of the lane's row) and two
// scale bytes per row.  A step of 32 k is exactly one MXFP4 block, so one scale
// serves both of its k blocks.  The nibbles become bf16 MFMA operands in
// registers (v_cvt_scalef32_pk_bf16_fp4: two values and their scale per
// instruction, exact).
//
// RS (row split) > 1 serves the last column tile of a matrix whose width is not
// a multiple of the tile's: only NW / RS waves would have columns there, so the
// waves form RS groups that share those columns and split the row blocks
// (group rg takes row blocks rg, rg + RS, ...).  RBT is then the row blocks per
// wave, RBT * RS are staged per step (blocks past the tile's rbt repeat its
// last one and are not stored).
//
// gemm_tile is the down GEMM; gate_up, whose row operand is scattered, is
// gemm_tile_gl below.
template <int RBT, int RS, typename C, bool STREAM>
__device__ __forceinline__ void gemm_tile(const uint4 *__restrict__ a_frag,  // [rb][KB][64]
                                          const uint4 *__restrict__ b_frag,  // expert's [nb/2][KB/2][64] chunks
                                          const uint16_t *__restrict__ b_scale,  // expert's [nb/2][KB/2][32] byte pairs
                                          int KB, int rb0, int rbt, int nb0, int nb_valid,
                                          const float *__restrict__ bias,  // expert's
                                          float *__restrict__ y, int out_ld,
                                          // One __restrict__ pointer per LDS stage: after
                                          // inlining the compiler can tell a read of one stage
                                          // from the DMA that fills another and waits only for
                                          // the fill of the stage it reads.
                                          uint4 *__restrict__ s0, uint4 *__restrict__ s1,
                                          uint4 *__restrict__ s2, uint4 *__restrict__ s3,
                                          // The epilogue buffers are not carved out of the
                                          // ring: the compiler would make every read of them
                                          // wait for all outstanding vector memory operations,
                                          // the epilogue's own stores included.
                                          uint4 *__restrict__ epi) {
  StageRing<C::R> ring;
  {
    uint4 *const all[4] = {s0, s1, s2, s3};
#pragma unroll
    for (int i = 0; i < C::R; i++) ring.p[i] = all[i];
  }
  constexpr int NBW = C::NBW, KPS = C::KPS, R = C::R, NW = C::NW;
  static_assert(KPS == 2, "the step is software-pipelined as two k blocks");
  constexpr int A_CH = RBT * RS * KPS;       // 1 KB chunks of the row operand per step
  constexpr int LA = (A_CH + NW - 1) / NW;   // DMA loads per wave per step (a short last pass repeats a chunk)
  constexpr int LB = 2;                      // register loads per wave per step (nibbles, scales)
  constexpr int LPS = LA + LB;
  static_assert(LPS * (R - 2) + LA <= 63, "vmcnt is a 6-bit counter");
  static_assert(NBW == 2, "an MXFP4 chunk holds the pair of column blocks of one wave");
  constexpr int NM = RBT * NBW;              // MFMAs per k block
  constexpr int DEC = NBW;         // decode items per k block (one column block each)
  constexpr int SIDE1 = (RBT + LB + DEC + NM - 1) / NM;  // side items per MFMA, k block 0
  constexpr int SIDE2 = (LA + RBT + DEC + NM - 1) / NM;  // ... k block 1
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  static_assert(NW % RS == 0 && RBT * RS <= C::RBT_MAX, "row split");
  const int cw = RS == 1 ? w : w % (NW / RS);  // the wave's place among the columns
  const int rg = RS == 1 ? 0 : w / (NW / RS);  // ... and among the row groups

  // The accumulators start from the bias.  Register q of lane l is token
  // 8*(q/4) + 4*(l/32) + q%4 of its row block, lane l column l % 32.  The bias
  // loads go out first and are consumed after the pipeline's loads have been issued.
  float bias_d[NBW];
#pragma unroll
  for (int j = 0; j < NBW; j++) bias_d[j] = bias[kRowBlock * (nb0 + min(cw * NBW + j, nb_valid - 1)) + (lane & 31)];
  f32x16 acc[RBT][NBW];

  const int n_steps = KB / KPS;
  const uint4 *a_src = a_frag + (size_t)rb0 * KB * 64 + lane;
  // Column blocks past the end of the matrix (last column tile only) re-load
  // the last valid block; their products are never stored.
  const size_t pair = (size_t)((nb0 + min(cw * NBW, nb_valid - NBW)) >> 1);
  const uint4 *b_src = b_frag + pair * n_steps * 64 + lane;
  const uint16_t *s_src = b_scale + pair * n_steps * 32 + (lane & 31);

  // Row operand: chunk c of a step (c = pass*NW + wave) is row block c / KPS, k block c % KPS.
  auto issue_a = [&](uint4 *st, int ks, int m) {
    const int c = min(m * NW + w, A_CH - 1);
    const int blk = RS == 1 ? c / KPS : min(c / KPS, rbt - 1);
    dma_to_lds_16(a_src + ((size_t)blk * KB + ks * KPS + c % KPS) * 64, st + c * 64);
  };
  // Column operand: load 0 of a slot is the chunk of nibbles, load 1 the two scale bytes.
  u32x4 bq[R];
  uint32_t bsc[R];
  auto issue_b = [&](int slot, int ks, int m) {
    if (m == 0) {
      bq[slot] = load_cols<STREAM>(b_src + (size_t)ks * 64);
    } else {
      bsc[slot] = s_src[(size_t)ks * 32];
    }
  };
  // The decoded operands of the step at hand, [column block][k block].
  // Those of k block 0 are decoded during the previous step's second half,
  // those of k block 1 during this step's first half.
  bf16x8 bdec[NBW][KPS];
  auto decode = [&](int slot, int j, int kk) {
    const float scale = __uint_as_float(((bsc[slot] >> (8 * j)) & 0xffu) << 23);  // 2^(s - 127)
    const uint32_t nib = bq[slot][j * KPS + kk];
    const bf16x2 p0 = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp4(nib, scale, 0);
    const bf16x2 p1 = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp4(nib, scale, 1);
    const bf16x2 p2 = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp4(nib, scale, 2);
    const bf16x2 p3 = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp4(nib, scale, 3);
    bdec[j][kk] = bf16x8{p0[0], p0[1], p1[0], p1[1], p2[0], p2[1], p3[0], p3[1]};
  };
  // Two register sets of row fragments: while the MFMAs of one k block run, the
  // fragments of the next are read from LDS.
  bf16x8 fa[2][RBT];
  auto read_a = [&](const uint4 *st, int kk, int buf, int i) {
    fa[buf][i] = __builtin_bit_cast(bf16x8, st[((i * RS + rg) * KPS + kk) * 64 + lane]);
  };
  auto mma = [](bf16x8 rows, bf16x8 colv, f32x16 c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(rows, colv, c, 0, 0, 0);
  };
  static_assert(R >= 3 && R <= 4, "up to four stage arrays are passed in");
  // "Step s of the row operand has landed" as a bound on the vector-memory
  // counter.  The loads are issued in the order A(0) B(0) A(1) B(1) ... and
  // complete in that order, so all but the newest n outstanding means step s has
  // landed with n = everything issued behind it.  Open question: in a configuration
  // since removed (ring of 7, two or three workgroups per CU, DMA of 32 bytes of
  // scattered token rows, this mixed count of DMAs and register loads) whole tiles of
  // wrong token rows were once seen, different from run to run.  A cause that fits, not tested
  // there: the column refills of the steps left over, which the compiler dropped, were counted all
  // the same, so that from the second of them on a wait could leave its rows in flight
  // (in a ring of 4 the second is the last that runs, and reads no further rows).  The half-height
  // kernels share three of those properties (two workgroups per CU, scattered DMA in
  // gate_up, the mixed count).  tests/test_counted_waits.py holds the counts against the built code,
  // and test_large_batches_repeat_bit_for_bit looks for other bits in all of them.
  constexpr int WAIT_DMA_FILL = LPS * (R - 2) + LA;  // A(0), A(0..R-1) issued
  constexpr int WAIT_DMA_STEP = LPS * (R - 2);       // B(ks+1), and with it A(ks+1), at step ks

  // Issue order per wave: A(0) B(0) A(1) B(1) ... ; at the top of step ks the row
  // operand is issued through step ks+R-1 and the column operand through ks+R-2
  // (step indices past the tile's last are clamped to it).
  const int last = n_steps - 1;
#pragma unroll
  for (int s = 0; s < R - 1; s++) {
#pragma unroll
    for (int m = 0; m < LA; m++) issue_a(ring.p[s], min(s, last), m);
#pragma unroll
    for (int m = 0; m < LB; m++) issue_b(s, min(s, last), m);
    __builtin_amdgcn_sched_barrier(0);  // the counted waits rely on this issue order
  }
#pragma unroll
  for (int j = 0; j < NBW; j++)
#pragma unroll
    for (int i = 0; i < RBT; i++)
#pragma unroll
      for (int q = 0; q < 16; q++) acc[i][j][q] = bias_d[j];
#pragma unroll
  for (int m = 0; m < LA; m++) issue_a(ring.p[R - 1], min(R - 1, last), m);
  WAIT_VMCNT(WAIT_DMA_FILL);
  lds_barrier();
#pragma unroll
  for (int i = 0; i < RBT; i++) read_a(ring.p[0], 0, 0, i);
#pragma unroll
  for (int j = 0; j < NBW; j++) decode(0, j, 0);

  // Step ks, slot u = ks % R:
  //   [MFMAs of k block 0 | read row fragments of k block 1, load B(ks+R-1) into slot u-1]
  //   wait until step ks+1 has arrived, barrier
  //   [MFMAs of k block 1 | DMA A(ks+R) into stage u, read row fragments of step ks+1]
  // The side work is spread over the MFMAs so that it issues in their shadow.
  // Inside the loop every step is the same straight code with the same count in its wait: the
  // refills of a tile's last steps, for which there is nothing left to load, load its last step
  // again (cache hits that nobody reads) instead of being skipped.  Skipping them costs more: with
  // refills guarded at run time the waits can no longer be counted and the last six steps took
  // twice their time (-3.4 % on gate_up, -4.9 % on down with the loads kept).  The wave ends with
  // those loads in flight; s_endpgm waits for them.  The steps left over behind the loop (u = 0 ..
  // R-2) are straight code of their own.  Nothing reads what they would ask for, and the
  // compiler drops such loads of registers: they are left out by rule, and the count is of what is
  // there.  Behind B(ks+1) these are A(ks+2) .. A(ks+R-1-u) and B(ks+2) .. B(ks+R-2-u).
  auto step = [&](auto u_c, auto left_over, int ks) {
    constexpr int u = decltype(u_c)::value;
    constexpr bool refill = decltype(left_over)::value == 0, is_last = !refill && u == R - 2;
    const uint4 *cur = ring.p[u];
    const int ks_b = min(ks + R - 1, last);
    const int ks_a = min(ks + R, last);
#pragma unroll
    for (int m = 0; m < NM; m++) {
#pragma unroll
      for (int t = m * SIDE1; t < (m + 1) * SIDE1; t++) {
        if (t < RBT) {
          read_a(cur, 1, 1, t);
        } else if (t < RBT + LB) {
          if constexpr (refill) issue_b((u + R - 1) % R, ks_b, t - RBT);
        } else if (t < RBT + LB + DEC) {
          decode(u, t - RBT - LB, 1);
        }
      }
      acc[m / NBW][m % NBW] = mma(fa[0][m / NBW], bdec[m % NBW][0], acc[m / NBW][m % NBW]);
      __builtin_amdgcn_sched_barrier(0);
    }
    if constexpr (!is_last) {
      WAIT_VMCNT(refill ? WAIT_DMA_STEP : LPS * (R - 2 - u) - LB);
      lds_barrier();  // step ks+1 is complete in LDS; every wave is done with stage u
    }
    const uint4 *nxt = ring.p[(u + 1) % R];
#pragma unroll
    for (int m = 0; m < NM; m++) {
#pragma unroll
      for (int t = m * SIDE2; t < (m + 1) * SIDE2; t++) {
        if (t < LA) {
          if constexpr (refill) issue_a(ring.p[u], ks_a, t);
        } else if (t < LA + RBT) {
          if constexpr (!is_last) read_a(nxt, 0, 0, t - LA);
        } else if (t < LA + RBT + DEC) {
          if constexpr (!is_last) decode((u + 1) % R, t - LA - RBT, 0);  // landed: the wait above covers it
        }
      }
      acc[m / NBW][m % NBW] = mma(fa[1][m / NBW], bdec[m % NBW][1], acc[m / NBW][m % NBW]);
      __builtin_amdgcn_sched_barrier(0);
    }
  };
  int ks0 = 0;
  for (; ks0 + R <= n_steps; ks0 += R)
    static_for<R>([&](auto u_c) { step(u_c, IC<0>{}, ks0 + decltype(u_c)::value); });
  static_left<R - 1>(n_steps - ks0, [&](auto u_c) { step(u_c, IC<1>{}, ks0 + decltype(u_c)::value); });

  // Epilogue.
  if (cw * NBW >= nb_valid) return;  // a wave without columns (last column tile only)
  constexpr int LD = C::EPI_LD;  // +8 floats keep the two lane halves on different banks
  float *ef = reinterpret_cast<float *>(epi + w * C::EPI_WAVE);
  const int n = lane & 31;
  const int rsub = 4 * (lane >> 5);
  const int col0 = kRowBlock * (nb0 + cw * NBW);
#pragma unroll
  for (int i = 0; i < RBT; i++) {
    const int blk = i * RS + rg;
    if (RS > 1 && blk >= rbt) break;
#pragma unroll
    for (int j = 0; j < NBW; j++)
#pragma unroll
      for (int q = 0; q < 16; q++) {
        const int r = 8 * (q >> 2) + rsub + (q & 3);
        ef[r * LD + 32 * j + n] = acc[i][j][q];
      }
    const size_t row0 = (size_t)(rb0 + blk) * kRowBlock;
#pragma unroll
    for (int t = 0; t < NBW * 4; t++) {
      const int idx = t * 64 + lane;
      const int r = idx / (NBW * 8);
      const int c4 = idx % (NBW * 8);
      const f32x4 v = *reinterpret_cast<const f32x4 *>(ef + r * LD + 4 * c4);
      if (cw * NBW + c4 / 8 < nb_valid)
        store_output<STREAM>(reinterpret_cast<f32x4 *>(y + (row0 + r) * out_ld + col0 + 4 * c4), v);
    }
  }
}

// gate_up of the large batches without a gathered copy of the routed rows: the
// row operand's DMA reads the token rows themselves, WHOLE CACHE LINES at a time.
// One instruction fetches 8 rows x 128 bytes (64 k); a scattered DMA that takes
// 32 bytes of 32 rows per instruction costs
// the main loop a quarter more, and 64 bytes of 16 rows an eighth.
//
// So the row operand is staged in double steps: a double stage holds 64 k of
// all rows of the tile (two 16 KB arrays: row blocks 0-3 and 4-7), R2 of them
// form the ring, and the refill comes every other step.  Wave w fetches rows
// 8w .. 8w+7 of every row block; inside its kilobyte a lane holds one 16-byte
// piece of one of the 8 rows, and WHICH is chosen so that (a) the four lanes of
// a quad read 64 contiguous bytes of one row and (b) the MFMA operand reads
// (lane = row, all lanes the same piece) find 8 consecutive rows on the 8
// different 16-byte slots of 128 bytes of LDS and 16 consecutive rows on the 16
// of 256 bytes: quad Q = 4 * (row / 2) + 2 * (half of the line ^ w % 2) + row % 2,
// and lane j of the quad holds piece (j - row / 2) mod 4 of that half.
//
// The column operand keeps its ring of RB register slots of one step each.
// Loads are issued in the order  B(0) B(1) B(2) A2(0) A2(1) A2(2) A2(3) | step 0:
// B(3) | step 1: B(4) A2(4) | step 2: B(5) | step 3: B(6) A2(5) | ...  (R2 = RB =
// 4).  The counted wait in the middle of a step leaves the newest 2 LB + LA2
// loads in flight (see gemm_tile for the assumption and the open question): that covers A2(d+1), which
// an odd step 2d+1 needs, and B(ks+1), which every step's successor needs.  Even
// steps need no barrier: they read a double stage that landed before the
// previous odd step's barrier and refill nothing.
template <int RBT, int RS, typename C, bool STREAM>
__device__ __forceinline__ void gemm_tile_gl(const uint4 *__restrict__ x_rows,  // token rows [T][KB * 2] of 16 bytes
                                             const uint4 *__restrict__ b_frag,
                                             const uint16_t *__restrict__ b_scale, int KB, int rb0, int rbt,
                                             int nb0, int nb_valid, const int *__restrict__ rowmap,
                                             const float *__restrict__ bias_a,
                                             const float *__restrict__ bias_b, void *__restrict__ outp,
                                             int out_ld, float limit, uint4 *__restrict__ s0,
                                             uint4 *__restrict__ s1, uint4 *__restrict__ s2,
                                             uint4 *__restrict__ s3, uint4 *__restrict__ s4,
                                             uint4 *__restrict__ s5, uint4 *__restrict__ s6,
                                             uint4 *__restrict__ s7) {
  constexpr int NBW = C::NBW, KPS = C::KPS, RB = C::R, NW = C::NW, R2 = kLineStages;
  static_assert(KPS == 2 && NW == 4 && RB == 4 && C::RBT_MAX <= 8 && (RS == 1 || RS == 2), "shape of the line gather");
  constexpr int NB = RBT * RS;                // row blocks staged per step
  constexpr int LA2 = NB;                     // DMA loads per wave and double step: one per row block
  constexpr int LB = 2;                       // register loads per wave and step (nibbles, scales)
  static_assert(NBW == 2, "an MXFP4 chunk holds the pair of column blocks of one wave");
  constexpr int NM = RBT * NBW;               // MFMAs per k block
  constexpr int DEC = NBW;
  static_assert(R2 >= 3, "with 2 double stages an odd step would have to wait for all but 2 * LB loads");
  constexpr int WAIT_FILL = (R2 - 1) * LA2;  // the loads behind A2(0) in the first filling
  constexpr int WAIT_MID = 2 * LB + LA2;                                     // see the steps
  static_assert(WAIT_FILL <= 63 && WAIT_MID <= 63, "vmcnt is a 6-bit counter");
  uint4 *const arr[8] = {s0, s1, s2, s3, s4, s5, s6, s7};
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int cw = RS == 1 ? w : w % (NW / RS);
  const int rg = RS == 1 ? 0 : w / (NW / RS);

  float4 bias_g[NBW / 2][4], bias_u[NBW / 2][4];
  {
    const int P_last = ((nb0 + nb_valid) >> 1) - 1;
    const int P0 = (nb0 + cw * NBW) >> 1;
#pragma unroll
    for (int p = 0; p < NBW / 2; p++) {
      const int P = min(P0 + p, P_last);
#pragma unroll
      for (int g = 0; g < 4; g++) {
        const int j = kRowBlock * P + 8 * g + 4 * (lane >> 5);
        bias_g[p][g] = *reinterpret_cast<const float4 *>(bias_a + j);
        bias_u[p][g] = *reinterpret_cast<const float4 *>(bias_b + j);
      }
    }
  }
  f32x16 acc[RBT][NBW];
  const int n_steps = KB / KPS;  // even: the depth is a multiple of 64
  const int last = n_steps - 1, last_d = n_steps / 2 - 1;

  // this lane's source in a double step of row block m: its token's row and its piece of the line.
  // The row map is asked for here; the answer is used after the column operand's
  // first loads have gone out (below), so that its latency costs the tile nothing.
  uint32_t lane_src[LA2];
  int lane_piece;
  {
    const int Q = lane >> 2, j = lane & 3;  // quad Q of the kilobyte: row 2 * (Q / 4) + Q % 2, one half of its line
    const int row8 = 2 * (Q >> 2) + (Q & 1);
    lane_piece = 4 * (((Q >> 1) & 1) ^ (w & 1)) + ((j - (Q >> 2)) & 3);
#pragma unroll
    for (int m = 0; m < LA2; m++) {
      const int blk = RS == 1 ? m : min(m, rbt - 1);
      lane_src[m] = (uint32_t)rowmap[(rb0 + blk) * kRowBlock + 8 * w + row8];
    }
  }
  // where this lane finds its operand of (parity of the step, k block) inside a row block's 4 KB
  int lane_rd[2][KPS];
  {
    const int r = lane & 31, h = lane >> 5, sub = r >> 3, row8 = r & 7;
#pragma unroll
    for (int par = 0; par < 2; par++)
#pragma unroll
      for (int kk = 0; kk < KPS; kk++)
        lane_rd[par][kk] = sub * 64 + (4 * (row8 >> 1) + 2 * (par ^ (sub & 1)) + (row8 & 1)) * 4 +
                           ((kk * 2 + h + (row8 >> 1)) & 3);
  }
  const size_t pair = (size_t)((nb0 + min(cw * NBW, nb_valid - NBW)) >> 1);
  const uint4 *b_src = b_frag + pair * n_steps * 64 + lane;
  const uint16_t *s_src = b_scale + pair * n_steps * 32 + (lane & 31);

  // double step jd of row block m into double stage slot d
  auto issue_a2 = [&](int d, int jd, int m) {
    dma_to_lds_16(x_rows + lane_src[m] + jd * 8, arr[2 * d + (m >= 4 ? 1 : 0)] + ((m & 3) * 4 + w) * 64);
  };
  u32x4 bq[RB];
  uint32_t bsc[RB];
  auto issue_b = [&](int slot, int ks, int m) {
    if (m == 0) {
      bq[slot] = load_cols<STREAM>(b_src + (size_t)ks * 64);
    } else {
      bsc[slot] = s_src[(size_t)ks * 32];
    }
  };
  bf16x8 bdec[NBW][KPS];
  auto decode = [&](int slot, int j, int kk) {
    const float scale = __uint_as_float(((bsc[slot] >> (8 * j)) & 0xffu) << 23);
    const uint32_t nib = bq[slot][j * KPS + kk];
    const bf16x2 p0 = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp4(nib, scale, 0);
    const bf16x2 p1 = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp4(nib, scale, 1);
    const bf16x2 p2 = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp4(nib, scale, 2);
    const bf16x2 p3 = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp4(nib, scale, 3);
    bdec[j][kk] = bf16x8{p0[0], p0[1], p1[0], p1[1], p2[0], p2[1], p3[0], p3[1]};
  };
  bf16x8 fa[2][RBT];
  // fragment of the wave's row block i from double stage slot d
  auto read_a = [&](int d, int par, int kk, int buf, int i) {
    const uint4 *st = arr[2 * d + (i * RS >= 4 ? 1 : 0)];
    fa[buf][i] = __builtin_bit_cast(bf16x8, st[(((i * RS + rg) & 3) * 4) * 64 + lane_rd[par][kk]]);
  };
  auto mma = [](bf16x8 rows, bf16x8 colv, f32x16 c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(colv, rows, c, 0, 0, 0);
  };

  // one double step of the row operand / one step of the column operand, all of the wave's loads
  auto issue_a2_all = [&](int d, int jd) {
#pragma unroll
    for (int m = 0; m < LA2; m++) issue_a2(d, min(jd, last_d), m);
  };
  auto issue_b_all = [&](int slot, int ks) {
#pragma unroll
    for (int m = 0; m < LB; m++) issue_b(slot, min(ks, last), m);
  };
  // first filling: B(0) .. B(RB-2), then (the row map has answered meanwhile) A2(0) .. A2(R2-1)
#pragma unroll
  for (int k = 0; k < RB - 1; k++) issue_b_all(k, k);
  __builtin_amdgcn_sched_barrier(0);  // the counted waits rely on this issue order
#pragma unroll
  for (int m = 0; m < LA2; m++) {
    const int a = (int)lane_src[m];
    const int tok = a >= 0 ? a / kTopK : 0;  // padding rows read token 0; their products are never used
    lane_src[m] = (uint32_t)tok * (uint32_t)(KB * 2) + lane_piece;
  }
#pragma unroll
  for (int k = 0; k < R2 - 1; k++) issue_a2_all(k, k);
  __builtin_amdgcn_sched_barrier(0);
#pragma unroll
  for (int p = 0; p < NBW / 2; p++)
#pragma unroll
    for (int g = 0; g < 4; g++)
#pragma unroll
      for (int i = 0; i < RBT; i++) {
        const float4 bg = bias_g[p][g], bu = bias_u[p][g];
        acc[i][2 * p][4 * g + 0] = bg.x; acc[i][2 * p][4 * g + 1] = bg.y;
        acc[i][2 * p][4 * g + 2] = bg.z; acc[i][2 * p][4 * g + 3] = bg.w;
        acc[i][2 * p + 1][4 * g + 0] = bu.x + 1.0f; acc[i][2 * p + 1][4 * g + 1] = bu.y + 1.0f;
        acc[i][2 * p + 1][4 * g + 2] = bu.z + 1.0f; acc[i][2 * p + 1][4 * g + 3] = bu.w + 1.0f;
      }
  issue_a2_all(R2 - 1, R2 - 1);
  WAIT_VMCNT(WAIT_FILL);
  lds_barrier();
#pragma unroll
  for (int i = 0; i < RBT; i++) read_a(0, 0, 0, 0, i);
#pragma unroll
  for (int j = 0; j < NBW; j++) decode(0, j, 0);

  // Step ks = 2 jd + par, u = ks mod PERIOD: column slot u % RB, double stage (u / 2) % R2.
  constexpr int PERIOD = R2 == 3 ? 12 : 2 * R2;  // a multiple of 2 * R2 and of RB
  static_assert(PERIOD % RB == 0 && PERIOD % (2 * R2) == 0, "one unrolled round serves both rings");
  // Steps left over behind the loop, at most.  The rows of all of them and the columns of three
  // have been asked for by then; what nothing reads is left out by rule (see gemm_tile).
  constexpr int LEFT = PERIOD - 1;
  auto step = [&](auto u_c, auto left_over, int ks) {
    constexpr int u = decltype(u_c)::value;
    constexpr bool left = decltype(left_over)::value != 0, is_last = left && u == LEFT - 1;
    constexpr bool refill_b = !left || u + RB - 1 < LEFT;
    constexpr int slot = u % RB, d = (u / 2) % R2, par = u % 2;
    constexpr int LAX = par && !left ? LA2 : 0;    // the refill comes with the odd steps
    constexpr int dn = par ? (d + 1) % R2 : d;     // the next step's double stage
    constexpr int SIDE1 = (RBT + LB + DEC + NM - 1) / NM;
    constexpr int SIDE2 = (LAX + RBT + DEC + NM - 1) / NM;
    const int ks_b = min(ks + RB - 1, last);
    const int jd_a = min(ks / 2 + R2, last_d);
#pragma unroll
    for (int m = 0; m < NM; m++) {
#pragma unroll
      for (int t = m * SIDE1; t < (m + 1) * SIDE1; t++) {
        if (t < RBT) {
          read_a(d, par, 1, 1, t);
        } else if (t < RBT + LB) {
          if constexpr (refill_b) issue_b((slot + RB - 1) % RB, ks_b, t - RBT);
        } else if (t < RBT + LB + DEC) {
          decode(slot, t - RBT - LB, 1);
        }
      }
      acc[m / NBW][m % NBW] = mma(fa[0][m / NBW], bdec[m % NBW][0], acc[m / NBW][m % NBW]);
      __builtin_amdgcn_sched_barrier(0);
    }
    // Every step says in its middle what has landed, as a count: all but the
    // column loads of the last two steps and the double step issued between
    // them.  An odd step needs A2(jd+1), which lies further back, for the
    // fragment reads that follow; every step needs B(ks+1) for its successor's
    // first MFMA, and with the count given here the compiler adds no wait of its
    // own (left to itself it waits for ALL loads before some of the steps).  Of the steps left over
    // only the first two have a double step behind B(ks+1).
    constexpr int n_b = !left ? 2 : (u < 1 || u + RB - 2 < LEFT ? 1 : 0) + (refill_b ? 1 : 0);
    if constexpr (!is_last) WAIT_VMCNT(n_b * LB + (!left || u < 2 ? LA2 : 0));
    if constexpr (is_last) {
      __builtin_amdgcn_sched_barrier(0);
    } else if constexpr (par == 1) {
      lds_barrier();  // double step jd+1 is complete in LDS; every wave is done with double stage d
    } else {
      __builtin_amdgcn_sched_barrier(0);
    }
#pragma unroll
    for (int m = 0; m < NM; m++) {
#pragma unroll
      for (int t = m * SIDE2; t < (m + 1) * SIDE2; t++) {
        if (t < LAX) {
          issue_a2(d, jd_a, t);
        } else if (t < LAX + RBT) {
          if constexpr (!is_last) read_a(dn, par ^ 1, 0, 0, t - LAX);
        } else if (t < LAX + RBT + DEC) {
          if constexpr (!is_last) decode((slot + 1) % RB, t - LAX - RBT, 0);
        }
      }
      acc[m / NBW][m % NBW] = mma(fa[1][m / NBW], bdec[m % NBW][1], acc[m / NBW][m % NBW]);
      __builtin_amdgcn_sched_barrier(0);
    }
  };
  int ks0 = 0;
  for (; ks0 + PERIOD <= n_steps; ks0 += PERIOD)
    static_for<PERIOD>([&](auto u_c) { step(u_c, IC<0>{}, ks0 + decltype(u_c)::value); });
  static_left<LEFT>(n_steps - ks0, [&](auto u_c) { step(u_c, IC<1>{}, ks0 + decltype(u_c)::value); });

  if (cw * NBW >= nb_valid) return;  // a wave without columns (last column tile only)
  gate_up_epilogue<RBT, RS, C, STREAM>(acc, outp, out_ld, limit, rb0, rbt, nb0, nb_valid, cw, rg, lane);
}

template <typename C, bool GATE_UP, bool STREAM>
__global__ __launch_bounds__(C::THREADS, C::WGS) void grouped_gemm_kernel(
    const uint4 *__restrict__ a_frag, const uint4 *__restrict__ w_frag,
    const uint16_t *__restrict__ w_scale,
    const float *__restrict__ bias_a, const float *__restrict__ bias_b,
    const TileDesc *__restrict__ tiles, const int *__restrict__ totals,
    const int *__restrict__ rowmap, void *__restrict__ outp, int K, int N, float limit) {
  static_assert(C::R <= 4 && (C::RBT_MAX == 4 || C::RBT_MAX == 8), "stage arrays and tile heights below");
  // gate_up: 4 KB per row block and double stage, four row blocks to an array;
  // down: one array per stage
  constexpr int ST_EVEN = GATE_UP ? 4 * 256 : C::STAGE;
  constexpr int ST_ODD = GATE_UP ? (C::RBT_MAX == 8 ? 4 * 256 : 1) : C::STAGE;
  __shared__ uint4 st0[ST_EVEN], st1[ST_ODD], st2[ST_EVEN], st3[ST_ODD];
  __shared__ uint4 st4[GATE_UP ? ST_EVEN : 1], st5[GATE_UP ? ST_ODD : 1], st6[GATE_UP ? ST_EVEN : 1],
      st7[GATE_UP ? ST_ODD : 1];
  __shared__ uint4 epi[GATE_UP ? 1 : C::NW * C::EPI_WAVE];
  const int KB = K / kFragK;
  const int nb_total = (GATE_UP ? 2 * N : N) / kRowBlock;  // weight row blocks per expert
  TileDesc tc;
  if (!locate_tile(tiles, totals + (GATE_UP ? kTotBoundsGateUp : kTotBoundsDown), tc)) return;
  const int nb0 = tc.nb0, nb_valid = tc.nbt;
  // per expert (nb_total/2) * (KB/2) chunks of 1 KB
  const uint4 *b_frag = w_frag + (size_t)tc.e * nb_total * KB * 16;
  const uint16_t *b_scale = w_scale + (size_t)tc.e * nb_total * KB * 8;
  const float *ba = bias_a + (size_t)tc.e * N;
  const float *bb = GATE_UP ? bias_b + (size_t)tc.e * N : nullptr;
  // the tile with n row blocks per wave and the waves in rs row groups
  auto tile = [&](auto n_c, auto rs_c) {
    constexpr int n = decltype(n_c)::value, rs = decltype(rs_c)::value;
    if constexpr (n * rs <= C::RBT_MAX) {
      if constexpr (GATE_UP) {
        gemm_tile_gl<n, rs, C, STREAM>(a_frag, b_frag, b_scale, KB, tc.rb0, tc.rbt, nb0, nb_valid, rowmap,
                                            ba, bb, outp, N, limit, st0, st1, st2, st3, st4, st5, st6, st7);
      } else {
        gemm_tile<n, rs, C, STREAM>(a_frag, b_frag, b_scale, KB, tc.rb0, tc.rbt, nb0, nb_valid, ba,
                                         static_cast<float *>(outp), N, st0, st1, st2, st3, epi);
      }
    }
  };
  // the last column tile, when only a quarter or half of the waves have columns in it
  const int rs = row_split_of(nb_valid, C::NW, C::NBW);
  if constexpr (!GATE_UP) {  // gate_up comes in (gate, up) pairs of pairs: never a quarter
    if (rs == 4) {
      if (tc.rbt <= 4) tile(IC<1>{}, IC<4>{}); else tile(IC<2>{}, IC<4>{});
      return;
    }
  }
  if (rs == 2) {
    switch ((tc.rbt + 1) >> 1) {
      case 1: tile(IC<1>{}, IC<2>{}); break;
      case 2: tile(IC<2>{}, IC<2>{}); break;
      case 3: tile(IC<3>{}, IC<2>{}); break;
      default: tile(IC<4>{}, IC<2>{}); break;
    }
    return;
  }
  switch (tc.rbt) {
    case 1: tile(IC<1>{}, IC<1>{}); break;
    case 2: tile(IC<2>{}, IC<1>{}); break;
    case 3: tile(IC<3>{}, IC<1>{}); break;
    case 4: tile(IC<4>{}, IC<1>{}); break;
    case 5: tile(IC<5>{}, IC<1>{}); break;
    case 6: tile(IC<6>{}, IC<1>{}); break;
    case 7: tile(IC<7>{}, IC<1>{}); break;
    default: tile(IC<8>{}, IC<1>{}); break;
  }
}

// 4 waves, one per SIMD, each 256 rows x 64 columns (8 x 2 accumulators = all
// 256 accumulation registers); 256 x 256 tiles; 4 ring slots.
using CfgFull = GemmCfg<4, 2, 4, 8, 1>;
// Tiles half as high, two workgroups per CU.  A step of MXFP4 weights is
// 4 KB, so that a second tile of the same columns costs next to nothing, and the
// decode, the fill and the epilogue of one workgroup run under the other's MFMAs.
// us per layer call, full / half height (2880 x 2880, even routing): 32 experts, 256
// tokens 175 / 143; 128 experts, 768: 533 / 428.  Runs where an expert has 17 to 63 rows
// on average and there are 512 tiles of one row tile per expert (32 experts: 129 to 511 tokens);
// with more rows gemm_fp4.hip has the same tiles and the other product.
using CfgHalf = GemmCfg<4, 2, 4, 4, 2>;
static_assert(CfgFull::RBT_MAX * kRowBlock == kTileRows && CfgHalf::RBT_MAX * kRowBlock == kHalfTileRows &&
                  CfgFull::TILE_NB == kGemmTileNb && CfgHalf::TILE_NB == kGemmTileNb,
              "tile plan of build_plan");

}  // namespace

// w holds MXFP4 chunks and w_scale their scale bytes (pack_fp4_kernel).  The plan is of tiles of tile_rows.
template <bool GATE_UP>
static hipError_t launch_gemm(const void *a, const void *w, const uint16_t *w_scale, const float *ba,
                              const float *bb, const DispatchBuffers &d, void *out, int K, int N,
                              float limit, int T, int E, int tile_rows, bool wide, bool stream, hipStream_t s) {
  const int nb_total = (GATE_UP ? 2 * N : N) / kRowBlock;
  const int n_ct = (nb_total + kGemmTileNb - 1) / kGemmTileNb;
  const dim3 grid(kXcds * xcd_tile_cap(gemm_tile_cap(T, E, tile_rows) * n_ct), wide ? 2 : 1);
  const TileDesc *tiles = GATE_UP ? d.tiles_gate_up : d.tiles_down;
  const uint4 *af = static_cast<const uint4 *>(a), *wf = static_cast<const uint4 *>(w);
  // the full-height kernels take a plan of either height, the others one of half height
#define MOE_GEMM(C, STREAM)                                                                                 \
  grouped_gemm_kernel<C, GATE_UP, STREAM><<<grid, C::THREADS, 0, s>>>(af, wf, w_scale, ba, bb, tiles, d.totals, \
                                                                      d.rowmap, out, K, N, limit)
  if (tile_rows != kHalfTileRows) MOE_GEMM(CfgFull, false);
  else if (stream) MOE_GEMM(CfgHalf, true);
  else MOE_GEMM(CfgHalf, false);
#undef MOE_GEMM
  return hipGetLastError();
}

hipError_t launch_gate_up(const uint16_t *x, const void *w1, const uint16_t *w1_scale, const float *b1g,
                          const float *b1u, const DispatchBuffers &d, uint16_t *act, int H, int IM,
                          float limit, int T, int E, int tile_rows, bool wide, bool cached, hipStream_t s) {
  if (H % 64 || IM % 64) return hipErrorInvalidValue;  // the kernels take steps of 32 in pairs
  const TileRoute r = tile_route(T, E, 2 * IM, w1_scale != nullptr, tile_rows, cached);
  if (r.kernel == kBf16Tiles)
    return launch_bf16_gate_up(x, w1, b1g, b1u, d, act, H, IM, limit, T, E, tile_rows, wide, r.past_caches, s);
  if (r.kernel == kFp4ManyTiles)
    return launch_fp4_gate_up(x, w1, w1_scale, b1g, b1u, d, act, H, IM, limit, T, E, r.past_caches, s);
  return launch_gemm<true>(x, w1, w1_scale, b1g, b1u, d, act, H, IM, limit, T, E, tile_rows, wide, r.past_caches, s);
}

hipError_t launch_down(const uint16_t *act, const void *w2, const uint16_t *w2_scale, const float *b2,
                       const DispatchBuffers &d, float *y, int H, int IM, int T, int E, int tile_rows,
                       bool wide, bool cached, hipStream_t s) {
  if (H % 64 || IM % 64) return hipErrorInvalidValue;  // the kernels take steps of 32 in pairs
  const TileRoute r = tile_route(T, E, 2 * IM, w2_scale != nullptr, tile_rows, cached);
  if (r.kernel == kBf16Tiles) return launch_bf16_down(act, w2, b2, d, y, H, IM, T, E, tile_rows, wide, r.past_caches, s);
  if (r.kernel == kFp4ManyTiles) return launch_fp4_down(act, w2, w2_scale, b2, d, y, H, IM, T, E, r.past_caches, s);
  return launch_gemm<false>(act, w2, w2_scale, b2, nullptr, d, y, IM, H, 0.f, T, E, tile_rows, wide, r.past_caches, s);
}

}  // namespace moe

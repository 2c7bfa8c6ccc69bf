// Grouped expert GEMMs with MXFP4 weights, for batches with many rows per expert: the
// kernels of gemm.hip (whose header has the data layout, the tiling, the tile order and
// the loads) at tiles of 128 rows with v_mfma_f32_16x16x32_bf16 in place of 32x32x16.
//
// At thousands of tokens the clock falls from 2.4 to 1.7-2.1 GHz whenever all CUs multiply, so
// that the energy of a product counts.  From registers alone, on all CUs, 16x16x32 runs at
// 2030-2050 TFLOP/s and 32x32x16 at 1810-1830 (operands of unit scale); the sums are the same bits.  us per layer call, 32x32x16 / this: 32 experts, 512 tokens 174 / 162,
// 4096: 745 / 695; 7168, Zipf's routing (exponent 1.2) 1215 / 1128; 128 experts, 3072: 688 / 655.
// Where the time is that of loads the smaller products are more instructions for nothing (fp4_many_rows).
#include "gemm_common.h"

namespace moe {
namespace {

// The product of 16 rows and 16 columns over 32 k.  The weights are the first operand,
// so a lane ends with four consecutive columns of one row.
__device__ __forceinline__ void mma(f32x4 &acc, bf16x8 rows, bf16x8 cols) {
  acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(cols, rows, acc, 0, 0, 0);
}
// Lane 16 q + r of either operand holds row (column) r of the 16 and piece q of 8 k of the step's
// four.  Where piece q stands in a pair of fragments (two k blocks of 32 rows), for the first 16 rows:
__device__ __forceinline__ int piece_at(int q, int r16) { return (q >> 1) * 64 + (q & 1) * 32 + r16; }

// The operands of the two groups of 16 columns of block j out of a lane's chunk and the
// scale bytes of its row.  A lane of a chunk holds row lane % 32 and the piece lane / 32 of
// both k blocks: exchanging lane halves between the k blocks and then 16-lane rows between the
// results leaves the four pieces of 16 rows in either register (part 0); parts 1 to 4 convert a
// quarter each.  In parts, because a wave alone on its SIMD has 16 clocks of one product to
// hide instructions under, and two conversions take that (in one piece: 32 experts, 4096
// tokens 705 us per layer call instead of 693; spread evenly over the products 728).
constexpr int kDecodeParts = 5;
struct Fp4Decoder {
  u32x2 nibbles;
  float scale[2];
  __device__ __forceinline__ void part(int n, u32x4 chunk, uint32_t scales, int j, bf16x8 (&out)[2]) {
    if (n == 0) {
      const u32x2 ss = __builtin_amdgcn_permlane16_swap(scales, scales, false, false);
      const u32x2 kk = __builtin_amdgcn_permlane32_swap(chunk[2 * j], chunk[2 * j + 1], false, false);
      nibbles = __builtin_amdgcn_permlane16_swap(kk[0], kk[1], false, false);
#pragma unroll
      for (int h = 0; h < 2; h++) scale[h] = __uint_as_float(((ss[h] >> (8 * j)) & 0xffu) << 23);  // 2^(s - 127)
    } else if (n & 1) {
      const int h = n >> 1;
      const bf16x2 p0 = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp4(nibbles[h], scale[h], 0);
      const bf16x2 p1 = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp4(nibbles[h], scale[h], 1);
      out[h][0] = p0[0]; out[h][1] = p0[1]; out[h][2] = p1[0]; out[h][3] = p1[1];
    } else {
      const int h = (n >> 1) - 1;
      const bf16x2 p2 = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp4(nibbles[h], scale[h], 2);
      const bf16x2 p3 = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp4(nibbles[h], scale[h], 3);
      out[h][4] = p2[0]; out[h][5] = p2[1]; out[h][6] = p3[0]; out[h][7] = p3[1];
    }
  }
};

// Epilogue of the gate_up GEMM: SwiGLU of the (gate, up) accumulator pairs, bf16,
// stored in the fragment order the down GEMM reads as its row operand.
template <int RBT, int RS, typename C>
__device__ __forceinline__ void gate_up_epilogue(const f32x4 (&acc)[2 * RBT][2 * C::NBW], void *__restrict__ outp,
                                                 int out_ld, float limit, int rb0, int rbt, int nb0,
                                                 int nb_valid, int cw, int rg, int lane) {
  constexpr int NBW = C::NBW;
  // Column blocks come in (gate, up) pairs (see pack_weight_kernel): blocks 2P
  // and 2P+1 of the product hold gate_j and up_j of j = 32P .. 32P+31 in the
  // same lane and register.  The activation goes out as bf16 in the fragment
  // order the down GEMM reads as its row operand: column j is k block j/16,
  // lane ((j%16)/8)*32 + token, element j % 8.  Lane 16 q + r of group g and columns c
  // holds row r of the 16 and j = 16 c + 4 q .. +3.  One exchange between the 16-lane
  // rows of two neighbouring groups (v_permlane16_swap) per dword completes the 16
  // bytes of every fragment lane; nothing goes through LDS.
  uint4 *act = reinterpret_cast<uint4 *>(outp);
  const int kb2_total = out_ld / kFragK;
  const int P0 = (nb0 + cw * NBW) >> 1;                // first pair of this wave
  const int pairs_valid = (nb_valid - cw * NBW) >> 1;  // >= 1 here
#pragma unroll
  for (int i = 0; i < RBT; i++) {
    const int blk = i * RS + rg;
    if (RS > 1 && blk >= rbt) break;
#pragma unroll
    for (int p = 0; p < NBW / 2; p++) {
      uint4 *dst = act + ((size_t)(rb0 + blk) * kb2_total + 2 * (P0 + p)) * 64 + lane;
#pragma unroll
      for (int c = 0; c < 2; c++) {
        uint32_t pk[2][2];
#pragma unroll
        for (int h = 0; h < 2; h++)
#pragma unroll
          for (int d = 0; d < 2; d++) {
            const f32x4 g = acc[2 * i + h][4 * p + c], u = acc[2 * i + h][4 * p + 2 + c];
            pk[h][d] = pack_bf16(swiglu_shifted(g[2 * d], u[2 * d], limit),
                                 swiglu_shifted(g[2 * d + 1], u[2 * d + 1], limit));
          }
        const u32x2 s0 = __builtin_amdgcn_permlane16_swap(pk[0][0], pk[1][0], false, false);
        const u32x2 s1 = __builtin_amdgcn_permlane16_swap(pk[0][1], pk[1][1], false, false);
        if (p < pairs_valid) dst[c * 64] = make_uint4(s0[0], s1[0], s0[1], s1[1]);
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
  constexpr int NC = 2 * NBW;                // groups of 16 columns
  constexpr int NM = RBT * NC;               // MFMAs per half of a step
  constexpr int SIDE1 = (kDecodeParts + RBT + LB + NM - 1) / NM;  // side items per MFMA, first half
  constexpr int SIDE2 = (LA + RBT + kDecodeParts + NM - 1) / NM;  // ... second half
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  static_assert(NW % RS == 0 && RBT * RS <= C::RBT_MAX, "row split");
  const int cw = RS == 1 ? w : w % (NW / RS);  // the wave's place among the columns
  const int rg = RS == 1 ? 0 : w / (NW / RS);  // ... and among the row groups

  const int r16 = lane & 15, q = lane >> 4;
  // The accumulators start from the bias: lane 16 q + r of columns c holds row r and columns
  // 16 c + 4 q .. +3.  The bias loads go out first and are consumed after the
  // pipeline's loads have been issued.
  f32x4 bias_d[NC];
#pragma unroll
  for (int c = 0; c < NC; c++)
    bias_d[c] = *reinterpret_cast<const f32x4 *>(bias + kRowBlock * (nb0 + min(cw * NBW + (c >> 1), nb_valid - 1)) +
                                                 16 * (c & 1) + 4 * q);
  f32x4 acc[2 * RBT][NC];

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
  // Two register sets of row fragments, the two halves of the wave's groups of 16 rows:
  // while the MFMAs of one half run, the fragments of the next are read from LDS.
  bf16x8 fa[2][RBT];
  const int lane_rd = piece_at(q, r16);
  auto read_a = [&](const uint4 *st, int hf, int i) {
    const int g = hf * RBT + i;  // group of 16 rows: half g % 2 of the wave's row block g / 2
    fa[hf][i] = __builtin_bit_cast(bf16x8, st[((g >> 1) * RS + rg) * KPS * 64 + (g & 1) * 16 + lane_rd]);
  };
  // The decoded operands.  Those of column block 0 are decoded during the step before, by the
  // step's parity, those of block 1 in front of the step's first products.
  bf16x8 bdec0[2][2], bdec1[2];
  Fp4Decoder dec;
  auto decode = [&](int slot, int par, int j, int n) {
    if (j == 0) dec.part(n, bq[slot], bsc[slot], 0, bdec0[par]); else dec.part(n, bq[slot], bsc[slot], 1, bdec1);
  };
  // product m of half hf: the half's row groups times block 0, then times block 1
  auto product = [&](int par, int hf, int m) {
    const int j = m / (2 * RBT), i = m / 2 % RBT, h = m % 2;
    mma(acc[hf * RBT + i][2 * j + h], fa[hf][i], j == 0 ? bdec0[par][h] : bdec1[h]);
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
  for (int g = 0; g < 2 * RBT; g++)
#pragma unroll
    for (int c = 0; c < NC; c++) acc[g][c] = bias_d[c];
#pragma unroll
  for (int m = 0; m < LA; m++) issue_a(ring.p[R - 1], min(R - 1, last), m);
  WAIT_VMCNT(WAIT_DMA_FILL);
  lds_barrier();
#pragma unroll
  for (int i = 0; i < RBT; i++) read_a(ring.p[0], 0, i);
#pragma unroll
  for (int n = 0; n < kDecodeParts; n++) decode(0, 0, 0, n);

  // Step ks, slot u = ks % R:
  //   [first half of the row groups | decode column block 1, read the second half, load B(ks+R-1) into slot u-1]
  //   wait until step ks+1 has arrived, barrier
  //   [second half | DMA A(ks+R) into stage u, read the first half of step ks+1, decode its column block 0]
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
        if (t < kDecodeParts) {
          decode(u, u & 1, 1, t);
        } else if (t < kDecodeParts + RBT) {
          read_a(cur, 1, t - kDecodeParts);
        } else if (t < kDecodeParts + RBT + LB) {
          if constexpr (refill) issue_b((u + R - 1) % R, ks_b, t - kDecodeParts - RBT);
        }
      }
      product(u & 1, 0, m);
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
          if constexpr (!is_last) read_a(nxt, 0, t - LA);
        } else if (t < LA + RBT + kDecodeParts) {
          if constexpr (!is_last) decode((u + 1) % R, (u + 1) & 1, 0, t - LA - RBT);  // landed: the wait above covers it
        }
      }
      product(u & 1, 1, m);
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
  const int col0 = kRowBlock * (nb0 + cw * NBW);
#pragma unroll
  for (int i = 0; i < RBT; i++) {
    const int blk = i * RS + rg;
    if (RS > 1 && blk >= rbt) break;
#pragma unroll
    for (int h = 0; h < 2; h++)
#pragma unroll
      for (int c = 0; c < NC; c++)
        *reinterpret_cast<f32x4 *>(ef + (16 * h + r16) * LD + 16 * c + 4 * q) = acc[2 * i + h][c];
    const size_t row0 = (size_t)(rb0 + blk) * kRowBlock;
#pragma unroll
    for (int t = 0; t < NBW * 4; t++) {
      const int idx = t * 64 + lane;
      const int r = idx / (NBW * 8);
      const int c4 = idx % (NBW * 8);
      const float4 v = *reinterpret_cast<const float4 *>(ef + r * LD + 4 * c4);
      if (cw * NBW + c4 / 8 < nb_valid)
        *reinterpret_cast<float4 *>(y + (row0 + r) * out_ld + col0 + 4 * c4) = v;
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
// all rows of the tile (16 KB), R2 of them form the ring, and the refill comes every other step.  Wave w fetches rows
// 8w .. 8w+7 of every row block; inside its kilobyte a lane holds one 16-byte
// piece of one of the 8 rows, and WHICH is chosen so that (a) the four lanes of
// a quad read 64 contiguous bytes of one row and (b) the MFMA operand reads (16 lanes
// to a piece of 8 k) find 16 different slots of 256 bytes, whichever of the four pieces'
// lanes the LDS serves side by side: quad Q = 4 * (row / 2) + 2 * (half of the line ^ w % 2)
// + row % 2, and lane j of the quad holds piece j ^ (row / 2) of that half.
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
                                             uint4 *__restrict__ s3) {
  constexpr int NBW = C::NBW, KPS = C::KPS, RB = C::R, NW = C::NW, R2 = kLineStages;
  static_assert(KPS == 2 && NW == 4 && RB == 4 && C::RBT_MAX == 4 && RS <= 2, "shape of the line gather");
  constexpr int NB = RBT * RS;                // row blocks staged per step
  constexpr int LA2 = NB;                     // DMA loads per wave and double step: one per row block
  constexpr int LB = 2;                       // register loads per wave and step (nibbles, scales)
  static_assert(NBW == 2, "an MXFP4 chunk holds the pair of column blocks of one wave");
  constexpr int NC = 2 * NBW;                 // groups of 16 columns
  constexpr int NM = RBT * NC;                // MFMAs per half of a step
  static_assert(R2 == 4, "stage arrays");
  constexpr int WAIT_FILL = (R2 - 1) * LA2;  // the loads behind A2(0) in the first filling
  constexpr int WAIT_MID = 2 * LB + LA2;                                     // see the steps
  static_assert(WAIT_FILL <= 63 && WAIT_MID <= 63, "vmcnt is a 6-bit counter");
  uint4 *const arr[4] = {s0, s1, s2, s3};
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int cw = RS == 1 ? w : w % (NW / RS);
  const int rg = RS == 1 ? 0 : w / (NW / RS);

  const int r16 = lane & 15, q = lane >> 4;
  f32x4 bias[NC];  // of each pair of column blocks two groups of gate, two of up
  {
    const int P_last = ((nb0 + nb_valid) >> 1) - 1;
    const int P0 = (nb0 + cw * NBW) >> 1;
#pragma unroll
    for (int c = 0; c < NC; c++)
      bias[c] = *reinterpret_cast<const f32x4 *>((c % 4 < 2 ? bias_a : bias_b) + kRowBlock * min(P0 + c / 4, P_last) +
                                                 16 * (c & 1) + 4 * q);
  }
  f32x4 acc[2 * RBT][NC];
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
    lane_piece = 4 * (((Q >> 1) & 1) ^ (w & 1)) + (j ^ (Q >> 2));
#pragma unroll
    for (int m = 0; m < LA2; m++) {
      const int blk = RS == 1 ? m : min(m, rbt - 1);
      lane_src[m] = (uint32_t)rowmap[(rb0 + blk) * kRowBlock + 8 * w + row8];
    }
  }
  // where this lane finds its operand of (parity of the step, half of the row block) inside a row block's 4 KB
  int lane_rd[2][2];
#pragma unroll
  for (int par = 0; par < 2; par++)
#pragma unroll
    for (int h = 0; h < 2; h++) {
      const int sub = 2 * h + (r16 >> 3), row8 = r16 & 7;
      lane_rd[par][h] = sub * 64 + (4 * (row8 >> 1) + 2 * (par ^ (sub & 1)) + (row8 & 1)) * 4 + (q ^ (row8 >> 1));
    }
  const size_t pair = (size_t)((nb0 + min(cw * NBW, nb_valid - NBW)) >> 1);
  const uint4 *b_src = b_frag + pair * n_steps * 64 + lane;
  const uint16_t *s_src = b_scale + pair * n_steps * 32 + (lane & 31);

  // double step jd of row block m into double stage slot d
  auto issue_a2 = [&](int d, int jd, int m) {
    dma_to_lds_16(x_rows + lane_src[m] + jd * 8, arr[d] + (m * 4 + w) * 64);
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
  bf16x8 fa[2][RBT];
  // operand i of half hf of the wave's groups of 16 rows from double stage slot d
  auto read_a = [&](int d, int par, int hf, int i) {
    const int g = hf * RBT + i, blk = g >> 1;
    fa[hf][i] = __builtin_bit_cast(bf16x8, arr[d][(blk * RS + rg) * 256 + lane_rd[par][g & 1]]);
  };
  bf16x8 bdec0[2][2], bdec1[2];
  Fp4Decoder dec;
  auto decode = [&](int slot, int par, int j, int n) {
    if (j == 0) dec.part(n, bq[slot], bsc[slot], 0, bdec0[par]); else dec.part(n, bq[slot], bsc[slot], 1, bdec1);
  };
  // product m of half hf: the half's row groups times block 0, then times block 1
  auto product = [&](int par, int hf, int m) {
    const int j = m / (2 * RBT), i = m / 2 % RBT, h = m % 2;
    mma(acc[hf * RBT + i][2 * j + h], fa[hf][i], j == 0 ? bdec0[par][h] : bdec1[h]);
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
  for (int g = 0; g < 2 * RBT; g++)
#pragma unroll
    for (int c = 0; c < NC; c++) acc[g][c] = c % 4 < 2 ? bias[c] : bias[c] + 1.0f;
  issue_a2_all(R2 - 1, R2 - 1);
  WAIT_VMCNT(WAIT_FILL);
  lds_barrier();
#pragma unroll
  for (int i = 0; i < RBT; i++) read_a(0, 0, 0, i);
#pragma unroll
  for (int n = 0; n < kDecodeParts; n++) decode(0, 0, 0, n);

  // Step ks = 2 jd + par, u = ks mod PERIOD: column slot u % RB, double stage (u / 2) % R2.
  constexpr int PERIOD = 2 * R2;  // a multiple of RB, too
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
    constexpr int SIDE1 = (kDecodeParts + RBT + LB + NM - 1) / NM;
    constexpr int SIDE2 = (LAX + RBT + kDecodeParts + NM - 1) / NM;
    const int ks_b = min(ks + RB - 1, last);
    const int jd_a = min(ks / 2 + R2, last_d);
#pragma unroll
    for (int m = 0; m < NM; m++) {
#pragma unroll
      for (int t = m * SIDE1; t < (m + 1) * SIDE1; t++) {
        if (t < kDecodeParts) {
          decode(slot, slot & 1, 1, t);
        } else if (t < kDecodeParts + RBT) {
          read_a(d, par, 1, t - kDecodeParts);
        } else if (t < kDecodeParts + RBT + LB) {
          if constexpr (refill_b) issue_b((slot + RB - 1) % RB, ks_b, t - kDecodeParts - RBT);
        }
      }
      product(slot & 1, 0, m);
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
          if constexpr (!is_last) read_a(dn, par ^ 1, 0, t - LAX);
        } else if (t < LAX + RBT + kDecodeParts) {
          if constexpr (!is_last) decode((slot + 1) % RB, (slot + 1) & 1, 0, t - LAX - RBT);
        }
      }
      product(slot & 1, 1, m);
      __builtin_amdgcn_sched_barrier(0);
    }
  };
  int ks0 = 0;
  for (; ks0 + PERIOD <= n_steps; ks0 += PERIOD)
    static_for<PERIOD>([&](auto u_c) { step(u_c, IC<0>{}, ks0 + decltype(u_c)::value); });
  static_left<LEFT>(n_steps - ks0, [&](auto u_c) { step(u_c, IC<1>{}, ks0 + decltype(u_c)::value); });

  if (cw * NBW >= nb_valid) return;  // a wave without columns (last column tile only)
  gate_up_epilogue<RBT, RS, C>(acc, outp, out_ld, limit, rb0, rbt, nb0, nb_valid, cw, rg, lane);
}

template <typename C, bool GATE_UP, bool STREAM>
__global__ __launch_bounds__(C::THREADS, C::WGS) void fp4_gemm_kernel(
    const uint4 *__restrict__ a_frag, const uint4 *__restrict__ w_frag,
    const uint16_t *__restrict__ w_scale,
    const float *__restrict__ bias_a, const float *__restrict__ bias_b,
    const TileDesc *__restrict__ tiles, const int *__restrict__ totals,
    const int *__restrict__ rowmap, void *__restrict__ outp, int K, int N, float limit) {
  static_assert(C::R == 4 && C::RBT_MAX == 4, "stage arrays and tile heights below");
  // gate_up: 4 KB per row block and double stage; down: a stage of one step
  constexpr int ST = GATE_UP ? 4 * 256 : C::STAGE;
  __shared__ uint4 st0[ST], st1[ST], st2[ST], st3[ST];
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
    if constexpr (GATE_UP) {
      gemm_tile_gl<n, rs, C, STREAM>(a_frag, b_frag, b_scale, KB, tc.rb0, tc.rbt, nb0, nb_valid, rowmap, ba, bb, outp,
                                     N, limit, st0, st1, st2, st3);
    } else {
      gemm_tile<n, rs, C, STREAM>(a_frag, b_frag, b_scale, KB, tc.rb0, tc.rbt, nb0, nb_valid, ba,
                                  static_cast<float *>(outp), N, st0, st1, st2, st3, epi);
    }
  };
  // the last column tile, when only a quarter or half of the waves have columns in it
  const int rs = row_split_of(nb_valid, C::NW, C::NBW);
  if constexpr (!GATE_UP) {  // gate_up comes in (gate, up) pairs of pairs: never a quarter
    if (rs == 4) {
      tile(IC<1>{}, IC<4>{});
      return;
    }
  }
  if (rs == 2) {
    if (tc.rbt <= 2) tile(IC<1>{}, IC<2>{}); else tile(IC<2>{}, IC<2>{});
    return;
  }
  switch (tc.rbt) {
    case 1: tile(IC<1>{}, IC<1>{}); break;
    case 2: tile(IC<2>{}, IC<1>{}); break;
    case 3: tile(IC<3>{}, IC<1>{}); break;
    default: tile(IC<4>{}, IC<1>{}); break;
  }
}

using Cfg = GemmCfg<4, 2, 4, 4, 2>;  // two workgroups per CU
static_assert(Cfg::RBT_MAX * kRowBlock == kHalfTileRows && Cfg::TILE_NB == kGemmTileNb, "tile plan of build_plan");

template <bool GATE_UP>
hipError_t launch(const void *a, const void *w, const uint16_t *w_scale, const float *ba, const float *bb,
                  const DispatchBuffers &d, void *out, int K, int N, float limit, int T, int E, bool stream,
                  hipStream_t s) {
  const int nb_total = (GATE_UP ? 2 * N : N) / kRowBlock;
  const int n_ct = (nb_total + kGemmTileNb - 1) / kGemmTileNb;
  const int grid = kXcds * xcd_tile_cap(gemm_tile_cap(T, E, kHalfTileRows) * n_ct);
  const TileDesc *tiles = GATE_UP ? d.tiles_gate_up : d.tiles_down;
  const uint4 *af = static_cast<const uint4 *>(a), *wf = static_cast<const uint4 *>(w);
  if (stream)
    fp4_gemm_kernel<Cfg, GATE_UP, true><<<grid, Cfg::THREADS, 0, s>>>(af, wf, w_scale, ba, bb, tiles, d.totals, d.rowmap,
                                                                      out, K, N, limit);
  else
    fp4_gemm_kernel<Cfg, GATE_UP, false><<<grid, Cfg::THREADS, 0, s>>>(af, wf, w_scale, ba, bb, tiles, d.totals, d.rowmap,
                                                                       out, K, N, limit);
  return hipGetLastError();
}

}  // namespace

hipError_t launch_fp4_gate_up(const uint16_t *x, const void *w1, const uint16_t *w1_scale, const float *b1g,
                              const float *b1u, const DispatchBuffers &d, uint16_t *act, int H, int IM, float limit,
                              int T, int E, bool stream, hipStream_t s) {
  return launch<true>(x, w1, w1_scale, b1g, b1u, d, act, H, IM, limit, T, E, stream, s);
}

hipError_t launch_fp4_down(const uint16_t *act, const void *w2, const uint16_t *w2_scale, const float *b2,
                           const DispatchBuffers &d, float *y, int H, int IM, int T, int E, bool stream, hipStream_t s) {
  return launch<false>(act, w2, w2_scale, b2, nullptr, d, y, IM, H, 0.f, T, E, stream, s);
}

}  // namespace moe

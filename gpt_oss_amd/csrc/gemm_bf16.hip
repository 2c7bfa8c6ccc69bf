// Grouped expert GEMMs with bf16 weights, for the batches that are not a stream of
// weights (stream.hip).  Same contract, data layout and tile plan as the MXFP4 kernels
// of gemm.hip (matmul/matmul.cpp:1023-1914, SwiGLU of run.cpp:709-726).
//
// Tiling.  A workgroup of eight waves, two on a SIMD, owns a tile of rbt x 32 rows and
// 256 columns of one expert.  Wave w holds the 64 columns w % 4 of the row blocks w / 4,
// w / 4 + 2, ...: an odd height splits into two waves of a SIMD that have one row
// block more and one less, so that every SIMD has the same work and the tile's rows
// still pad to at most 31.  In the last column tile of a matrix whose width is not a
// multiple of 256 fewer waves have columns; they then take every fourth or eighth row
// block (S).  A tile of up to six row blocks may have 320 columns (bf16_wide_tiles has when, and the
// figures): 60 of the 64 blocks of sums that the registers hold, in the same 160 KB of rings.  Its last two column
// blocks are two waves' of either half of the rows, so that every SIMD still has the same work.
//
// Feeding the matrix cores.  Both operands go through LDS by DMA, and a wave reads 8 KB
// of rows and 4 KB of columns per step of 32 k (LDS reads run at 226 bytes per clock and
// CU here, a step of a full tile takes 1024).  The columns stand in a ring of four slots
// of a step, the rows in three stages of a double step (64 k, because gate_up fetches
// whole 128-byte lines of scattered token rows, see row_source), all 160 KB together.
// One barrier per step, in its middle: behind it the step's slot is free (its operands
// are in registers), and the next step's has landed.  Loads go out one of columns and one
// of rows per half step, so that the CU's address unit, 16 clocks a load, is never asked
// for more than it takes in that time (six loads behind every second barrier: 489
// instead of 476 us for gate_up at 4096 tokens and 32 experts).
//
// What bounds it.  At thousands of tokens two things, neither of them alone.  The tile
// plan: the flops of 4096 tokens at 32 experts take 457 + 276 us as ragged experts and 402 +
// 220 as four dense ones (the same kernel and operands; down's 948 tiles are 3.7 rounds of the
// CUs, 768 are 3).  The clock, which falls from 2.4 to 1.7-2.1 GHz whenever all CUs multiply
// numbers that toggle: with zero weights the ragged experts take 408 + 252.  So the
// energy of a product counts.  v_mfma_f32_16x16x32_bf16 takes less than 32x32x16 (from
// registers alone, all CUs: 2030-2050 against 1810-1830 TFLOP/s with operands of unit scale,
// 1955-1994 against 1670-1840 with weights of 0.02) and gives the same bits.  Workgroups that
// stay and load the next tile under the epilogue of the last one spend no time between
// tiles, but their steps take longer, 1033 instead of 931 clocks.  us per layer call at
// 2880 x 2880, 32 x 32 x 16 with the columns through registers and four waves, which this replaced / the
// same with 16 x 16 x 32 / this: 4096 tokens, 32 experts 830 / 816 / 808; 7168, Zipf's routing
// (exponent 1.2) 1406 / 1347 / 1323.  6144 tokens at 128 experts (1662 / 1649 / 1645), 512 tokens, Zipf's (366 /
// 367 / 362), and 672 of 896 rows active (345 / 344 / 342) gained no more than two runs of one
// side differ.  With few rows per expert it is HBM: a tile's fill and epilogue are not under
// its stream.
#include <type_traits>

#include "moe_internal.h"
#include "swiglu.h"

namespace moe {
namespace {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

constexpr int kWaves = 8, kThreads = kWaves * 64;
constexpr int kRowBlockBytes = 4096;  // a double step (64 k) of a row block in LDS
constexpr int kColBlockBytes = 2048;  // a step (32 k) of a column block
constexpr uint32_t kColSlots = 4, kRowStages = 3;
// The rings of a tile of up to W column blocks and H row blocks, the rows' behind the columns'.
template <int W, int H>
struct Rings {
  static constexpr uint32_t ColSlot = W * kColBlockBytes, RowRing = ColSlot * kColSlots;
  static constexpr uint32_t RowStage = H * kRowBlockBytes, End = RowRing + RowStage * kRowStages;
};
using Square = Rings<8, 8>;
using Wide = Rings<10, 6>;
constexpr uint32_t kLds = Square::End;  // 160 KB
static_assert(Wide::End <= kLds, "rings");
static_assert(kTileRows == 8 * kRowBlock, "tile plan of build_plan");

// ---- 16 bytes per lane from global memory to LDS, lane l at lds + 16 l ----
// In assembly, because the compiler, which does not know one stage from another here,
// would make every LDS read wait for all of them.  There is no output register; the
// waits are the counted ones below and the barriers.  m0 is named as written, which the
// compiler remarks on, as on any register that it does not allocate.
#pragma clang diagnostic push
#pragma clang diagnostic ignored "-Winline-asm"
__device__ __forceinline__ void dma_lanes(uint32_t lds, const char *g) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, off" ::"s"(lds), "v"(g) : "m0", "memory");
}
// ... from base + lane_off + OFF, where OFF counts on both sides.  STREAM: past the caches
// (gemm_streams_weights).
template <int OFF, bool STREAM>
__device__ __forceinline__ void dma_wave(uint32_t lds, const char *base, uint32_t lane_off) {
  if constexpr (STREAM)
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2 offset:%3 nt" ::"s"(lds), "v"(lane_off),
                 "s"(base), "n"(OFF)
                 : "m0", "memory");
  else
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2 offset:%3" ::"s"(lds), "v"(lane_off),
                 "s"(base), "n"(OFF)
                 : "m0", "memory");
}
#pragma clang diagnostic pop
typedef __attribute__((address_space(3))) const u32x4 lds_u32x4;
typedef __attribute__((address_space(3))) const char lds_char;
__device__ __forceinline__ bf16x8 lds_operand(uint32_t byte, int off) {
  return __builtin_bit_cast(bf16x8, *(lds_u32x4 *)((lds_char *)(uintptr_t)byte + off));
}

// s_waitcnt with only the vector-memory counter constrained (gfx9 encoding): loads land
// in the order in which they went out, so "at most n outstanding" means "all but the newest n".
#define WAIT_VMCNT(n) \
  __builtin_amdgcn_s_waitcnt(((n) & 0xf) | (((n) >> 4) << 14) | (0x7 << 4) | (0xf << 8))
// Orders LDS traffic only (a __syncthreads would wait for the loads in flight as well).
__device__ __forceinline__ void lds_barrier() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }

struct Tile {
  const char *a;       // gate_up: token rows; down: activation fragments
  const char *b;       // expert's weights
  const float *ba, *bb;
  const int *rowmap;
  void *out;
  int KB, N, rb0, rbt, nb0, nb_valid;
  float limit;
};

// A wave's share of a tile: RBW row blocks (rg, rg + S, ...; one past the tile's last repeats
// it and is not stored) times NU units of columns.  A unit is what ends as 32 columns of down (a column
// block) or 16 of the activation (half a pair of gate and up blocks): units 2 wn and 2 wn + 1, and with
// NU = 3 unit 8 + wx.  LA: its loads of rows per double step, LB: of columns per step.
template <int RBW, int LA, int S, int NU, int LB, typename R, bool GATE_UP, bool STREAM, bool PAST>
__device__ __forceinline__ void wave_tile(const Tile &t, uint32_t lds0) {
  constexpr int NC = 2 * NU;  // groups of 16 columns: gate_up: the units' gates, then their ups; down: the units' halves
  const int tid = threadIdx.x, lane = tid & 63;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wn = w % (kWaves / S), rg = w / (kWaves / S);
  // waves 0, 1 and 6, 7 of a tile of ten blocks have the third units, one on each SIMD (wave w runs on SIMD w % 4)
  const int wx = R::ColSlot == Wide::ColSlot ? (wn & 1) : wn;
  const int sub = w & 3, lg = w >> 2;  // DMA: quarter `sub` of row blocks lg, lg + 2, ...
  const int KB = t.KB, n_steps = KB >> 1, last = n_steps - 1, last_d = (n_steps >> 1) - 1;
  constexpr int RB1 = RBW ? RBW : 1;
  auto unit = [&](int j) { return j < 2 ? 2 * wn + j : 8 + wx; };

  // The accumulators start from the bias.  gate_up's weights are the first operand: lane
  // 16 q + r of group c ends with columns 4 q .. + 3 of row r, the gate (c < NU) and the
  // up (c + NU) of a unit in the same lane (see pack_weight_kernel).  down's rows
  // are: the lane ends with rows 4 q .. + 3 of column r, for stores of whole lines.
  f32x4 bias[NC];
#pragma unroll
  for (int c = 0; c < NC; c++) {
    if constexpr (GATE_UP) {
      const int u = t.nb0 + min(unit(c % NU), t.nb_valid - 1);
      bias[c] = *reinterpret_cast<const f32x4 *>((c < NU ? t.ba : t.bb) + 16 * u + 4 * (lane >> 4));
    } else {
      const float v = t.ba[kRowBlock * (t.nb0 + min(unit(c >> 1), t.nb_valid - 1)) + 16 * (c & 1) + (lane & 15)];
      bias[c] = f32x4{v, v, v, v};
    }
  }
  // Sources of the rows' loads.  gate_up: wave w fetches rows 8 sub .. 8 sub + 7 of a row block, one whole
  // line (64 k) of each.  Lane l's 16 bytes land at place l of the kilobyte; which it takes
  // is chosen so that (a) the four lanes of a quad read 64 contiguous bytes of a row and (b) the
  // operand reads below, 16 lanes to a piece of 8 k, find 16 different slots of 256 bytes whichever
  // of the four pieces the LDS serves side by side: quad Q = 4 (row / 2) + 2 (half of the line ^
  // sub % 2) + row % 2, lane j of it piece j ^ (row / 2) of that half.  down: fragments (gemm.hip's
  // epilogue has the same), a kilobyte each.
  const char *a_src[LA ? LA : 1];
  constexpr int A_STEP = GATE_UP ? 128 : kRowBlockBytes;
  if constexpr (GATE_UP) {
    const int Q = lane >> 2, j = lane & 3;
    const int row8 = 2 * (Q >> 2) + (Q & 1);
    const int piece = 4 * (((Q >> 1) & 1) ^ (sub & 1)) + (j ^ (Q >> 2));
    int a[LA ? LA : 1];
#pragma unroll
    for (int m = 0; m < LA; m++)
      a[m] = t.rowmap[(t.rb0 + min(2 * m + lg, t.rbt - 1)) * kRowBlock + 8 * sub + row8];
#pragma unroll
    for (int m = 0; m < LA; m++) {
      const int tok = a[m] >= 0 ? a[m] / kTopK : 0;  // padding rows read token 0; their products are never used
      a_src[m] = t.a + (size_t)tok * (KB * 32) + piece * 16;
    }
  } else {
#pragma unroll
    for (int m = 0; m < LA; m++)
      a_src[m] = t.a + ((size_t)(t.rb0 + min(2 * m + lg, t.rbt - 1)) * KB + sub) * 1024 + lane * 16;
  }
  const int r16 = lane & 15, p4 = lane >> 4;  // operand layout: row of the group, piece of 8 k
  uint32_t rd_a[2][2];  // [parity of the step][half of the row block]
#pragma unroll
  for (int par = 0; par < 2; par++)
#pragma unroll
    for (int h = 0; h < 2; h++) {
      const int r = 16 * h + r16;
      if constexpr (GATE_UP) {
        const int sb = r >> 3, row8 = r & 7;
        rd_a[par][h] = lds0 + rg * kRowBlockBytes + (sb * 64 + (4 * (row8 >> 1) + 2 * (par ^ (sb & 1)) + (row8 & 1)) * 4 +
                                           (p4 ^ (row8 >> 1))) * 16;
      } else {
        rd_a[par][h] = lds0 + rg * kRowBlockBytes + (2 * par + (p4 >> 1)) * 1024 + ((p4 & 1) * 32 + r) * 16;
      }
    }
  // a pair's blocks of gate and up stand side by side, and a group of 16 is a half of either
  const uint32_t rd_lane = lds0 + (p4 >> 1) * 1024 + ((p4 & 1) * 32 + r16) * 16;
  const uint32_t rd_b = rd_lane + wn * (2 * kColBlockBytes);
  const uint32_t rd_x = rd_lane + (GATE_UP ? (8 + (wx & ~1)) * kColBlockBytes + (wx & 1) * 256 : (8 + wx) * kColBlockBytes);
  const char *b_src = t.b + (size_t)(t.nb0 + min(w, t.nb_valid - 1)) * KB * 1024;
  const char *x_src = t.b + ((size_t)(t.nb0 + min(8 + (w >> 1), t.nb_valid - 1)) * KB + (w & 1)) * 1024;
  const uint32_t lane16 = lane * 16;
  const uint32_t dst_a = lds0 + lg * kRowBlockBytes + sub * 1024, dst_b = lds0 + w * kColBlockBytes;
  const uint32_t dst_x = lds0 + 8 * kColBlockBytes + w * 1024;

  auto issue_a = [&](uint32_t stage, int m) { dma_lanes(dst_a + stage + m * 2 * kRowBlockBytes, a_src[m]); };
  auto issue_b = [&](uint32_t slot, int ks, int n, uint32_t off) {
    const size_t at = (size_t)ks * kColBlockBytes;
    if (n == 0) dma_wave<0, STREAM>(dst_b + slot, b_src + at, off);
    else if (n == 1) dma_wave<kFragBytes, STREAM>(dst_b + slot, b_src + at, off);
    else dma_wave<0, STREAM>(dst_x + slot, x_src + at, off);
  };
  // Lanes' offsets of a load of step ks.  Past the tile's end, where nothing reads what is loaded: the same 16 bytes
  // in every lane with weights past the caches, whose loads would come from HBM once more (672 of 896 tokens 313.3
  // / 312.1 us per call, on another box 318.8 / 314.3, 1400 364.1 / 362.3, 6144 at 128 experts 1440 / 1434).
  auto lanes_of = [&](int ks) -> uint32_t {
    if constexpr (STREAM) return ks > last ? 0u : lane16;
    return lane16;
  };
  auto adv_a = [&](int jd_next) {
    const int d = jd_next <= last_d ? A_STEP : 0;
#pragma unroll
    for (int m = 0; m < LA; m++) a_src[m] += d;
  };
  constexpr int G = 2 * RBW;        // groups of 16 rows
  f32x4 acc[2 * RB1][NC];
  bf16x8 fa[2][RB1], fb[2][NC];     // fa: first and second half of the groups; fb: steps of either parity
  auto read_a = [&](uint32_t stage, int par, int hf, int i) {
    const int g = hf * RBW + i;
    fa[hf][i] = lds_operand(rd_a[par][g & 1] + stage, (g >> 1) * S * kRowBlockBytes);
  };
  auto read_b = [&](uint32_t slot, int par, int c) {
    const int j = GATE_UP ? c % NU : c >> 1, second = GATE_UP ? c / NU : c & 1;  // unit; its up, its second half
    if (j == 2) fb[par][c] = lds_operand(rd_x + slot, second * (GATE_UP ? kColBlockBytes : 256));
    else fb[par][c] = lds_operand(rd_b + slot, GATE_UP ? second * kColBlockBytes + j * 256 : j * kColBlockBytes + second * 256);
  };
#pragma unroll
  for (int g = 0; g < G; g++)
#pragma unroll
    for (int c = 0; c < NC; c++) acc[g][c] = GATE_UP && c >= NU ? bias[c] + 1.0f : bias[c];
  WAIT_VMCNT(0);  // bias and row map: from here on the counter belongs to the loads of A and B
  __builtin_amdgcn_sched_barrier(0);
  // First filling: A(0) B(0) B(1) A(1) B(2) and what the steps before step 0 would have asked for
  // of B(3) and A(2).
  auto fill_a = [&](int d) {
#pragma unroll
    for (int m = 0; m < LA; m++) issue_a(R::RowRing + d * R::RowStage, m);
    adv_a(d + 1);
  };
  auto fill_b = [&](int ks) {
#pragma unroll
    for (int n = 0; n < LB; n++) issue_b(ks * R::ColSlot, min(ks, last), n, lane16);
  };
  fill_a(0);
  fill_b(0);
  fill_b(1);
  fill_a(1);
  fill_b(2);
  issue_b(3 * R::ColSlot, min(3, last), 0, lane16);
  if (LA > 0) issue_a(R::RowRing + 2 * R::RowStage, 0);
  WAIT_VMCNT(LA + (LA > 0) + 2 * LB + 1);  // A(0), B(0)
  lds_barrier();
  if constexpr (RBW > 0) {
#pragma unroll
    for (int c = 0; c < NC; c++) read_b(0, 0, c);
#pragma unroll
    for (int i = 0; i < RBW; i++) read_a(R::RowRing, 0, 0, i);
  }
  uint32_t sa = R::RowRing, sb = 0;
  constexpr int NM = RBW * NC;  // MFMAs of half a step
  auto mma = [&](int par, int hf, int m) {
    const int i = m / NC, c = m % NC, g = hf * RBW + i;
    if constexpr (GATE_UP) acc[g][c] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(fb[par][c], fa[hf][i], acc[g][c], 0, 0, 0);
    else acc[g][c] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(fa[hf][i], fb[par][c], acc[g][c], 0, 0, 0);
  };
  // Step ks = 2 jd + par: the products of the first half of the row groups, barrier, those of the
  // second.  Meanwhile the operands of the next half are read, and one or two loads of columns and one
  // of rows go out: B(ks + 4)'s first behind the barrier of step ks, its others before that of
  // step ks + 1; A(jd + 3) m = 0 behind the barrier of the odd step 2 jd + 1, m = 1, 2, 3 in the
  // halves that follow.  At the barrier of step ks B(ks + 1) has to have landed, and at an odd one
  // A(jd + 1).  Behind B(ks + 1) an even step has issued twice B, m = 1, 2, 3 of A(jd + 1) and m =
  // 0, 1 of A(jd + 2); behind A(jd + 1) an odd one twice B and A(jd + 2).  Every step
  // is the same code with the same counts: past the tile's end the refills load its last step again
  // (lanes_of), which nobody reads.  The wave ends with those in flight; s_endpgm waits for them.
  constexpr int WAIT_EVEN = 2 * LB + (LA > 1) + (LA > 2) + (LA > 3) + (LA > 0) + (LA > 1);
  constexpr int WAIT_ODD = 2 * LB + LA;
  auto step = [&](auto par_c, int ks) {
    constexpr int par = decltype(par_c)::value;
    uint32_t sbn, sbp;  // next and last slot of columns
    if constexpr ((R::RowRing & (R::RowRing - 1)) == 0) {
      sbn = (sb + R::ColSlot) & (R::RowRing - 1);
      sbp = (sb - R::ColSlot) & (R::RowRing - 1);
    } else {
      sbn = sb + R::ColSlot == R::RowRing ? 0 : sb + R::ColSlot;
      sbp = (sb == 0 ? R::RowRing : sb) - R::ColSlot;
    }
    const uint32_t san = par ? (sa + R::RowStage == R::End ? R::RowRing : sa + R::RowStage) : sa;
    const uint32_t sap = (sa == R::RowRing ? R::End : sa) - R::RowStage;
    constexpr int NM1 = NM ? NM : 1;
    {  // first half: even: A(jd + 2) m = 1; odd: m = 3
      constexpr int RD = RBW, AM = par ? 3 : 1, SD = RD + LB - 1 + (AM < LA), SIDE = (SD + NM1 - 1) / NM1;
      const int ks_b = min(ks + 3, last);
#pragma unroll
      for (int m = 0; m < NM1; m++) {
#pragma unroll
        for (int s = m * SIDE; s < (m + 1) * SIDE; s++) {
          if (s < RD) {
            read_a(sa, par, 1, s);
          } else if (s < RD + LB - 1) {
            issue_b(sbp, ks_b, 1 + s - RD, lanes_of(ks + 3));
          } else if (s < SD) {
            issue_a(sap, AM);
          }
        }
        if constexpr (RBW > 0) mma(par, 0, m);
        __builtin_amdgcn_sched_barrier(0);
      }
    }
    if constexpr (par) adv_a((ks >> 1) + 3);
    if constexpr (par) WAIT_VMCNT(WAIT_ODD); else WAIT_VMCNT(WAIT_EVEN);
    lds_barrier();
    {  // second half: even: A(jd + 2) m = 2; odd: A(jd + 3) m = 0
      constexpr int RD = RBW ? RBW + NC : 0, AM = par ? 0 : 2, SD = RD + 1 + (AM < LA),
                    SIDE = (SD + NM1 - 1) / NM1;  // side items per MFMA
      const int ks_b = min(ks + 4, last);
#pragma unroll
      for (int m = 0; m < NM1; m++) {
#pragma unroll
        for (int s = m * SIDE; s < (m + 1) * SIDE; s++) {
          if (s < RD) {
            if (s < NC) read_b(sbn, par ^ 1, s);
            else read_a(san, par ^ 1, 0, s - NC);
          } else if (s == RD) {
            issue_b(sb, ks_b, 0, lanes_of(ks + 4));
          } else if (s < SD) {
            if constexpr (par) issue_a(sa, AM); else issue_a(sap, AM);
          }
        }
        if constexpr (RBW > 0) mma(par, 1, m);
        __builtin_amdgcn_sched_barrier(0);
      }
    }
    sb = sbn;
    sa = san;
  };
  for (int ks = 0; ks < n_steps; ks += 2) {
    step(std::integral_constant<int, 0>{}, ks);
    step(std::integral_constant<int, 1>{}, ks + 1);
  }
  if constexpr (RBW > 0) {
    if (2 * wn >= t.nb_valid) return;  // a wave without columns (last column tile only)
    if constexpr (GATE_UP) {
      // bf16 fragments, as the down GEMM reads them: one exchange of 16-lane rows between the two
      // row groups of a block per dword gives every lane 8 consecutive columns of a row.
      u32x4 *act = reinterpret_cast<u32x4 *>(t.out);
      const int kb2_total = t.N / kFragK;
#pragma unroll
      for (int i = 0; i < RBW; i++) {
        const int blk = i * S + rg;
        if (S > 2 && blk >= t.rbt) break;
        u32x4 *dst = act + ((size_t)(t.rb0 + blk) * kb2_total + t.nb0) * 64 + lane;
#pragma unroll
        for (int j = 0; j < NU; j++) {
          if (j > 1 && unit(j) >= t.nb_valid) break;
          uint32_t pk[2][2];
#pragma unroll
          for (int h = 0; h < 2; h++)
#pragma unroll
            for (int d = 0; d < 2; d++)
              pk[h][d] = pack_bf16(swiglu_shifted(acc[2 * i + h][j][2 * d], acc[2 * i + h][j + NU][2 * d], t.limit),
                                   swiglu_shifted(acc[2 * i + h][j][2 * d + 1], acc[2 * i + h][j + NU][2 * d + 1], t.limit));
          const u32x2 s0 = __builtin_amdgcn_permlane16_swap(pk[0][0], pk[1][0], false, false);
          const u32x2 s1 = __builtin_amdgcn_permlane16_swap(pk[0][1], pk[1][1], false, false);
          store_output<PAST>(&dst[unit(j) * 64], u32x4{s0[0], s1[0], s0[1], s1[1]});
        }
      }
    } else {
      float *y = reinterpret_cast<float *>(t.out);
      // The same exchange between two groups of columns: a store then writes 128 bytes of two rows
      // (16 bytes per lane of 16 rows: 4.2 us per tile instead of 1.9).
      const int col = kRowBlock * t.nb0 + (lane & 31), row = 8 * (lane >> 5);
#pragma unroll
      for (int i = 0; i < RBW; i++) {
        const int blk = i * S + rg;
        if (S > 2 && blk >= t.rbt) break;
#pragma unroll
        for (int h = 0; h < 2; h++)
#pragma unroll
          for (int q = 0; q < 4; q++)
#pragma unroll
            for (int j = 0; j < NU; j++) {
              if (j > 1 && unit(j) >= t.nb_valid) break;
              const f32x4 u = acc[2 * i + h][2 * j], v = acc[2 * i + h][2 * j + 1];
              const u32x2 x = __builtin_amdgcn_permlane16_swap(__float_as_uint(u[q]), __float_as_uint(v[q]), false, false);
              float *dst = y + ((size_t)(t.rb0 + blk) * kRowBlock + 16 * h + row + q) * t.N + col + kRowBlock * unit(j);
              store_output<PAST>(dst, __uint_as_float(x[0]));
              store_output<PAST>(dst + 4 * (size_t)t.N, __uint_as_float(x[1]));
            }
      }
    }
  }
}

// A tile whose row blocks two waves split: rbw of them, MAX at most, are this one's.
template <int MAX, int NU, int LB, typename R, bool GATE_UP, bool STREAM, bool PAST>
__device__ __forceinline__ void split_rows(const Tile &t, uint32_t lds0, int rbw) {
  switch (rbw) {
    case 0: wave_tile<0, 0, 2, NU, LB, R, GATE_UP, STREAM, PAST>(t, lds0); break;
    case 1: wave_tile<1, 1, 2, NU, LB, R, GATE_UP, STREAM, PAST>(t, lds0); break;
    case 2: wave_tile<2, 2, 2, NU, LB, R, GATE_UP, STREAM, PAST>(t, lds0); break;
    case MAX: wave_tile<MAX, MAX, 2, NU, LB, R, GATE_UP, STREAM, PAST>(t, lds0); break;
    default:
      if constexpr (MAX > 3) wave_tile<3, 3, 2, NU, LB, R, GATE_UP, STREAM, PAST>(t, lds0);
  }
}

template <bool GATE_UP, bool STREAM, bool PAST>
__global__ __launch_bounds__(kThreads, 2) void bf16_gemm_kernel(const char *__restrict__ a, const char *__restrict__ wt,
                                                           const float *__restrict__ ba, const float *__restrict__ bb,
                                                           const TileDesc *__restrict__ tiles,
                                                           const int *__restrict__ totals,
                                                           const int *__restrict__ rowmap, void *__restrict__ out,
                                                           int K, int N, float limit) {
  __shared__ u32x4 lds[kLds / 16];
  const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) u32x4 *)lds;
  const int *bounds = totals + (GATE_UP ? kTotBoundsGateUp : kTotBoundsDown);
  const int xcd = blockIdx.x & (kXcds - 1);
  const int L = bounds[xcd] + (blockIdx.x >> 3);
  if (L >= bounds[xcd + 1]) return;
  const TileDesc tc = tiles[L];
  Tile t;
  t.KB = K / kFragK;
  const int nb_total = (GATE_UP ? 2 * N : N) / kRowBlock;
  t.a = a;
  t.b = wt + (size_t)tc.e * nb_total * t.KB * 1024;
  t.ba = ba + (size_t)tc.e * N;
  t.bb = GATE_UP ? bb + (size_t)tc.e * N : nullptr;
  t.rowmap = rowmap;
  t.out = out;
  t.N = N;
  t.rb0 = tc.rb0;
  t.rbt = tc.rbt;
  t.nb0 = tc.nb0;
  t.nb_valid = tc.nbt;
  t.limit = limit;
  const int w = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
  const int rbw = (t.rbt + 1 - (w >> 2)) >> 1;  // the wave's row blocks where the waves split them in two
  if constexpr (STREAM && PAST) {
    if (t.nb_valid > kGemmTileNb) {  // plans for these loads and stores only (bf16_wide_tiles)
      switch (w >> 1) {
        case 0: split_rows<3, 3, 3, Wide, GATE_UP, STREAM, PAST>(t, lds0, rbw); break;
        case 1: split_rows<3, 2, 3, Wide, GATE_UP, STREAM, PAST>(t, lds0, rbw); break;
        case 2: split_rows<3, 2, 2, Wide, GATE_UP, STREAM, PAST>(t, lds0, rbw); break;
        default: split_rows<3, 3, 2, Wide, GATE_UP, STREAM, PAST>(t, lds0, rbw); break;
      }
      return;
    }
  }
  if (t.nb_valid > 4) {
    split_rows<4, 2, 2, Square, GATE_UP, STREAM, PAST>(t, lds0, rbw);
  } else if (t.nb_valid > 2) {
    if (t.rbt <= 4) wave_tile<1, 2, 4, 2, 2, Square, GATE_UP, STREAM, PAST>(t, lds0);
    else wave_tile<2, 4, 4, 2, 2, Square, GATE_UP, STREAM, PAST>(t, lds0);
  } else {
    if (t.rbt <= 4) wave_tile<1, 2, 8, 2, 2, Square, GATE_UP, STREAM, PAST>(t, lds0);
    else wave_tile<1, 4, 8, 2, 2, Square, GATE_UP, STREAM, PAST>(t, lds0);
  }
}

template <bool GATE_UP>
hipError_t launch(const void *a, const void *w, const float *ba, const float *bb, const DispatchBuffers &d, void *out,
                  int K, int N, float limit, int T, int E, int tile_rows, bool wide, bool stream, hipStream_t s) {
  const int nb_total = (GATE_UP ? 2 * N : N) / kRowBlock;
  const int n_ct = (nb_total + kGemmTileNb - 1) / kGemmTileNb;
  const int grid = kXcds * xcd_tile_cap(gemm_tile_cap(T, E, tile_rows) * n_ct);
  const TileDesc *tiles = GATE_UP ? d.tiles_gate_up : d.tiles_down;
  const char *ac = static_cast<const char *>(a), *wc = static_cast<const char *>(w);
#define MOE_GEMM(STREAM, PAST)                                                                                   \
  bf16_gemm_kernel<GATE_UP, STREAM, PAST><<<grid, kThreads, 0, s>>>(ac, wc, ba, bb, tiles, d.totals, d.rowmap, out, K, \
                                                                    N, limit)
  if (wide || (stream && bf16_stores_past(GATE_UP, E * n_ct, T, E))) MOE_GEMM(true, true);
  else if (stream) MOE_GEMM(true, false);
  else MOE_GEMM(false, false);
#undef MOE_GEMM
  return hipGetLastError();
}

}  // namespace

hipError_t launch_bf16_gate_up(const uint16_t *x, const void *w1, const float *b1g, const float *b1u,
                               const DispatchBuffers &d, uint16_t *act, int H, int IM, float limit, int T, int E,
                               int tile_rows, bool wide, bool stream, hipStream_t s) {
  return launch<true>(x, w1, b1g, b1u, d, act, H, IM, limit, T, E, tile_rows, wide, stream, s);
}

hipError_t launch_bf16_down(const uint16_t *act, const void *w2, const float *b2, const DispatchBuffers &d, float *y,
                            int H, int IM, int T, int E, int tile_rows, bool wide, bool stream, hipStream_t s) {
  return launch<false>(act, w2, b2, nullptr, d, y, IM, H, 0.f, T, E, tile_rows, wide, stream, s);
}

}  // namespace moe

// Device code shared by the grouped GEMMs with MXFP4 weights (gemm.hip, gemm_fp4.hip).
#pragma once

#include <type_traits>
#include <utility>

#include "moe_internal.h"
#include "swiglu.h"

namespace moe {

template <int V>
using IC = std::integral_constant<int, V>;

// f(IC<0>{}), f(IC<1>{}), ..., f(IC<N-1>{})
template <typename F, int... I>
__device__ __forceinline__ void static_for_impl(F &&f, std::integer_sequence<int, I...>) {
  (f(IC<I>{}), ...);
}
template <int N, typename F>
__device__ __forceinline__ void static_for(F &&f) {
  static_for_impl(f, std::make_integer_sequence<int, N>{});
}

// f(IC<0>{}), ..., f(IC<left-1>{}) for left <= N, each inside the condition of the one before it: no
// path leaves out a step in front of one that runs.
template <int N, int U = 0, typename F>
__device__ __forceinline__ void static_left(int left, F &&f) {
  if constexpr (U < N) {
    if (left > U) {
      f(IC<U>{});
      static_left<N, U + 1>(left, f);
    }
  }
}

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));

typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

// Row split of a column tile with nb_valid of its NW * NBW column blocks inside
// the matrix: 4 when a quarter of the waves have columns, 2 when half have.
__host__ __device__ inline int row_split_of(int nb_valid, int nw, int nbw) {
  const int waves = (nb_valid + nbw - 1) / nbw;
  return (nw == 4 && waves == 1) ? 4 : ((nw == 4 && waves == 2) ? 2 : 1);
}

// Maps the workgroup id to a tile (see "Tile order" above): two dependent
// loads, the XCD's range and the tile's descriptor.  Returns false for the
// surplus workgroups of the upper-bound grid.  A wide plan (tile_width; a handle with layers of both formats,
// dispatched before the layer is named) has two workgroups to a tile, for its first column blocks and the rest.
__device__ __forceinline__ bool locate_tile(const TileDesc *__restrict__ tiles,
                                            const int *__restrict__ bounds, TileDesc &d) {
  const int bid = blockIdx.x;
  const int xcd = bid & (kXcds - 1);
  const int L = bounds[xcd] + (bid >> 3);
  if (L >= bounds[xcd + 1]) return false;
  d = tiles[L];
  const int first = blockIdx.y * kGemmTileNb, nbt = min(d.nbt - first, kGemmTileNb);
  d.nb0 += first;
  d.nbt = (uint16_t)nbt;
  return nbt > 0;
}

// ---- vector-memory instructions of the main loop ----

// 16 bytes per lane from global memory straight into LDS at base + 16*lane
// (global_load_lds_dwordx4; the LDS base must be wave-uniform).
__device__ __forceinline__ void dma_to_lds_16(const uint4 *g, uint4 *lds_wave_base) {
  __builtin_amdgcn_global_load_lds(g, lds_wave_base, 16, 0, 0);
}

// 16 bytes of the column operand.  STREAM: past the caches (see gemm_streams_weights).
template <bool STREAM>
__device__ __forceinline__ u32x4 load_cols(const uint4 *g) {
  const u32x4 *v = reinterpret_cast<const u32x4 *>(g);
  if constexpr (STREAM) return __builtin_nontemporal_load(v);
  return *v;
}

// s_waitcnt with only the vector-memory counter constrained (gfx9 encoding).
// Loads return in order, so "at most n outstanding" means "all but the newest n
// have landed".  The compiler places its own waits before the first use of
// loaded data in the same wave; these explicit ones stand before the barriers,
// where other waves are about to read what this wave's DMA wrote.
#define WAIT_VMCNT(n) \
  __builtin_amdgcn_s_waitcnt(((n) & 0xf) | (((n) >> 4) << 14) | (0x7 << 4) | (0xf << 8))

// Workgroup barrier that orders LDS traffic only.  A __syncthreads (or a
// workgroup fence) would also drain the vector-memory counter and with it the
// loads of the steps still in flight.  The memory clobber keeps the compiler
// from moving memory accesses across the barrier.
__device__ __forceinline__ void lds_barrier() {
  asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
}

template <int R>
struct StageRing {
  uint4 *p[R];
};

// NW waves side by side over the columns, NBW column blocks per wave, R ring
// slots (LDS stages for the row operand, register slots for the column operand),
// tiles of up to RBT_MAX row blocks, WGS workgroups per CU.
template <int NW_, int NBW_, int R_, int RBT_MAX_, int WGS_>
struct GemmCfg {
  static constexpr int NW = NW_, NBW = NBW_, R = R_, RBT_MAX = RBT_MAX_, WGS = WGS_, KPS = 2;
  static constexpr int THREADS = NW * 64;
  static constexpr int TILE_NB = NW * NBW;              // column blocks per tile
  static constexpr int STAGE = RBT_MAX * KPS * 64;      // uint4 per LDS stage (16 KB at 8 row blocks)
  static constexpr int EPI_LD = NBW * 32 + 8;            // floats per buffered output row
  static constexpr int EPI_WAVE = 32 * EPI_LD / 4;       // uint4 per wave of epilogue buffer
};

// double stages of the row operand in gemm_tile_gl (3: 96 KB of LDS, 4: 128 KB)
constexpr int kLineStages = 4;

}  // namespace moe

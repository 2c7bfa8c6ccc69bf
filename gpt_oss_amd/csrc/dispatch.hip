// Token -> expert dispatch: LDS histogram, prefix sum, stable permutation and
// the tile plan of the grouped GEMMs, and the combine that ends the layer.  Replaces
// count_expert_assignments_kernel, exclusive_scan_small_kernel and
// build_expert_assignments_kernel (utility/utility.cpp:1058-1106, :758-777),
// whose order inside an expert segment is the order global atomics happen to
// resolve in (utility.cpp:1101).  Here the order is fixed: inside a segment
// assignments are sorted by token index, then by slot.  No global atomics.
#include "moe_internal.h"

namespace moe {

constexpr int kDispThreads = 256;  // tokens per workgroup in count / scatter
typedef float f32x4 __attribute__((ext_vector_type(4)));

// Pass 1 of batches beyond kOnceTokens: per-workgroup histogram of expert ids over active rows.  Also resets
// rowmap and perm to -1 (a fill kernel rather than a memset so that the call
// sequence can be captured in a graph).
__global__ __launch_bounds__(kDispThreads) void dispatch_count_kernel(
    const int *__restrict__ topk_i, const int *__restrict__ pos, int T, int E,
    int *__restrict__ blk_counts, int *__restrict__ rowmap, int a_pad_cap, int *__restrict__ perm) {
  __shared__ int hist[256];
  const int tid = threadIdx.x;
  hist[tid] = 0;
  __syncthreads();
  const int t = blockIdx.x * kDispThreads + tid;
  if (t < T && !(pos && pos[t] < 0)) {
    const int4 ids = *reinterpret_cast<const int4 *>(topk_i + (size_t)t * kTopK);
    const int id[kTopK] = {ids.x, ids.y, ids.z, ids.w};
#pragma unroll
    for (int k = 0; k < kTopK; k++) {
      if (id[k] >= 0 && id[k] < E) atomicAdd(&hist[id[k]], 1);
    }
  }
  __syncthreads();
  if (tid < E) blk_counts[(size_t)blockIdx.x * E + tid] = hist[tid];
  for (int i = blockIdx.x * kDispThreads + tid; i < a_pad_cap; i += gridDim.x * kDispThreads)
    rowmap[i] = -1;
  for (int i = blockIdx.x * kDispThreads + tid; i < T * kTopK; i += gridDim.x * kDispThreads)
    perm[i] = -1;
}

// An expert's part of the plan, held in LDS for the workgroup's own use.
struct ExpertPlan {
  int row0;       // first padded row of the expert's segment (multiple of 32)
  int n_mt;       // number of row tiles
  int rb;         // row blocks of the expert's shorter tiles (0..8)
  int extra;      // its first `extra` tiles have rb + 1 row blocks
  int tiles0[2];  // tiles of all lower experts in the sequences of gate_up and down
};

// Where the plan of a batch goes, and what it is of.
struct PlanOut {
  int *offsets;
  int *totals;
  TileDesc *tiles_gate_up, *tiles_down;
  int tile_cap_gate_up, tile_cap_down;
  int tile_rb;  // row blocks of the tallest tile
  int nb[2];    // column blocks of an expert's matrices, gate_up and down (0: no tile tables)
  bool wide;    // tile_width
  TileCost cost;
  // column tiles of GEMM g over an expert whose tallest tile has so many row blocks
  __device__ __forceinline__ int col_tiles(int g, int height) const {
    return tile_width(height, wide) == kGemmTileNb ? (nb[g] + kGemmTileNb - 1) / kGemmTileNb
                                                   : (nb[g] + kWideTileNb - 1) / kWideTileNb;
  }
};

// The tiles of expert ee in the tile sequences of both GEMMs.  An expert's row
// tiles are taken in groups of at most kRowTileGroup (sizes as even as they go);
// tile L = (expert, group, column tile, row tile of the group), row tile fastest.
// The 32 CUs of an XCD then run a few column tiles of one group at a time: the
// group's rows are fetched once per generation of tiles instead of once per
// column tile (an expert with 28 row tiles otherwise streams all its rows
// through the 4 MB L2 for each of its 23 column tiles).  Measured at 7168 tokens
// with Zipf routing: the gate_up GEMM's reads from beyond L2 3.78 -> 2.77 GB, the
// down GEMM's 1.75 -> 1.51 GB, durations unchanged; experts with up to
// kRowTileGroup row tiles (even routing at 4096 tokens) are laid out as before.
// One wave; its lanes run over the expert's tiles of both GEMMs in one sweep.
__device__ __forceinline__ void write_expert_tiles(int ee, const ExpertPlan p, int lane, const PlanOut &out) {
  const int nmt = p.n_mt, rbe = p.rb, exe = p.extra, rowblk = p.row0 / kRowBlock;
  if (nmt == 0) return;
  const int height = rbe + (exe ? 1 : 0), width = tile_width(height, out.wide);
  const int n_ct_up = out.col_tiles(0, height), n_ct_down = out.col_tiles(1, height);
  const int n_up = nmt * n_ct_up, n = n_up + nmt * n_ct_down;
  for (int ii = lane; ii < n; ii += 64) {
    const bool g = ii >= n_up;
    const int i = g ? ii - n_up : ii;
    const int L = (g ? p.tiles0[1] : p.tiles0[0]) + i;
    const int n_ct = g ? n_ct_down : n_ct_up;
    const int n_grp = (nmt + kRowTileGroup - 1) / kRowTileGroup;
    const int gs = nmt / n_grp, gx = nmt - gs * n_grp;  // the first gx groups hold gs + 1 row tiles
    const int big = gx * (gs + 1) * n_ct;               // tiles of those groups
    int grp, r, gsz;
    if (i < big) {
      grp = i / ((gs + 1) * n_ct);
      r = i - grp * (gs + 1) * n_ct;
      gsz = gs + 1;
    } else {
      grp = gx + (i - big) / (gs * n_ct);
      r = (i - big) - (grp - gx) * gs * n_ct;
      gsz = gs;
    }
    const int nt = r / gsz;
    const int mt = grp * gs + min(grp, gx) + (r - nt * gsz);
    TileDesc d;
    d.e = ee;
    d.nb0 = nt * width;
    d.nbt = (uint16_t)min(width, out.nb[g] - nt * width);
    d.rbt = (uint16_t)(rbe + (mt < exe ? 1 : 0));
    d.rb0 = rowblk + mt * rbe + min(mt, exe);
    if (L < (g ? out.tile_cap_down : out.tile_cap_gate_up)) (g ? out.tiles_down : out.tiles_gate_up)[L] = d;
  }
}

// The plan of one batch from the experts' row counts (thread e < 256 holds expert e's count; all threads of the
// workgroup call this together, those from 256 on only take part in the barriers).  Returns the
// expert's part; the rows of all lower experts and of all experts go where the pointers say.
// write_global: this workgroup stores the plan (offsets, padded rows,
// XCD bounds); the others only need the values returned to them.
__device__ __forceinline__ ExpertPlan build_plan(int count, int E, const PlanOut &out, bool write_global,
                                                 int *ex_count_out, int *tot_count_out) {
  constexpr int kSums = 5, kSumsPlan = 2;  // the last ones are of the tile tables
  __shared__ int sh_wave[4][kSums];  // [wave][quantity]: the waves' sums
  __shared__ int sh_mt[257], sh_rb[257];  // exclusive prefixes of the experts' row tiles and row blocks
  __shared__ int sh_tiles[2][257];        // ... and tiles in either GEMM
  __shared__ int sh_bound[2][kXcds + 1];
  const int e = threadIdx.x;
  const int lane = e & 63;
  const int w = e >> 6;
  int *offsets = out.offsets;
  int *totals = out.totals;
  const int n_rb = (count + kRowBlock - 1) / kRowBlock;
  const int n_mt = (n_rb + out.tile_rb - 1) / out.tile_rb;
  const int rb = n_mt ? n_rb / n_mt : 0;
  const int extra = n_mt ? n_rb - rb * n_mt : 0;
  const int height = rb + (extra ? 1 : 0);
  const bool tables = out.nb[0] > 0;
  const int n_up = n_mt * out.col_tiles(0, height), n_down = n_mt * out.col_tiles(1, height);
  // Exclusive prefix sums over the experts of five quantities at once: rows,
  // padded rows, row tiles, tiles of either GEMM.  In a wave by lane shifts, across the four
  // waves through LDS.
  const int own[kSums] = {count, n_rb * kRowBlock, n_mt, n_up, n_down};
  int incl[kSums];
#pragma unroll
  for (int i = 0; i < kSums; i++) incl[i] = own[i];
#pragma unroll
  for (int off = 1; off < 64; off <<= 1) {
#pragma unroll
    for (int i = 0; i < kSums; i++) {
      if (i >= kSumsPlan && !tables) break;
      const int up = __shfl_up(incl[i], off, 64);
      if (lane >= off) incl[i] += up;
    }
  }
  if (lane == 63 && w < 4) {
#pragma unroll
    for (int i = 0; i < kSums; i++) sh_wave[w][i] = incl[i];
  }
  __syncthreads();
  int ex[kSums], tot[kSums];
#pragma unroll
  for (int i = 0; i < kSums; i++) {
    int below = 0, all = 0;
#pragma unroll
    for (int ww = 0; ww < 4; ww++) {
      const int v = sh_wave[ww][i];
      below += ww < w ? v : 0;
      all += v;
    }
    ex[i] = below + incl[i] - own[i];
    tot[i] = all;
  }
  const int ex_count = ex[0], ex_pad = ex[1], ex_mt = ex[2];
  const int tot_count = tot[0], tot_pad = tot[1], tot_mt = tot[2];
  const ExpertPlan mine = {ex_pad, n_mt, rb, extra, {ex[3], ex[4]}};
  *ex_count_out = ex_count;
  *tot_count_out = tot_count;
  if (write_global) {
    if (e < E) offsets[e] = ex_count;
    if (e == 0) {
      offsets[E] = tot_count;
      totals[kTotRows] = tot_pad;
    }
  }
  // Without column tiles (stream.hip) the XCDs' ranges are of no tiles: their search and its
  // divisions are left out (us per call, 128 experts, 200 tokens 313.8 / 310.0; 512 x 512, 32 experts, 128
  // tokens 35.7 / 33.8).
  if (!write_global || !tables) return mine;  // (the same for the whole workgroup)
  if (e < 256) {
    sh_mt[e] = ex_mt;
    sh_rb[e] = ex_pad / kRowBlock;
    sh_tiles[0][e] = ex[3];
    sh_tiles[1][e] = ex[4];
  }
  if (e == 0) {
    sh_mt[256] = tot_mt;
    sh_rb[256] = tot_pad / kRowBlock;
    sh_tiles[0][256] = tot[3];
    sh_tiles[1][256] = tot[4];
  }
  __syncthreads();
  // Lane (c, g, x) of the first wave: boundary x of GEMM g = first tile at which the cost so far reaches x/8 of the
  // total (an expert's tiles taken as equally dear: their heights differ by one block at most), with candidate c
  // for the fixed part of a tile's cost.
  if (w == 0) {
    const int c = e >> 5, g = (e >> 4) & 1, x = min(e & 15, kXcds);
    const int fixed = c ? out.cost.few : out.cost.fixed;
    // cost of kGemmTileNb column blocks' worth of the row tiles of all lower experts: of tiles of any width, whose
    // cost goes by it
    auto cost_of = [&](int part, int i) { return part * sh_mt[i] + kCostPerRowBlock * sh_rb[i]; };
    const int total_tiles = tot[3 + g], tot_cost = cost_of(fixed, 256);
    const long long target = (long long)tot_cost * x;  // kXcds times the cost in front of the boundary
    // last expert whose first tile starts at or before the target
    int lo = 0, hi = 255;
    while (lo < hi) {
      const int mid = (lo + hi + 1) >> 1;
      if ((long long)cost_of(fixed, mid) * kXcds <= target) lo = mid; else hi = mid - 1;
    }
    const int c_e = cost_of(fixed, lo + 1) - cost_of(fixed, lo);  // > 0 in front of the end: an expert with tiles
    const int n_e = sh_tiles[g][lo + 1] - sh_tiles[g][lo];
    const long long rest = target - (long long)cost_of(fixed, lo) * kXcds;  // of kXcds * c_e, the expert's share
    int k = c_e ? min((int)((float)rest / ((float)c_e * kXcds) * (float)n_e), n_e) : 0;  // its tiles in front
    int bound = sh_tiles[g][lo] + k;
    if (x == kXcds) bound = total_tiles;
    // Few rounds (see TileCost): the slowest XCD's time, as its rounds of tiles of its mean cost, decides.
    bool few = false;
    if (out.cost.few && total_tiles <= out.cost.rounds * kCus) {
      const int slow = out.cost.slow;
      const float before = x == kXcds ? (float)cost_of(slow, 256)
                                      : (float)cost_of(slow, lo) +
                                            (n_e ? (float)k * (float)(cost_of(slow, lo + 1) - cost_of(slow, lo)) / (float)n_e
                                                 : 0.f);
      const int n = __shfl_down(bound, 1, 16) - bound;
      const float sum = __shfl_down(before, 1, 16) - before;
      constexpr int kCusPerXcd = kCus / kXcds;
      float time = (e & 15) < kXcds && n > 0 ? (float)((n + kCusPerXcd - 1) / kCusPerXcd) * sum / (float)n : 0.f;
#pragma unroll
      for (int off = 1; off < 16; off <<= 1) time = fmaxf(time, __shfl_xor(time, off, 16));
      const float other = __shfl_xor(time, 32, 64);
      few = (c ? time : other) < out.cost.gain * (c ? other : time);
    }
    if (c == (few ? 1 : 0) && (e & 15) <= kXcds) sh_bound[g][x] = bound;
  }
  __syncthreads();
  // keep every range within what the launch grid provides for (xcd_tile_cap)
  if (e < 2) {
    const int total_tiles = tot[3 + e];
    const int cap = xcd_tile_cap(total_tiles);
    int *bounds = totals + (e ? kTotBoundsDown : kTotBoundsGateUp);
    int prev = 0, want[kXcds];
#pragma unroll
    for (int x = 1; x < kXcds; x++) want[x] = sh_bound[e][x];
    bounds[0] = 0;
#pragma unroll
    for (int x = 1; x < kXcds; x++) {
      int bnd = want[x];
      bnd = max(bnd, max(prev, total_tiles - (kXcds - x) * cap));
      bnd = min(bnd, prev + cap);
      bounds[x] = bnd;
      prev = bnd;
    }
    bounds[kXcds] = total_tiles;
  }
  return mine;
}

// The row-tile plan (see build_plan): an expert with M rows has ceil(M / 32) row
// blocks, cut into n_mt = ceil(row blocks / tile_rb) tiles as evenly as they go: the
// first `extra` tiles are rb + 1 row blocks high, the others rb.  Its segment in
// the padded row space is its row blocks and no more, so an expert pads to at
// most 31 rows.  The tile sequence of either GEMM (n_ct column tiles per row
// tile) is cut into the 8 ranges of the XCDs by estimated cost: a tile of r row
// blocks costs TileCost's fixed part + kCostPerRowBlock * r.

// Ranks inside one wave: for each of the lane's kTopK expert ids, how many of
// the wave's assignments to the same expert come before it in (lane, slot)
// order, and how many there are in all.  Instead of a loop over the experts
// (kTopK ballots each), the ids are compared bit plane by bit plane: one ballot
// per slot and bit of the id, then a lane's id selects plane or complement and
// the AND over the planes is the mask of the lanes that hold the same id in
// that slot.  The work no longer grows with the number of experts (4 x faster
// at 128).  Ids < 0 match nothing; their results are not used.
template <int NBITS>
struct IdPlanes {
  unsigned long long valid[kTopK], plane[kTopK][NBITS];
  __device__ __forceinline__ explicit IdPlanes(const int (&id)[kTopK]) {
#pragma unroll
    for (int k = 0; k < kTopK; k++) {
      valid[k] = __ballot(id[k] >= 0);
#pragma unroll
      for (int b = 0; b < NBITS; b++) plane[k][b] = __ballot(id[k] >= 0 && ((id[k] >> b) & 1));
    }
  }
  // lanes that hold expert e in slot k
  __device__ __forceinline__ unsigned long long holders(int k, int e) const {
    unsigned long long m = valid[k];
#pragma unroll
    for (int b = 0; b < NBITS; b++) m &= ((e >> b) & 1) ? plane[k][b] : ~plane[k][b];
    return m;
  }
};
template <int NBITS>
__device__ __forceinline__ void wave_ranks(const IdPlanes<NBITS> &p, const int (&id)[kTopK], int lane,
                                           int (&rank)[kTopK], int (&total)[kTopK]) {
  const unsigned long long me = 1ull << lane;
  const unsigned long long lt = me - 1ull;
#pragma unroll
  for (int k = 0; k < kTopK; k++) {
    int r = 0, n = 0;
#pragma unroll
    for (int k2 = 0; k2 < kTopK; k2++) {
      const unsigned long long m = p.holders(k2, id[k]);
      n += __popcll(m);
      r += __popcll(m & lt);             // lower lanes, any slot
      if (k2 < k) r += (m & me) ? 1 : 0;  // this lane, lower slots
    }
    rank[k] = r;
    total[k] = n;
  }
}

// Pass 2 of batches beyond kOnceTokens: the plan and the stable permutation in one launch.  Every workgroup
// adds up the per-workgroup counts of pass 1 itself (at most a few dozen loads
// per expert): the experts' totals, from which it derives offsets and padded
// first rows exactly as every other does, and the counts of the workgroups
// before it, its own base inside every expert.  One more workgroup, the last, stores the
// plan for the GEMMs, whose search for the XCDs' bounds the others need not wait for.
// Rank of an assignment inside its expert = (assignments of lower workgroups)
// + (lower waves of this workgroup) + (lower lanes of this wave) + (lower slots
// of this token), all for the same expert.
template <int NBITS>
__global__ __launch_bounds__(kDispThreads) void dispatch_scatter_kernel(
    const int *__restrict__ topk_i, const int *__restrict__ pos, int T, int E,
    const int *__restrict__ blk_counts, int n_blk, int *__restrict__ perm, int *__restrict__ rowmap,
    int *__restrict__ inv, int *__restrict__ blk_expert, PlanOut plan) {
  __shared__ int wave_cnt[kDispThreads / 64][256];
  __shared__ int sh_base[256], sh_off[256];
  __shared__ ExpertPlan sh_plan[256];
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int w = tid >> 6;
  // the token's ids first: their loads run while the counts are added up
  const int t = blockIdx.x * kDispThreads + tid;
  int id[kTopK] = {-1, -1, -1, -1};
  if (t < T && !(pos && pos[t] < 0)) {
    const int4 ids = *reinterpret_cast<const int4 *>(topk_i + (size_t)t * kTopK);
    id[0] = ids.x; id[1] = ids.y; id[2] = ids.z; id[3] = ids.w;
#pragma unroll
    for (int k = 0; k < kTopK; k++)
      if (id[k] >= E) id[k] = -1;
  }
  int count = 0, base = 0;
  if (tid < E) {
    for (int b0 = 0; b0 < n_blk; b0 += 16) {  // 16 independent loads at a time
      int c[16];
#pragma unroll
      for (int i = 0; i < 16; i++) c[i] = b0 + i < n_blk ? blk_counts[(size_t)(b0 + i) * E + tid] : 0;
#pragma unroll
      for (int i = 0; i < 16; i++) {
        if (b0 + i < (int)blockIdx.x) base += c[i];
        count += c[i];
      }
    }
  }
  int ex_count, tot_count;
  const ExpertPlan mine = build_plan(count, E, plan, /*write_global=*/(int)blockIdx.x == n_blk, &ex_count, &tot_count);
  if ((int)blockIdx.x == n_blk) return;
  sh_base[tid] = base;
  sh_off[tid] = ex_count;
  sh_plan[tid] = mine;
  for (int e = tid; e < (kDispThreads / 64) * 256; e += kDispThreads) (&wave_cnt[0][0])[e] = 0;
  int rank[kTopK], total[kTopK];
  wave_ranks(IdPlanes<NBITS>(id), id, lane, rank, total);
  __syncthreads();
  // The tile sequences of the GEMMs: the waves of all workgroups take the
  // experts in turn.
  for (int ee = blockIdx.x * (kDispThreads / 64) + w; ee < E; ee += n_blk * (kDispThreads / 64)) {
    write_expert_tiles(ee, sh_plan[ee], lane, plan);
  }
#pragma unroll
  for (int k = 0; k < kTopK; k++)
    if (id[k] >= 0) wave_cnt[w][id[k]] = total[k];  // the same value from every lane that holds the id
  __syncthreads();
  if (t >= T) return;
  int out_inv[kTopK];
#pragma unroll
  for (int k = 0; k < kTopK; k++) {
    const int e = id[k];
    const int a = t * kTopK + k;
    if (e < 0) { out_inv[k] = -1; continue; }
    int r = sh_base[e] + rank[k];
    for (int ww = 0; ww < w; ww++) r += wave_cnt[ww][e];
    const int prow = sh_plan[e].row0 + r;
    perm[sh_off[e] + r] = a;
    rowmap[prow] = a;
    if (blk_expert && prow % kRowBlock == 0) blk_expert[prow / kRowBlock] = e;
    out_inv[k] = prow;
  }
  *reinterpret_cast<int4 *>(inv + (size_t)t * kTopK) =
      make_int4(out_inv[0], out_inv[1], out_inv[2], out_inv[3]);
}

// Both passes in one launch for batches of at most kOnceGroups x 64 tokens: every workgroup counts the whole
// batch, 64 tokens to a wave (lane l counts experts l, l + 64, ...: the holders of each are a mask of
// bits, see IdPlanes), so that it needs no launch in front, and scatters 256 tokens, one wave
// to a SIMD.  One more workgroup, the last, stores the plan.  Same result as the two launches, bit for bit.
// Bound by latency: a launch and a chain of LDS steps.  us of the stage in a call, two launches (one
// workgroup up to 256 tokens) / this: 200 tokens 14.3 / 10.7, 512 15.5 / 9.8, 896 14.5 / 10.4, 1900 14.6 / 12.2; 128
// experts, 1000 tokens 18.5 / 13.5.  Every further 1024 tokens are another round of counting, at 4096
// tokens nothing is left of the gain (14.8 with two launches).
constexpr int kOnceThreads = 1024, kOnceWaves = kOnceThreads / 64;
constexpr int kOnceRounds = 2, kOnceGroups = kOnceRounds * kOnceWaves;
constexpr int kOnceTokens = 64 * kOnceGroups;

template <int NBITS>
__global__ __launch_bounds__(kOnceThreads) void dispatch_once_kernel(
    const int *__restrict__ topk_i, const int *__restrict__ pos, int T, int E, PlanOut plan, int n_blk,
    int *__restrict__ perm, int *__restrict__ rowmap, int *__restrict__ inv, int *__restrict__ blk_expert) {
  __shared__ int cnt[kOnceGroups][256];  // per group of 64 tokens and expert: count, then the rows before the group's
  __shared__ int sh_off[256];
  __shared__ ExpertPlan sh_plan[256];
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int groups = (T + 63) / 64;
  int4 ids[kOnceRounds];
#pragma unroll
  for (int r = 0; r < kOnceRounds; r++) {
    const int t = (w + r * kOnceWaves) * 64 + lane;
    ids[r] = make_int4(-1, -1, -1, -1);
    if (t < T && !(pos && pos[t] < 0)) ids[r] = *reinterpret_cast<const int4 *>(topk_i + (size_t)t * kTopK);
  }
  int own[kTopK] = {-1, -1, -1, -1}, rank[kTopK], total[kTopK], own_group = -1;
#pragma unroll 1
  for (int r = 0; r < kOnceRounds; r++) {
    const int g = w + r * kOnceWaves;
    if (g >= groups) break;
    static_assert(kOnceRounds == 2, "which round's ids");
    const int4 v = r ? ids[1] : ids[0];
    int id[kTopK] = {v.x, v.y, v.z, v.w};
#pragma unroll
    for (int k = 0; k < kTopK; k++)
      if (id[k] >= E) id[k] = -1;
    const IdPlanes<NBITS> planes(id);
    for (int e = lane; e < E; e += 64) {
      int c = 0;
#pragma unroll
      for (int k = 0; k < kTopK; k++) c += __popcll(planes.holders(k, e));
      cnt[g][e] = c;
    }
    if (g / (kDispThreads / 64) == (int)blockIdx.x) {
      own_group = g;
#pragma unroll
      for (int k = 0; k < kTopK; k++) own[k] = id[k];
      wave_ranks(planes, id, lane, rank, total);
    }
  }
  __syncthreads();
  int count = 0;
  if (tid < E) {
    for (int g = 0; g < groups; g++) {
      const int c = cnt[g][tid];
      cnt[g][tid] = count;
      count += c;
    }
  }
  int ex_count, tot_count;
  const ExpertPlan mine = build_plan(count, E, plan, /*write_global=*/(int)blockIdx.x == n_blk, &ex_count, &tot_count);
  if ((int)blockIdx.x == n_blk) {
    // -1 where the scatter below writes nothing: the padding rows of the experts
    // and the tail of perm that inactive rows and invalid ids leave unused
    if (tid < E) {
      const int end = mine.row0 + (count + kRowBlock - 1) / kRowBlock * kRowBlock;
      for (int i = mine.row0 + count; i < end; i++) rowmap[i] = -1;
    }
    for (int i = tot_count + tid; i < T * kTopK; i += kOnceThreads) perm[i] = -1;
    return;
  }
  if (tid < E) {
    sh_off[tid] = ex_count;
    sh_plan[tid] = mine;
  }
  __syncthreads();
  if (plan.nb[0] > 0) {  // the tile sequences of the GEMMs: the waves of all workgroups take the experts in turn
    for (int ee = blockIdx.x * kOnceWaves + w; ee < E; ee += n_blk * kOnceWaves)
      write_expert_tiles(ee, sh_plan[ee], lane, plan);
  }
  const int t = own_group * 64 + lane;
  if (own_group < 0 || t >= T) return;
  int out_inv[kTopK];
#pragma unroll
  for (int k = 0; k < kTopK; k++) {
    const int e = own[k];
    if (e < 0) { out_inv[k] = -1; continue; }
    const int rk = cnt[own_group][e] + rank[k];
    const int prow = sh_plan[e].row0 + rk;
    perm[sh_off[e] + rk] = t * kTopK + k;
    rowmap[prow] = t * kTopK + k;
    if (blk_expert && prow % kRowBlock == 0) blk_expert[prow / kRowBlock] = e;
    out_inv[k] = prow;
  }
  *reinterpret_cast<int4 *>(inv + (size_t)t * kTopK) = make_int4(out_inv[0], out_inv[1], out_inv[2], out_inv[3]);
}

// out[t,:] (+)= sum_k topk_v[t,k] * y[inv[t,k],:], slots added in order 0..3
// (descending router score, as reduce_mlp2_slots_kernel does,
// utility/utility.cpp:701-726).  Every token owns its K rows of y, so there
// are no atomics.
//
// RESID: instead of writing the fp32 sum, adds it to the bf16 residual stream
// in place, x = bf16(float(x) + sum) (residual_add_batch_kernel,
// utility/utility.cpp:158-173; call getp_run.cpp:846-852); inactive rows are
// left alone.
//
// One workgroup per token; for few tokens gridDim.y workgroups share its columns
// (a single token: 5.4 -> 2.7 us with that and inv in place of a ballot over the ids).
//
// PAST: y is read past the caches.  Bound by HBM with many tokens: the down GEMM's last rows of a large y are
// all that the caches hold, and nothing reads a row again.  us of this kernel's stage, through / past: 4096
// tokens 41.3 / 41.0 (MXFP4, residual stream, 43.3 / 40.7), 7168 80.1 / 71.1, 6144 at 128 experts, where
// the rows that it leaves in the caches cost the next call as well, 73.1 / 66.5 (1442 / 1412 per call); 1500 (69 MB)
// 19.8 / 20.4.
constexpr size_t kCombinePastBytes = (size_t)128 << 20;
template <bool RESID, bool PAST>
__global__ __launch_bounds__(256) void combine_kernel(const float *__restrict__ y,
                                                     const int *__restrict__ inv,
                                                     const float *__restrict__ topk_v,
                                                     const int *__restrict__ pos, void *outp, int H,
                                                     int ldy, int accumulate) {
  const int t = blockIdx.x;
  const bool active = !(pos && pos[t] < 0);
  if (!active && (accumulate || RESID)) return;
  int p[kTopK] = {-1, -1, -1, -1};
  float w[kTopK] = {0.f, 0.f, 0.f, 0.f};
  if (active) {
    const int4 pi = *reinterpret_cast<const int4 *>(inv + (size_t)t * kTopK);
    const float4 wv = *reinterpret_cast<const float4 *>(topk_v + (size_t)t * kTopK);
    p[0] = pi.x; p[1] = pi.y; p[2] = pi.z; p[3] = pi.w;
    w[0] = wv.x; w[1] = wv.y; w[2] = wv.z; w[3] = wv.w;
  }
  float4 *o = reinterpret_cast<float4 *>(reinterpret_cast<float *>(outp) + (size_t)t * H);
  uint2 *xr = reinterpret_cast<uint2 *>(reinterpret_cast<uint16_t *>(outp) + (size_t)t * H);
  for (int c = blockIdx.y * 256 + threadIdx.x; c < H / 4; c += gridDim.y * 256) {
    float4 s = (!RESID && accumulate) ? o[c] : make_float4(0.f, 0.f, 0.f, 0.f);
#pragma unroll
    for (int k = 0; k < kTopK; k++) {
      if (p[k] >= 0) {
        const f32x4 *row = reinterpret_cast<const f32x4 *>(y + (size_t)p[k] * ldy);
        const f32x4 v = PAST ? __builtin_nontemporal_load(row + c) : row[c];
        s.x += w[k] * v[0]; s.y += w[k] * v[1]; s.z += w[k] * v[2]; s.w += w[k] * v[3];
      }
    }
    if (RESID) {
      const uint2 xv = xr[c];
      const float r0 = __uint_as_float(xv.x << 16) + s.x, r1 = __uint_as_float(xv.x & 0xffff0000u) + s.y;
      const float r2 = __uint_as_float(xv.y << 16) + s.z, r3 = __uint_as_float(xv.y & 0xffff0000u) + s.w;
      xr[c] = make_uint2(f32_to_bf16_rne(r0) | ((uint32_t)f32_to_bf16_rne(r1) << 16),
                         f32_to_bf16_rne(r2) | ((uint32_t)f32_to_bf16_rne(r3) << 16));
    } else {
      o[c] = s;
    }
  }
}

hipError_t launch_dispatch(const int *topk_i, const int *pos, int T, int E, int nb_gate_up, int nb_down,
                           int tile_rows, bool wide, TileCost tile_cost, const DispatchBuffers &d, hipStream_t s) {
  const int n_blk = (T + kDispThreads - 1) / kDispThreads;
  // Rows of the padded space this batch can reach: every expert rounds its
  // rows up to a multiple of 32.
  const long long A = (long long)T * kTopK;
  const long long reach = A + (long long)kTileGran * E;
  const int fill_rows = (int)(reach < d.a_pad_cap ? reach : d.a_pad_cap);
  PlanOut plan;
  plan.offsets = d.offsets;
  plan.totals = d.totals;
  plan.tiles_gate_up = d.tiles_gate_up;
  plan.tiles_down = d.tiles_down;
  plan.tile_cap_gate_up = d.tile_cap_gate_up;
  plan.tile_cap_down = d.tile_cap_down;
  plan.tile_rb = tile_rows / kRowBlock;
  plan.nb[0] = nb_gate_up;
  plan.nb[1] = nb_down;
  plan.wide = wide;
  plan.cost = tile_cost;
  // ids are compared in as many bits as the experts have
#define MOE_BY_EXPERTS(LAUNCH)  \
  do {                          \
    if (E <= 32) LAUNCH(5);     \
    else if (E <= 128) LAUNCH(7); \
    else LAUNCH(8);             \
  } while (0)
  if (T <= kOnceTokens) {
#define MOE_ONCE(BITS)                                                                                         \
  dispatch_once_kernel<BITS><<<n_blk + 1, kOnceThreads, 0, s>>>(topk_i, pos, T, E, plan, n_blk, d.perm, d.rowmap, \
                                                                d.inv, d.blk_expert)
    MOE_BY_EXPERTS(MOE_ONCE);
#undef MOE_ONCE
    return hipGetLastError();
  }
  dispatch_count_kernel<<<n_blk, kDispThreads, 0, s>>>(topk_i, pos, T, E, d.blk_counts, d.rowmap,
                                                       fill_rows, d.perm);
#define MOE_SCATTER(BITS)                                                                                         \
  dispatch_scatter_kernel<BITS><<<n_blk + 1, kDispThreads, 0, s>>>(topk_i, pos, T, E, d.blk_counts, n_blk, d.perm, \
                                                               d.rowmap, d.inv, d.blk_expert, plan)
  MOE_BY_EXPERTS(MOE_SCATTER);
#undef MOE_SCATTER
#undef MOE_BY_EXPERTS
  return hipGetLastError();
}

template <bool RESID>
static hipError_t launch_combine_any(const float *y, int ldy, const int *inv, const float *topk_v, const int *pos,
                                     void *out, int T, int H, int accumulate, hipStream_t s) {
  // workgroups of one token each fill the GPU from about four per CU on
  const dim3 grid(T, T < 4 * kCus ? (H / 4 + 255) / 256 : 1);
  if ((size_t)T * kTopK * ldy * sizeof(float) > kCombinePastBytes)
    combine_kernel<RESID, true><<<grid, 256, 0, s>>>(y, inv, topk_v, pos, out, H, ldy, accumulate);
  else
    combine_kernel<RESID, false><<<grid, 256, 0, s>>>(y, inv, topk_v, pos, out, H, ldy, accumulate);
  return hipGetLastError();
}

hipError_t launch_combine(const float *y, int ldy, const int *inv, const float *topk_v, const int *pos, float *out,
                          int T, int H, int accumulate, hipStream_t s) {
  return launch_combine_any<false>(y, ldy, inv, topk_v, pos, out, T, H, accumulate, s);
}

hipError_t launch_combine_residual(const float *y, int ldy, const int *inv, const float *topk_v, const int *pos,
                                   uint16_t *x, int T, int H, hipStream_t s) {
  return launch_combine_any<true>(y, ldy, inv, topk_v, pos, x, T, H, 0, s);
}

}  // namespace moe

// ---- dispatch for callers that cannot allocate ----
//
// moe_dispatch_static runs the same kernels as moe_dispatch, but needs no
// handle and calls no allocating routine: the buffers the kernels use beyond
// the caller's inputs and outputs (per-workgroup counts, the padded row map,
// the inverse map and the plan's totals) live in one
// file-scope device array.  Every GPU the library runs on holds that array
// until the process ends; every call on a GPU shares it, so calls that overlap
// on one GPU (two streams, two threads) race.  The kernels rewrite everything
// they later read, so nothing of an earlier call survives into the next.
namespace moe {
namespace {

constexpr int kStaticMaxTokens = MOE_DISPATCH_STATIC_MAX_TOKENS;
constexpr int kStaticMaxExperts = MOE_DISPATCH_STATIC_MAX_EXPERTS;
constexpr size_t align256(size_t n) { return (n + 255) & ~(size_t)255; }
constexpr size_t kStaticBlkCounts = 0;
constexpr size_t kStaticRowmap =
    kStaticBlkCounts + align256(sizeof(int) * ((kStaticMaxTokens + kDispThreads - 1) / kDispThreads) * kStaticMaxExperts);
constexpr int kStaticPadRows = kStaticMaxTokens * kTopK + kTileGran * kStaticMaxExperts;
constexpr size_t kStaticInv = kStaticRowmap + align256(sizeof(int) * kStaticPadRows);
constexpr size_t kStaticTotals = kStaticInv + align256(sizeof(int) * kStaticMaxTokens * kTopK);
constexpr size_t kStaticBytes = kStaticTotals + align256(sizeof(int) * kTotInts);

static __device__ __align__(256) unsigned char scratch[kStaticBytes];

// Device address of this GPU's copy of `scratch`: looked up once per device
// (each GPU holds its own copy at its own address), never taken from the
// array's name, which on the host is only a stand-in for the symbol.
constexpr int kMaxDevices = 64;
unsigned char *g_scratch_ptr[kMaxDevices];  // written once per device, then only read

hipError_t static_scratch(unsigned char **out) {
  int dev = 0;
  hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess) return e;
  if (dev < 0 || dev >= kMaxDevices) return hipErrorInvalidDevice;
  unsigned char *p = __atomic_load_n(&g_scratch_ptr[dev], __ATOMIC_ACQUIRE);
  if (!p) {
    e = hipGetSymbolAddress(reinterpret_cast<void **>(&p), HIP_SYMBOL(scratch));
    if (e != hipSuccess) return e;
    if (!p) return hipErrorInvalidSymbol;
    __atomic_store_n(&g_scratch_ptr[dev], p, __ATOMIC_RELEASE);  // the same value from every thread
  }
  *out = p;
  return hipSuccess;
}

}  // namespace
}  // namespace moe

extern "C" int moe_dispatch_static(const int *topk_i, const int *pos, int n_tokens, int n_experts,
                                   int *offsets, int *perm, void *stream) {
  using namespace moe;
  if (n_tokens < 0) return set_error(MOE_ERR_BAD_ARG, "n_tokens %d is negative", n_tokens);
  if (n_tokens > kStaticMaxTokens)
    return set_error(MOE_ERR_CAPACITY, "moe_dispatch_static: n_tokens %d exceeds its fixed maximum of %d",
                     n_tokens, kStaticMaxTokens);
  if (n_experts < 1 || n_experts > kStaticMaxExperts)
    return set_error(MOE_ERR_CAPACITY, "moe_dispatch_static: n_experts %d outside [1,%d]", n_experts,
                     kStaticMaxExperts);
  if (!offsets || (n_tokens > 0 && (!topk_i || !perm)))
    return set_error(MOE_ERR_BAD_ARG, "null device pointer");
  unsigned char *base = nullptr;
  const hipError_t e = static_scratch(&base);
  if (e != hipSuccess)
    return set_error(MOE_ERR_HIP, "hipGetSymbolAddress(scratch) failed: %s", hipGetErrorString(e));
  DispatchBuffers d{};
  d.blk_counts = reinterpret_cast<int *>(base + kStaticBlkCounts);
  d.rowmap = reinterpret_cast<int *>(base + kStaticRowmap);
  d.inv = reinterpret_cast<int *>(base + kStaticInv);
  d.totals = reinterpret_cast<int *>(base + kStaticTotals);
  d.offsets = offsets;
  d.perm = perm;
  d.a_pad_cap = kStaticPadRows;
  // no GEMM follows: with no column tiles the plan kernel writes no tile tables
  d.tiles_gate_up = d.tiles_down = nullptr;
  d.tile_cap_gate_up = d.tile_cap_down = 0;
  const hipError_t el = launch_dispatch(topk_i, pos, n_tokens, n_experts, 0, 0, kTileRows, false, TileCost{}, d,
                                       static_cast<hipStream_t>(stream));
  if (el != hipSuccess)
    return set_error(MOE_ERR_HIP, "dispatch launch failed: %s", hipGetErrorString(el));
  return MOE_OK;
}

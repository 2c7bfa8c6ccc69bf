// Router: logits = x * Wr^T + br, top-4 with ties to the lower expert id,
// softmax over the four selected logits.  Replaces matmul_router_kernel
// (matmul/matmul.cpp:945-1019) and fused_topk_softmax_batch_kernel
// (utility/utility.cpp:273-365).  The expert ids must be those of the
// reference's CPU path (run.cpp:356-369 matmul: float products accumulated in a
// double, rounded to float once; :669-671 bias added in float; :388-421 top-k;
// :336-354 softmax), bit for bit.
//
// Two passes in one kernel:
//   1. All logits on the bf16 matrix cores (v_mfma_f32_16x16x32_bf16).  The
//      products are exact; the fp32 accumulation inside the matrix core is not,
//      so a wave hands its fp32 sums over to fp64 accumulators every FLUSH
//      MFMAs (every one while the experts are few and the hand-over is cheap).
//      That bounds the error of a logit by gamma * sum_k |x_k w_ek|
//      <= gamma * |x| * |w_e| (Cauchy-Schwarz; |x|^2 comes out of one more
//      MFMA per chunk, x times its own transpose, and max_e |w_e| is computed
//      at upload).
//   2. A token whose five best logits are further apart than twice that bound
//      is decided: ids, order and (to about 1e-7) weights are those of the
//      exact arithmetic.  For any other token the experts that can still reach
//      the top four -- those within the bound of the fourth best -- get their
//      logit recomputed exactly: float products (exact for bf16 factors)
//      summed in fp64, rounded to float once, bias added in float, which is the
//      arithmetic of run.cpp:363-369 up to the order of the fp64 additions.
//      An expert outside that set is below four experts by more than the two
//      error bounds, so it cannot be among the exact top four; inside the set
//      all values are exact, so the selection (value descending, index
//      ascending) is the reference's.
// At the benchmark shapes a few per cent of the tokens take the second pass,
// with four to six experts each, instead of every token paying fp64 for every
// expert.
#include "moe_internal.h"

namespace moe {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

// Error of one fp32 chain of `flush` MFMAs (of 32 k each) started from zero,
// relative to the sum of the magnitudes of its 32 * flush products: every one
// of its 33 * flush additions is taken to lose at most 2^-23 of the running
// magnitude (covers truncation as well as rounding), and the result is doubled.
__host__ __device__ constexpr float router_gamma(int flush) { return 2.0f * 33.0f * flush * 1.1920929e-7f; }
constexpr int kNone = 0x7fffffff;

// The selection's rule is that of the reference's CPU top-k under a stable sort (run.cpp:388-421): value descending,
// index ascending.  Beside NaNs, which no sort orders, it is that of one walk over the experts left, from the first on,
// where a candidate replaces the incumbent only if it compares strictly greater: the greatest number
// left, but a NaN while it is the first expert left (a row of NaNs selects 0, 1, 2, 3).
//
// A logit as a whole number of the same order, zeros of either sign the same one.
constexpr uint32_t kTakenKey = 0u, kNanKey = 1u;  // below every number's, minus infinity's too
__device__ __forceinline__ uint32_t order_key(float v) {
  const uint32_t u = __float_as_uint(v + 0.f);
  return v != v ? kNanKey : u ^ ((uint32_t)((int32_t)u >> 31) | 0x80000000u);
}
__device__ __forceinline__ float key_value(uint32_t key) {  // kNanKey: a NaN
  return __uint_as_float(key ^ (~(uint32_t)((int32_t)key >> 31) | 0x80000000u));
}

// Among the LPT lanes of a token (a wave, or either half of one): the largest value of each of N tokens, in every lane, and
// the first lane that has something, which one of them does.
template <int LPT, int N>
__device__ __forceinline__ void lanes_max(uint32_t (&x)[N]) {
  static_assert(LPT == 32 || LPT == 64, "a token has a wave or half of one");
#define MOE_DPP_MAX(CTRL, ROWS)                                                                              \
  _Pragma("unroll") for (int n = 0; n < N; n++)                                                               \
    x[n] = max(x[n], (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x[n], CTRL, ROWS, 0xf, false))
  MOE_DPP_MAX(0x111, 0xf);  // row_shr 1, 2, 4, 8: lane 15 of a row of 16 has the row's
  MOE_DPP_MAX(0x112, 0xf);
  MOE_DPP_MAX(0x114, 0xf);
  MOE_DPP_MAX(0x118, 0xf);
  MOE_DPP_MAX(0x142, 0xa);  // row_bcast15 into rows 1 and 3, row_bcast31 into 2 and 3
  if constexpr (LPT == 64) MOE_DPP_MAX(0x143, 0xc);
#undef MOE_DPP_MAX
#pragma unroll
  for (int n = 0; n < N; n++) {
    const uint32_t high = (uint32_t)__builtin_amdgcn_readlane((int)x[n], 63);
    x[n] = LPT == 64 || (threadIdx.x & 32) ? high : (uint32_t)__builtin_amdgcn_readlane((int)x[n], 31);
  }
}
template <int LPT>
__device__ __forceinline__ int first_lane(bool has) {
  const unsigned long long m = __ballot(has);
  return LPT == 64 ? __builtin_ctzll(m) : __builtin_ctz((uint32_t)(m >> (threadIdx.x & 32)));
}

// Top-NSEL of the keys of N tokens side by side, lane q of a token's LPT owning those of experts q*PER .. q*PER+PER-1;
// places past the experts hold kTakenKey.  A round is a maximum over the lanes and the first one that holds it.  NANS:
// there may be NaNs.  All lanes end with the same result, kNone where no expert is left (a whole wave has more than 32).
template <int PER, int LPT, int N, int NSEL, bool NANS>
__device__ __forceinline__ void top_keys(uint32_t (&key)[N][PER], int q, float (&sel_v)[N][NSEL],
                                         int (&sel_i)[N][NSEL]) {
  static_assert(LPT == 64 || PER == 1, "a lane of half a wave has one expert");
#pragma unroll
  for (int r = 0; r < NSEL; r++) {
    uint32_t own[N], best[N];
#pragma unroll
    for (int n = 0; n < N; n++) {
      own[n] = key[n][0];
#pragma unroll
      for (int j = 1; j < PER; j++) own[n] = max(own[n], key[n][j]);
      best[n] = own[n];
    }
    lanes_max<LPT, N>(best);
#pragma unroll
    for (int n = 0; n < N; n++) {
      int l = first_lane<LPT>(own[n] == best[n]);
      if constexpr (NANS) {
        uint32_t first = kTakenKey;  // the lane's first key that is left
#pragma unroll
        for (int j = PER - 1; j >= 0; j--)
          if (key[n][j] != kTakenKey) first = key[n][j];
        const int lf = first_lane<LPT>(first != kTakenKey || best[n] == kTakenKey);
        if (__shfl((int)first, lf, LPT) == (int)kNanKey) {
          best[n] = kNanKey;
          l = lf;
        }
      }
      int at = 0;
#pragma unroll
      for (int j = PER - 1; j >= 0; j--)
        if (key[n][j] == best[n]) at = j;
      sel_v[n][r] = key_value(best[n]);
      if constexpr (LPT == 64) sel_i[n][r] = l * PER + __builtin_amdgcn_readlane(at, l);
      else sel_i[n][r] = best[n] == kTakenKey ? kNone : l;
#pragma unroll
      for (int j = 0; j < PER; j++)
        if (q == l && at == j) key[n][j] = kTakenKey;
    }
  }
}

// N tokens on a whole wave (more than 32 experts).  A chain of latencies, so two tokens go side by side, and their
// softmax and stores, too, on lanes of their own.  us of moe_router, with eight or sixteen lanes per token and
// comparisons / a wave for one token after the other / this: 128 experts of 2880, 24 tokens 16.4 / 16.9 / 14.7, 200 26.4 /
// 23.3 / 21.2, 7168 37.8 / 40.3 / 35.6; of 512, 64 9.6 / 10.3 / 7.7, 7168 21.2 / 22.4 / 17.9; 64 of 512, 64 8.5 / 6.8 / 6.1.
template <int PER, int N, int NSEL>
__device__ __forceinline__ void wave_top(const float (&v)[N][PER], int lane, int E, float (&sel_v)[N][NSEL],
                                         int (&sel_i)[N][NSEL]) {
  bool nan = false;
  uint32_t key[N][PER];
#pragma unroll
  for (int n = 0; n < N; n++)
#pragma unroll
    for (int j = 0; j < PER; j++) {
      key[n][j] = lane * PER + j < E ? order_key(v[n][j]) : kTakenKey;
      nan |= key[n][j] == kNanKey;
    }
  if (__ballot(nan) != 0ull) top_keys<PER, 64, N, NSEL, true>(key, lane, sel_v, sel_i);
  else top_keys<PER, 64, N, NSEL, false>(key, lane, sel_v, sel_i);
}

// Top-NSEL of one token's logits for up to 32 experts, one lane per expert (the
// 32 lanes of a half wave; lane e owns expert e, v = its logit, -inf for a lane
// without an expert).  row4 points at the token's E_pad logits in LDS, 16-byte
// aligned.  The same rule, found by counting instead of five rounds
// of maxima: an expert's place is the number of experts with a greater
// value; the lanes at places 0 .. NSEL-1 post themselves to `post` (LDS, NSEL
// floats then NSEL ints, owned by this token) and every lane reads the list
// back.  Of experts with equal values the lowest index takes the place (an
// atomic minimum) and the place behind it stays empty: an empty place among the
// first NSEL, like a NaN among the logits (which no count orders), sends the
// wave -- the branch is per wave -- through top_keys instead.  Places past the
// number of experts hold kNone.
template <int E_pad, int NSEL>
__device__ __forceinline__ void ranked_top(const float4 *row4, float v, int e, int E, float *post,
                                           float (&sel_v)[NSEL], int (&sel_i)[NSEL]) {
  static_assert(E_pad == 16 || E_pad == 32, "one lane per expert in a half wave");
  int *post_i = reinterpret_cast<int *>(post + NSEL);
  if (e < NSEL) post_i[e] = kNone;
  int place = 0;
#pragma unroll
  for (int j4 = 0; j4 < E_pad / 4; j4++) {
    const float4 o = row4[j4];  // the same address in all lanes of the half wave
    place += (o.x > v ? 1 : 0) + (o.y > v ? 1 : 0) + (o.z > v ? 1 : 0) + (o.w > v ? 1 : 0);
  }
  if (e < E && place < NSEL) {
    post[place] = v;  // equal values: the same float from every writer
    atomicMin(&post_i[place], e);
  }
  // the same wave wrote the list; LDS operations of a wave complete in order
  bool redo = v != v;
#pragma unroll
  for (int r = 0; r < NSEL; r++) {
    sel_v[r] = post[r];
    sel_i[r] = post_i[r];
    redo |= r < E && sel_i[r] == kNone;
  }
  if (__ballot(redo) != 0ull) {
    uint32_t key[1][1] = {{e < E ? order_key(v) : kTakenKey}};
    float best_v[1][NSEL];
    int best_i[1][NSEL];
    top_keys<1, 32, 1, NSEL, true>(key, e, best_v, best_i);
#pragma unroll
    for (int r = 0; r < NSEL; r++) {
      sel_v[r] = best_v[0][r];
      sel_i[r] = best_i[0][r];
    }
  }
}

// The softmax of run.cpp:336-354 over the four selected logits with the work
// spread over four lanes of the token (lane r < 4 computes exp and quotient of
// place r; the sum is formed in every lane in the order of the reference), and
// the token's ids and weights stored by those lanes.  base = the token's first
// lane in the wave.
__device__ __forceinline__ void store_topk_spread(const float (&v)[kTopK], const int (&id)[kTopK], int r,
                                                  int base, int *topk_i_row, float *topk_v_row) {
  const double mx = (double)v[0];
  const float mine = r == 0 ? v[0] : (r == 1 ? v[1] : (r == 2 ? v[2] : v[3]));
  const float ev = expf((float)((double)mine - mx));
  double sum = 0.0;
#pragma unroll
  for (int k = 0; k < kTopK; k++) sum += (double)__shfl(ev, base + k, 64);
  if (r < kTopK) {
    topk_i_row[r] = r == 0 ? id[0] : (r == 1 ? id[1] : (r == 2 ? id[2] : id[3]));
    topk_v_row[r] = (float)((double)ev / sum);
  }
}

// Bound on |first-pass logit - exact logit| of one token: the accumulation error plus the two float roundings
// (sum -> float, + bias) of either arithmetic.
struct LogitBound {
  float err0, bmax;
  __device__ __forceinline__ float up(float a) const { return a + (4.76837158e-7f * (fabsf(a) + bmax) + err0); }
  __device__ __forceinline__ float lo(float a) const { return a - (4.76837158e-7f * (fabsf(a) + bmax) + err0); }
  // whether the exact logits have the same best four in the same order
  __device__ __forceinline__ bool decides(const float (&s_v)[kTopK + 1], const int (&s_i)[kTopK + 1]) const {
    return lo(s_v[0]) > up(s_v[1]) && lo(s_v[1]) > up(s_v[2]) && lo(s_v[2]) > up(s_v[3]) &&
           (s_i[4] == kNone || lo(s_v[3]) > up(s_v[4]));
  }
  // everything not provably below the fourth best (a NaN anywhere makes the
  // comparison fail, and the expert a contender)
  __device__ __forceinline__ bool contends(float a, float fourth) const { return !(up(a) < lo(fourth)); }
};

__device__ __forceinline__ void unpack8(const uint4 v, float (&f)[8]) {
  f[0] = __uint_as_float(v.x << 16); f[1] = __uint_as_float(v.x & 0xffff0000u);
  f[2] = __uint_as_float(v.y << 16); f[3] = __uint_as_float(v.y & 0xffff0000u);
  f[4] = __uint_as_float(v.z << 16); f[5] = __uint_as_float(v.z & 0xffff0000u);
  f[6] = __uint_as_float(v.w << 16); f[7] = __uint_as_float(v.w & 0xffff0000u);
}

// One workgroup = MT * 16 tokens x all experts (NT = E_pad / 16 blocks of 16).
// Its WPC waves split the reduction dimension in chunks of 32 (wave w takes
// chunks w, w + WPC, ...); D register sets of loads run ahead of the MFMAs.
// rstat[0] = max_e |w_e| (slightly inflated), rstat[1] = max_e |b_e|.
//
// SPLIT: the first pass has run (router_logits_kernel), `first` holds its logits
// [T][E_pad], then its partial sums of squares [T][kSplitWaves].
constexpr int kSplitWaves = 4;
template <int NT, int WPC, int MT, int D, int FLUSH, bool SPLIT>
__global__ __launch_bounds__(WPC * 64) void router_kernel(
    const uint16_t *__restrict__ x, const int *__restrict__ pos, const uint16_t *__restrict__ wr,
    const float *__restrict__ br, const float *__restrict__ rstat, int T, int H, int E,
    float *__restrict__ score, int *__restrict__ topk_i, float *__restrict__ topk_v,
    const float *__restrict__ first) {
  constexpr int E_pad = NT * 16;
  constexpr int TOK = MT * 16;
  // selection: LPT lanes per token, each owning PER experts.
  // Up to 32 experts: one lane per expert, places found by counting (ranked_top), SW waves take part.
  // More: the waves take the tokens in turn, two at a time (wave_top), and then a wave's tokens have OWN lanes each.
  constexpr bool RANKED = E_pad <= 32;
  constexpr int LPT = RANKED ? 32 : 64;
  constexpr int PER = RANKED ? 1 : E_pad / LPT;
  constexpr int SW = TOK * LPT / 64;
  constexpr int TPV = RANKED ? 2 : TOK / WPC, OWN = 64 / TPV;  // tokens of a wave
  static_assert(RANKED ? SW <= WPC : TOK % WPC == 0 && TPV % 2 == 0 && OWN >= 2 * kTopK, "waves of the selection");
  constexpr int LOG_LD = RANKED ? E_pad + 4 : E_pad + 1;  // RANKED reads rows of logits in 16-byte pieces
  // cross-wave sum: GB blocks of 16 x 16 outputs at a time through 32 KB
  constexpr int NBLK = MT * NT;
  constexpr int GB = 32 / WPC < NBLK ? 32 / WPC : NBLK;
  static_assert(WPC >= 2 && NBLK % GB == 0, "groups of the cross-wave sum");
  __shared__ double part[SPLIT ? 1 : WPC / 2][GB][4][64];  // [wave][block][reg][lane]
  constexpr int SQ = SPLIT ? kSplitWaves : WPC;
  __shared__ float sumsq[SQ][TOK];
  __shared__ __attribute__((aligned(16))) float logits[TOK][LOG_LD];
  __shared__ float posted[RANKED ? TOK : 1][2 * (kTopK + 1)];  // ranked_top's lists
  __shared__ unsigned short tasks[TOK * E_pad];  // (token in tile) * E_pad + expert
  __shared__ int n_tasks;
  __shared__ float sh_br[E_pad];  // the bias, fetched while the first pass runs

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int w = tid >> 6;
  const int tok0 = blockIdx.x * TOK;
  const int row = lane & 15;  // token within a tile of 16 (first operand's row)
  const int g = lane >> 4;    // which 8 of the chunk's 32 k this lane holds
  const int kc_total = H / 32;
  if (tid == 0) n_tasks = 0;
  if (tid < E_pad) sh_br[tid] = br[tid];
  const int q = lane % OWN;  // place among the token's lanes
  auto token_of = [&](int i) { return RANKED ? w * TPV + i : w + i * WPC; };  // a wave's token i within the workgroup
  const int tr = token_of(lane / OWN), t = tok0 + tr;
  const bool active = (!RANKED || w < SW) && t < T && !(pos && pos[min(t, T - 1)] < 0);  // asked for long before it is needed
  const float wn_max = rstat[0], bmax = rstat[1];

  if constexpr (SPLIT) {
    // rows of tokens past the batch are not looked at
    for (int idx = tid; idx < TOK * E_pad / 4; idx += WPC * 64) {
      const int tt = idx / (E_pad / 4), e = idx % (E_pad / 4) * 4;
      const float4 f = *reinterpret_cast<const float4 *>(first + (size_t)min(tok0 + tt, T - 1) * E_pad + e);
      logits[tt][e] = f.x; logits[tt][e + 1] = f.y; logits[tt][e + 2] = f.z; logits[tt][e + 3] = f.w;
    }
    if (tid < TOK * SQ) sumsq[tid % SQ][tid / SQ] = first[(size_t)T * E_pad + (size_t)min(tok0 + tid / SQ, T - 1) * SQ + tid % SQ];
    __syncthreads();
  } else {
  f32x4 acc32[MT][NT], nrm[MT];
  double acc64[MT][NT][4];
#pragma unroll
  for (int m = 0; m < MT; m++) {
    nrm[m] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int n = 0; n < NT; n++) {
      acc32[m][n] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int i = 0; i < 4; i++) acc64[m][n][i] = 0.0;
    }
  }
  auto flush = [&]() {
#pragma unroll
    for (int m = 0; m < MT; m++)
#pragma unroll
      for (int n = 0; n < NT; n++) {
#pragma unroll
        for (int i = 0; i < 4; i++) acc64[m][n][i] += (double)acc32[m][n][i];
        acc32[m][n] = f32x4{0.f, 0.f, 0.f, 0.f};
      }
  };

  const uint16_t *xrow[MT];
#pragma unroll
  for (int m = 0; m < MT; m++) xrow[m] = x + (size_t)min(tok0 + 16 * m + row, T - 1) * H + g * 8;
  const uint16_t *wlane = wr + (size_t)lane * 8;
  uint4 xs[D][MT], wq[D][NT];
  auto load = [&](int d, int c) {
    const int cc = min(c, kc_total - 1);  // only the first D loads of a wave can lie past the end
#pragma unroll
    for (int m = 0; m < MT; m++) xs[d][m] = *reinterpret_cast<const uint4 *>(xrow[m] + cc * 32);
#pragma unroll
    for (int n = 0; n < NT; n++)
      wq[d][n] = *reinterpret_cast<const uint4 *>(wlane + ((size_t)n * kc_total + cc) * 512);
  };
#pragma unroll
  for (int d = 0; d < D; d++) load(d, w + d * WPC);
  int since_flush = 0;
  for (int c0 = w; c0 < kc_total; c0 += D * WPC) {
#pragma unroll
    for (int d = 0; d < D; d++) {
      const int c = c0 + d * WPC;
      if (c < kc_total) {  // the same for the whole wave
#pragma unroll
        for (int m = 0; m < MT; m++) {
          const bf16x8 xa = __builtin_bit_cast(bf16x8, xs[d][m]);
#pragma unroll
          for (int n = 0; n < NT; n++)
            acc32[m][n] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
                xa, __builtin_bit_cast(bf16x8, wq[d][n]), acc32[m][n], 0, 0, 0);
          nrm[m] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(xa, xa, nrm[m], 0, 0, 0);
        }
        if (c + D * WPC < kc_total) load(d, c + D * WPC);  // nothing is loaded that is not used
        if (FLUSH == 1 || ++since_flush == FLUSH) {
          flush();
          since_flush = 0;
        }
      }
    }
  }
  flush();

  // |x_t|^2 is the diagonal of x x^T: register i of lane l is (row 4*(l/16) + i,
  // column l % 16).
  if ((row >> 2) == g) {
#pragma unroll
    for (int m = 0; m < MT; m++) {
      const int i = row & 3;
      sumsq[w][16 * m + row] = i == 0 ? nrm[m][0] : (i == 1 ? nrm[m][1] : (i == 2 ? nrm[m][2] : nrm[m][3]));
    }
  }
  // The waves' fp64 sums are added up in a fixed order (the same sum in every
  // run): the upper half of the waves hands its sums to the lower half, whose
  // results all threads then add in wave order; GB blocks at a time.
#pragma unroll
  for (int b0 = 0; b0 < NBLK; b0 += GB) {
    if (w >= WPC / 2) {
#pragma unroll
      for (int b = 0; b < GB; b++)
#pragma unroll
        for (int i = 0; i < 4; i++) part[w - WPC / 2][b][i][lane] = acc64[(b0 + b) / NT][(b0 + b) % NT][i];
    }
    __syncthreads();
    if (w < WPC / 2) {
#pragma unroll
      for (int b = 0; b < GB; b++)
#pragma unroll
        for (int i = 0; i < 4; i++)
          part[w][b][i][lane] += acc64[(b0 + b) / NT][(b0 + b) % NT][i];
    }
    __syncthreads();
    // Register i of lane l is token 4*(l/16) + i of its tile, expert 16*n + l%16.
    for (int idx = tid; idx < GB * 256; idx += WPC * 64) {
      const int l = idx & 63;
      const int i = (idx >> 6) & 3;
      const int b = b0 + (idx >> 8);
      const int m = b / NT, n = b % NT;
      const int e = 16 * n + (l & 15);
      double sd = 0.0;
#pragma unroll
      for (int ww = 0; ww < WPC / 2; ww++) sd += part[ww][idx >> 8][i][l];
      float f = (float)sd;  // run.cpp:368
      f += sh_br[e];        // run.cpp:669-671
      logits[16 * m + 4 * (l >> 4) + i][e] = f;
    }
    __syncthreads();
  }
  }

  // Pass 2, selection.
  bool undecided = false;  // the lane's token
  auto bound = [&](int tr) {
    float ss = 0.f;
#pragma unroll
    for (int ww = 0; ww < SQ; ww++) ss += sumsq[ww][tr];
    return LogitBound{router_gamma(FLUSH) * sqrtf(ss * 1.002f) * wn_max, bmax};
  };
  auto store_inactive = [&](int t) {
    *reinterpret_cast<int4 *>(topk_i + (size_t)t * kTopK) = make_int4(-1, -1, -1, -1);
    *reinterpret_cast<float4 *>(topk_v + (size_t)t * kTopK) = make_float4(0.f, 0.f, 0.f, 0.f);
  };
  // Written out for either form: as one function of a token it cost batches of up to 64 tokens
  // 0.1 to 0.2 us where RANKED (one token, MXFP4, 24.62 / 24.75 us per call).
  if constexpr (RANKED) {
    if (w < SW) {
      const float v = q < E_pad ? logits[tr][q] : -__builtin_inff();
      float s_v[kTopK + 1];
      int s_i[kTopK + 1];
      ranked_top<E_pad, kTopK + 1>(reinterpret_cast<const float4 *>(&logits[tr][0]), v, q, E, posted[tr], s_v, s_i);
      if (active) {
        const LogitBound lb = bound(tr);
        if (lb.decides(s_v, s_i)) {
          // (tokens of one wave can differ here: the shuffles inside are among the
          // lanes of one token, which agree)
          const float sv[kTopK] = {s_v[0], s_v[1], s_v[2], s_v[3]};
          const int si[kTopK] = {s_i[0], s_i[1], s_i[2], s_i[3]};
          store_topk_spread(sv, si, q, lane - q, topk_i + (size_t)t * kTopK, topk_v + (size_t)t * kTopK);
        } else {
          undecided = true;
          if (q < E && lb.contends(v, s_v[3])) tasks[atomicAdd(&n_tasks, 1)] = (unsigned short)(tr * E_pad + q);
        }
      } else if (t < T && q == 0) {
        store_inactive(t);
      }
    }
  } else {
    float s_v[kTopK + 1] = {};  // of the lane's token
    int s_i[kTopK + 1] = {};
#pragma unroll 1
    for (int i = 0; i < TPV; i += 2) {
      float v[2][PER], two_v[2][kTopK + 1];
      int two_i[2][kTopK + 1];
#pragma unroll
      for (int n = 0; n < 2; n++)
#pragma unroll
        for (int j = 0; j < PER; j++) v[n][j] = logits[token_of(i + n)][lane * PER + j];
      wave_top<PER, 2, kTopK + 1>(v, lane, E, two_v, two_i);
#pragma unroll
      for (int n = 0; n < 2; n++)
#pragma unroll
        for (int r = 0; r <= kTopK; r++)
          if (lane / OWN == i + n) {
            s_v[r] = two_v[n][r];
            s_i[r] = two_i[n][r];
          }
    }
    if (active) {
      if (bound(tr).decides(s_v, s_i)) {
        const float sv[kTopK] = {s_v[0], s_v[1], s_v[2], s_v[3]};
        const int si[kTopK] = {s_i[0], s_i[1], s_i[2], s_i[3]};
        store_topk_spread(sv, si, q, lane - q, topk_i + (size_t)t * kTopK, topk_v + (size_t)t * kTopK);
      } else {
        undecided = true;
      }
    } else if (t < T && q == 0) {
      store_inactive(t);
    }
    for (unsigned long long left = __ballot(undecided && q == 0); left; left &= left - 1) {
      const int l = __builtin_ctzll(left), tri = token_of(l / OWN);
      const LogitBound lb = bound(tri);
      const float fourth = __uint_as_float((uint32_t)__builtin_amdgcn_readlane((int)__float_as_uint(s_v[3]), l));
#pragma unroll
      for (int j = 0; j < PER; j++) {
        const int e = lane * PER + j;
        if (e < E && lb.contends(logits[tri][e], fourth)) tasks[atomicAdd(&n_tasks, 1)] = (unsigned short)(tri * E_pad + e);
      }
    }
  }
  __syncthreads();

  // Exact logits of the contenders, one wave per (token, expert): float
  // products, fp64 sum, one rounding to float, bias added in float.  A wave
  // takes TPW tasks at a time and has all their loads in flight at once (the
  // phase is a chain of memory round trips otherwise).
  constexpr int TPW = WPC >= 8 ? 1 : 2;
  constexpr int PIECES = 6;  // 16-byte pieces per lane and operand in one round: 3072 k
  const int nt = n_tasks;
  const int n_pieces = H / 8;
  for (int task0 = w * TPW; task0 < nt; task0 += WPC * TPW) {
    double s[TPW];
    const uint16_t *xr[TPW], *we[TPW];
    int tt[TPW], ee[TPW];
#pragma unroll
    for (int j = 0; j < TPW; j++) {
      const int code = tasks[min(task0 + j, nt - 1)];
      tt[j] = code / E_pad;
      ee[j] = code % E_pad;
      xr[j] = x + (size_t)min(tok0 + tt[j], T - 1) * H;
      we[j] = wr + ((size_t)(ee[j] >> 4) * kc_total * 64 + (ee[j] & 15)) * 8;
      s[j] = 0.0;
    }
    for (int p0 = 0; p0 < n_pieces; p0 += 64 * PIECES) {
      uint4 xv[TPW][PIECES], wv[TPW][PIECES];
#pragma unroll
      for (int j = 0; j < TPW; j++)
#pragma unroll
        for (int i = 0; i < PIECES; i++) {
          // piece p: k = 8p .. 8p+7 = chunk p/4, quarter p%4; past the row's end: piece 0, not used
          const int pp = p0 + i * 64 + lane;
          const int p = pp < n_pieces ? pp : 0;
          xv[j][i] = *reinterpret_cast<const uint4 *>(xr[j] + p * 8);
          wv[j][i] = *reinterpret_cast<const uint4 *>(we[j] + ((size_t)(p >> 2) * 64 + (p & 3) * 16) * 8);
        }
#pragma unroll
      for (int j = 0; j < TPW; j++)
#pragma unroll
        for (int i = 0; i < PIECES; i++) {
          if (p0 + i * 64 + lane < n_pieces) {
            float xf[8], wf[8];
            unpack8(xv[j][i], xf);
            unpack8(wv[j][i], wf);
#pragma unroll
            for (int k = 0; k < 8; k++) s[j] += (double)(xf[k] * wf[k]);
          }
        }
    }
#pragma unroll
    for (int j = 0; j < TPW; j++) {
#pragma unroll
      for (int off = 32; off > 0; off >>= 1) s[j] += __shfl_xor(s[j], off, 64);
      if (lane == 0 && task0 + j < nt) {
        float f = (float)s[j];
        f += sh_br[ee[j]];
        logits[tt[j]][ee[j]] = f;
      }
    }
  }
  __syncthreads();

  if constexpr (RANKED) {
    if (w < SW && __ballot(undecided) != 0ull) {  // per wave: ranked_top is a wave's work
      const float v = q < E_pad ? logits[tr][q] : -__builtin_inff();
      float s_v[kTopK];
      int s_i[kTopK];
      ranked_top<E_pad, kTopK>(reinterpret_cast<const float4 *>(&logits[tr][0]), v, q, E, posted[tr], s_v, s_i);
      if (undecided) store_topk_spread(s_v, s_i, q, lane - q, topk_i + (size_t)t * kTopK, topk_v + (size_t)t * kTopK);
    }
  } else {
    for (unsigned long long left = __ballot(undecided && q == 0); left; left &= left - 1) {
      const int tri = token_of(__builtin_ctzll(left) / OWN);
      float v[1][PER], s_v[1][kTopK];
      int s_i[1][kTopK];
#pragma unroll
      for (int j = 0; j < PER; j++) v[0][j] = logits[tri][lane * PER + j];
      wave_top<PER, 1, kTopK>(v, lane, E, s_v, s_i);
      store_topk_spread(s_v[0], s_i[0], lane, 0, topk_i + (size_t)(tok0 + tri) * kTopK, topk_v + (size_t)(tok0 + tri) * kTopK);
    }
  }
  if (score) {
    for (int idx = tid; idx < TOK * E_pad; idx += WPC * 64) {
      const int tt = idx / E_pad, e = idx % E_pad;
      const int ts = tok0 + tt;
      if (e < E && ts < T && !(pos && pos[ts] < 0)) score[(size_t)ts * E + e] = logits[tt][e];
    }
  }
}

// The first pass of router_kernel<., 4, 1, ., 1> with a workgroup per 16 tokens and BLOCK of 16
// experts: with all 128 or 256 experts to a workgroup one CU takes in the whole router
// matrix (0.74 MB at 128 experts and 2880 columns, 12 us and more), and a small batch has few
// of them.  The same chunks to the same four waves and the same order of the sums: the same
// bits.  Written to `first` (see SPLIT), which a second launch reads.  us at 128 experts and
// 2880 columns, one kernel / both launches, with the selection by eight lanes per token: 6 tokens 16.7 / 5.0
// + 6.3, 200 tokens 32.5 / 7.7 + 17.2; with wave_top the second launch takes 4.3 and, by the tokens
// that take the second pass, 9 to 13.
template <int D>
__global__ __launch_bounds__(kSplitWaves * 64) void router_logits_kernel(
    const uint16_t *__restrict__ x, const uint16_t *__restrict__ wr, const float *__restrict__ br, int T, int H,
    int E_pad, float *__restrict__ first) {
  __shared__ double part[kSplitWaves / 2][4][64];
  const int tid = threadIdx.x;
  const int lane = tid & 63, w = tid >> 6;
  const int row = lane & 15, g = lane >> 4;
  const int tok0 = blockIdx.x * 16, n = blockIdx.y;
  const int kc_total = H / 32;
  const float bias = br[16 * n + row];
  const uint16_t *xrow = x + (size_t)min(tok0 + row, T - 1) * H + g * 8;
  const uint16_t *wlane = wr + ((size_t)n * kc_total * 64 + lane) * 8;
  f32x4 nrm = {0.f, 0.f, 0.f, 0.f};
  double acc64[4] = {0.0, 0.0, 0.0, 0.0};
  uint4 xs[D], wq[D];
  auto load = [&](int d, int c) {
    const int cc = min(c, kc_total - 1);  // only the first D loads of a wave can lie past the end
    xs[d] = *reinterpret_cast<const uint4 *>(xrow + cc * 32);
    wq[d] = *reinterpret_cast<const uint4 *>(wlane + (size_t)cc * 512);
  };
#pragma unroll
  for (int d = 0; d < D; d++) load(d, w + d * kSplitWaves);
  for (int c0 = w; c0 < kc_total; c0 += D * kSplitWaves) {
#pragma unroll
    for (int d = 0; d < D; d++) {
      const int c = c0 + d * kSplitWaves;
      if (c < kc_total) {  // the same for the whole wave
        const bf16x8 xa = __builtin_bit_cast(bf16x8, xs[d]);
        const f32x4 zero = {0.f, 0.f, 0.f, 0.f};
        const f32x4 p = __builtin_amdgcn_mfma_f32_16x16x32_bf16(xa, __builtin_bit_cast(bf16x8, wq[d]), zero, 0, 0, 0);
        nrm = __builtin_amdgcn_mfma_f32_16x16x32_bf16(xa, xa, nrm, 0, 0, 0);
        if (c + D * kSplitWaves < kc_total) load(d, c + D * kSplitWaves);
#pragma unroll
        for (int i = 0; i < 4; i++) acc64[i] += (double)p[i];
      }
    }
  }
  if (n == 0 && (row >> 2) == g && tok0 + row < T) {
    const int i = row & 3;
    first[(size_t)T * E_pad + (size_t)(tok0 + row) * kSplitWaves + w] =
        i == 0 ? nrm[0] : (i == 1 ? nrm[1] : (i == 2 ? nrm[2] : nrm[3]));
  }
  if (w >= kSplitWaves / 2) {
#pragma unroll
    for (int i = 0; i < 4; i++) part[w - kSplitWaves / 2][i][lane] = acc64[i];
  }
  __syncthreads();
  if (w < kSplitWaves / 2) {
#pragma unroll
    for (int i = 0; i < 4; i++) part[w][i][lane] += acc64[i];
  }
  __syncthreads();
  // thread -> register w of lane l: token 4 * (l / 16) + w, expert 16 n + l % 16
  double sd = 0.0;
#pragma unroll
  for (int ww = 0; ww < kSplitWaves / 2; ww++) sd += part[ww][w][lane];
  float f = (float)sd;  // run.cpp:368
  f += bias;            // run.cpp:669-671
  const int t = tok0 + 4 * g + w;
  if (t < T) first[(size_t)t * E_pad + 16 * n + row] = f;
}

// Statistics of a layer's router for the error bound of the first pass:
// rstat[0] = max_e |w_e|_2 over the bf16-rounded weights (inflated by 1e-3 for
// the rounding of this very sum), rstat[1] = max_e |b_e|.  One workgroup.
__global__ __launch_bounds__(256) void router_stats_kernel(const float *__restrict__ w,
                                                           const float *__restrict__ b, int E, int H,
                                                           float *__restrict__ rstat) {
  __shared__ float red[256];
  float wmax = 0.f, bmax = 0.f;
  for (int e = 0; e < E; e++) {
    float s = 0.f;
    for (int k = threadIdx.x; k < H; k += 256) {
      const float v = __uint_as_float((uint32_t)f32_to_bf16_rne(w[(size_t)e * H + k]) << 16);
      s += v * v;
    }
    red[threadIdx.x] = s;
    __syncthreads();
    for (int off = 128; off > 0; off >>= 1) {
      if ((int)threadIdx.x < off) red[threadIdx.x] += red[threadIdx.x + off];
      __syncthreads();
    }
    wmax = fmaxf(wmax, red[0]);
    __syncthreads();
    bmax = fmaxf(bmax, fabsf(__uint_as_float((uint32_t)f32_to_bf16_rne(b[e]) << 16)));
  }
  if (threadIdx.x == 0) {
    rstat[0] = sqrtf(wmax) * 1.001f;
    rstat[1] = bmax;
  }
}

hipError_t launch_router_stats(const float *w_src, const float *b_src, int E, int H, float *rstat,
                               hipStream_t s) {
  router_stats_kernel<<<1, 256, 0, s>>>(w_src, b_src, E, H, rstat);
  return hipGetLastError();
}

template <int NT>
static hipError_t launch_router_nt(const uint16_t *x, const int *pos, const uint16_t *wr,
                                   const float *br, const float *rstat, int T, int H, int E,
                                   float *score, int *topk_i, float *topk_v, float *first, hipStream_t s) {
  // As fine a split of the reduction as the registers allow: more waves keep
  // more loads in flight, and small batches still occupy the SIMDs.  D register
  // sets of 4 * (MT + NT) registers each run ahead.
  constexpr int WPC = NT <= 2 ? 16 : (NT <= 4 ? 8 : 4);
  constexpr int D = NT <= 2 ? 6 : (NT <= 4 ? 4 : (NT <= 8 ? 3 : 2));
  // MFMAs between two hand-overs to fp64: the fewer, the tighter the bound and
  // the fewer tokens take the second pass, at 8 * NT more fp64 instructions
  // each; the first pass is bound by its loads, so the hand-over after every
  // MFMA costs nothing
  constexpr int FLUSH = 1;
  // Every workgroup streams the whole router matrix through its CU; at 128
  // experts a workgroup takes two tiles of 16 tokens so that half as many do
  // (at 256 the accumulators of two tiles no longer fit the registers).
  if constexpr (NT >= 8) {
    static_assert(WPC == kSplitWaves, "router_logits_kernel adds up what router_kernel does, in its order");
    if (first && T <= split_router_tokens(NT * 16, H)) {
      router_logits_kernel<8><<<dim3((T + 15) / 16, NT), kSplitWaves * 64, 0, s>>>(x, wr, br, T, H, NT * 16, first);
      router_kernel<NT, 8, 1, 1, FLUSH, true><<<(T + 15) / 16, 8 * 64, 0, s>>>(x, pos, wr, br, rstat, T, H, E, score,
                                                                              topk_i, topk_v, first);
      return hipGetLastError();
    }
  }
  if (NT == 8 && T > 256 * 16) {
    constexpr int MT = NT == 8 ? 2 : 1;
    router_kernel<NT, WPC, MT, D, FLUSH, false><<<(T + 16 * MT - 1) / (16 * MT), WPC * 64, 0, s>>>(
        x, pos, wr, br, rstat, T, H, E, score, topk_i, topk_v, nullptr);
  } else {
    router_kernel<NT, WPC, 1, D, FLUSH, false><<<(T + 15) / 16, WPC * 64, 0, s>>>(x, pos, wr, br, rstat, T, H, E,
                                                                                 score, topk_i, topk_v, nullptr);
  }
  return hipGetLastError();
}

hipError_t launch_router(const uint16_t *x, const int *pos, const uint16_t *wr, const float *br,
                         const float *rstat, int T, int H, int E, int E_pad, float *score, int *topk_i,
                         float *topk_v, float *first, hipStream_t s) {
  if (T <= 0) return hipSuccess;
  switch (E_pad / 16) {
    case 1: return launch_router_nt<1>(x, pos, wr, br, rstat, T, H, E, score, topk_i, topk_v, first, s);
    case 2: return launch_router_nt<2>(x, pos, wr, br, rstat, T, H, E, score, topk_i, topk_v, first, s);
    case 4: return launch_router_nt<4>(x, pos, wr, br, rstat, T, H, E, score, topk_i, topk_v, first, s);
    case 8: return launch_router_nt<8>(x, pos, wr, br, rstat, T, H, E, score, topk_i, topk_v, first, s);
    case 16: return launch_router_nt<16>(x, pos, wr, br, rstat, T, H, E, score, topk_i, topk_v, first, s);
    default: return hipErrorInvalidValue;
  }
}

}  // namespace moe

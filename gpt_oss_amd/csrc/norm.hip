// RMS normalisation in front of the layer.  Replaces rmsnorm_batch_kernel
// (utility/utility.cpp:194-271; call getp_run.cpp:688-695) with the arithmetic of
// the CPU path (run.cpp:321-334): squares are exact in fp32 for bf16 inputs and
// are summed in fp64, the scale 1/sqrt(mean + 1e-5) is formed in fp32 with
// correctly rounded sqrt and division, the product weight * (scale * x) is
// rounded once to fp32 and then to bf16, the layer's input type.  The one
// difference from a sequential sum is the order of the fp64 additions, which
// reaches the fp32 scale only where two fp64 sums that differ in their last bit
// straddle an fp32 rounding boundary.
#include "moe_internal.h"

namespace moe {

// THREADS per token, 8 elements (16 bytes) per thread and pass: a workgroup, or a wave for rows short
// enough for its registers.  Bound by latency: row and weight are asked for at once and the
// row stays in registers (up to 16 elements per thread; longer ones read the rest again).  At 2880
// columns a wave per token, which walked the row twice, took 7.8 us for 6 tokens, 9.3 for 200, 16.0 for 4096; a
// workgroup 4.5, 5.4 and 15.0.  With short rows a workgroup is mostly idle threads: a call of
// moe_block_forward with 7168 tokens took 51 us instead of 47 at 64 columns, 69 instead of 64 at 256, 107
// instead of 101 at 512.
template <int THREADS>
__global__ __launch_bounds__(256) void rmsnorm_kernel(const uint16_t *__restrict__ x,
                                                     const float *__restrict__ weight,
                                                     const int *__restrict__ pos,
                                                     uint16_t *__restrict__ t_out, int T, int H) {
  constexpr int HELD = kNormHeld;
  static_assert(THREADS == 64 || THREADS == 256, "a wave or a workgroup");
  const int tid = threadIdx.x % THREADS;
  const int t = blockIdx.x * (256 / THREADS) + threadIdx.x / THREADS;
  if (t >= T) return;             // (waves of a short last workgroup)
  if (pos && pos[t] < 0) return;  // the row takes part in nothing downstream
  const uint4 *row = reinterpret_cast<const uint4 *>(x + (size_t)t * H);
  const int chunks = H / 8;
  uint4 held[HELD];
  float4 w0[HELD], w1[HELD];
#pragma unroll
  for (int i = 0; i < HELD; i++) {
    const int c = tid + THREADS * i;
    held[i] = make_uint4(0u, 0u, 0u, 0u);
    if (c < chunks) {
      held[i] = row[c];
      w0[i] = *reinterpret_cast<const float4 *>(weight + 8 * c);
      w1[i] = *reinterpret_cast<const float4 *>(weight + 8 * c + 4);
    }
  }
  double ss = 0.0;
  auto add = [&](const uint4 v) {
    const uint32_t u[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
    for (int i = 0; i < 4; i++) {
      const float a = __uint_as_float(u[i] << 16), b = __uint_as_float(u[i] & 0xffff0000u);
      ss += (double)(a * a);
      ss += (double)(b * b);
    }
  };
#pragma unroll
  for (int i = 0; i < HELD; i++) add(held[i]);
  for (int c = tid + THREADS * HELD; c < chunks; c += THREADS) add(row[c]);
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) ss += __shfl_xor(ss, off, 64);
  if constexpr (THREADS > 64) {
    __shared__ double sh_ss[THREADS / 64];
    if ((tid & 63) == 0) sh_ss[tid >> 6] = ss;
    __syncthreads();
    ss = ((sh_ss[0] + sh_ss[1]) + sh_ss[2]) + sh_ss[3];
  }
  ss /= (double)H;
  ss += (double)1e-5f;
  const float narrowed = (float)ss;
  const float root = (float)sqrt((double)narrowed);  // = sqrtf, correctly rounded
  const float scale = (float)(1.0 / (double)root);    // = 1.0f / root, correctly rounded
  uint4 *out = reinterpret_cast<uint4 *>(t_out + (size_t)t * H);
  auto put = [&](int c, const uint4 v, const float4 a4, const float4 b4) {
    const float w[8] = {a4.x, a4.y, a4.z, a4.w, b4.x, b4.y, b4.z, b4.w};
    const uint32_t u[4] = {v.x, v.y, v.z, v.w};
    uint32_t o[4];
#pragma unroll
    for (int i = 0; i < 4; i++) {
      const float a = __uint_as_float(u[i] << 16), b = __uint_as_float(u[i] & 0xffff0000u);
      const float ra = (float)((double)w[2 * i] * ((double)scale * (double)a));
      const float rb = (float)((double)w[2 * i + 1] * ((double)scale * (double)b));
      o[i] = f32_to_bf16_rne(ra) | ((uint32_t)f32_to_bf16_rne(rb) << 16);
    }
    out[c] = make_uint4(o[0], o[1], o[2], o[3]);
  };
#pragma unroll
  for (int i = 0; i < HELD; i++)
    if (tid + THREADS * i < chunks) put(tid + THREADS * i, held[i], w0[i], w1[i]);
  for (int c = tid + THREADS * HELD; c < chunks; c += THREADS)
    put(c, row[c], *reinterpret_cast<const float4 *>(weight + 8 * c), *reinterpret_cast<const float4 *>(weight + 8 * c + 4));
}

// Rows of H bf16 values copied into rows of Hp >= H, the rest zero: the grouped
// GEMMs reduce over multiples of 64, and a hidden size that is not one (the
// reference's 7M model has 32, export_model_bin/gpt-oss-7m/config.json:3) is
// widened here, once per call, rather than read past the end of its rows.
__global__ __launch_bounds__(256) void pad_rows_kernel(const uint4 *__restrict__ x, uint4 *__restrict__ xp,
                                                      int T, int H8, int Hp8) {
  const size_t n = (size_t)T * Hp8;
  for (size_t i = (size_t)blockIdx.x * 256 + threadIdx.x; i < n; i += (size_t)gridDim.x * 256) {
    const size_t t = i / Hp8;
    const int c = (int)(i % Hp8);
    xp[i] = c < H8 ? x[t * H8 + c] : make_uint4(0u, 0u, 0u, 0u);
  }
}

hipError_t launch_pad_rows(const uint16_t *x, uint16_t *xp, int T, int H, int Hp, hipStream_t s) {
  const size_t n = (size_t)T * (Hp / 8);
  const int grid = (int)((n + 255) / 256 < 4096 ? (n + 255) / 256 : 4096);
  pad_rows_kernel<<<grid, 256, 0, s>>>(reinterpret_cast<const uint4 *>(x), reinterpret_cast<uint4 *>(xp), T,
                                       H / 8, Hp / 8);
  return hipGetLastError();
}

hipError_t launch_rmsnorm(const uint16_t *x, const float *weight, const int *pos, uint16_t *t_out,
                          int T, int H, hipStream_t s) {
  if (norm_wave_per_token(T, H))
    rmsnorm_kernel<64><<<(T + 3) / 4, 256, 0, s>>>(x, weight, pos, t_out, T, H);
  else
    rmsnorm_kernel<256><<<T, 256, 0, s>>>(x, weight, pos, t_out, T, H);
  return hipGetLastError();
}

}  // namespace moe

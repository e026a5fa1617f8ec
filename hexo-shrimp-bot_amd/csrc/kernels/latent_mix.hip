// Latent self-mix for gfx950: the four latent rows of each position attend
// to each other (model.py:516-526), in fp32 like the reference's mix:
//   z    = LN(g_p)                          (4 x 128; affine folded into W)
//   q|k|v = z Wqkv + bqkv                   (4 x 384)
//   a_h  = softmax(q_h k_h^T / sqrt(32)) v_h  for each of the 4 heads of 32
//   g_p += a Wo + bo
// One workgroup of 1,024 threads per position.  The work is tiny (0.5 MFLOP
// per position); what bounds it is fetching the weights (256 KB in fp32,
// transposed so the threads read consecutive columns).  Every thread requests
// all of its weights (80 values: a column's half of q|k|v, an eighth of an
// output column) before its first row, so a launch waits for them once, and
// keeps them across its positions.  With 256 threads reading 32 values at a
// time it was five round trips one after the other: 13.8 us for one position
// (now 7.9), 20 for 512 (17.9).
#include "common.hpp"

namespace mantis {
namespace {

constexpr int kH = 128;
constexpr int kSlots = 4;
constexpr int kThreads = 1024;
constexpr int kParts = 8;  // cuts of the output projection's sums

__global__ void __launch_bounds__(kThreads)
latent_mix_kernel(float* __restrict__ g, int64_t ldg, int64_t n_pos, const float* __restrict__ wqkv_t,
                  const float* __restrict__ bqkv, const float* __restrict__ wo_t, const float* __restrict__ bo,
                  float scale) {
  __shared__ __attribute__((aligned(16))) float z[kSlots][kH];
  __shared__ float part[kParts * kSlots * kH];  // q|k|v: [2][4][384], then the output: [8][4][128]
  __shared__ float qkv[kSlots][3 * kH];
  __shared__ float prob[4][kSlots][kSlots];  // [head][query][key]
  __shared__ __attribute__((aligned(16))) float mixed[kSlots][kH];
  static_assert(kParts * kSlots * kH >= 2 * kSlots * 3 * kH, "the partial products share one array");
  const int t = threadIdx.x, wave = t / 64, lane = t % 64;
  // this thread's weights: column c1 of q|k|v over half the rows (the first
  // 768 threads), column c2 of the output over an eighth
  const int c1 = t % (3 * kH), half = t / (3 * kH), c2 = t % kH, oct = t / kH;
  float w1[kH / 2], w2[kH / kParts];
#pragma unroll
  for (int k = 0; k < kH / 2; ++k) w1[k] = half < 2 ? wqkv_t[(half * (kH / 2) + k) * 3 * kH + c1] : 0.f;
#pragma unroll
  for (int k = 0; k < kH / kParts; ++k) w2[k] = wo_t[(oct * (kH / kParts) + k) * kH + c2];
  for (int64_t p = blockIdx.x; p < n_pos; p += gridDim.x) {
    float* rows = g + p * kSlots * ldg;
    // LayerNorm: wave w normalises row w, two features per lane
    if (wave < kSlots) {
      const float x0 = rows[wave * ldg + lane], x1 = rows[wave * ldg + lane + 64];
      float s = x0 + x1;
#pragma unroll
      for (int o = 32; o > 0; o >>= 1) s += __shfl_xor(s, o);
      const float mean = s * (1.f / kH);
      const float d0 = x0 - mean, d1 = x1 - mean;
      float q = d0 * d0 + d1 * d1;
#pragma unroll
      for (int o = 32; o > 0; o >>= 1) q += __shfl_xor(q, o);
      const float rstd = rsqrtf(q * (1.f / kH) + 1e-5f);
      z[wave][lane] = d0 * rstd;
      z[wave][lane + 64] = d1 * rstd;
    }
    __syncthreads();
    // q | k | v: column c1 of the four rows, over this thread's half of the sum
    if (half < 2) {
      float acc[kSlots] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int k = 0; k < kH / 2; k += 4)
#pragma unroll
        for (int r = 0; r < kSlots; ++r) {
          const float4 x = *reinterpret_cast<const float4*>(&z[r][half * (kH / 2) + k]);
          acc[r] = fmaf(x.w, w1[k + 3], fmaf(x.z, w1[k + 2], fmaf(x.y, w1[k + 1], fmaf(x.x, w1[k], acc[r]))));
        }
#pragma unroll
      for (int r = 0; r < kSlots; ++r) part[(half * kSlots + r) * 3 * kH + c1] = acc[r];
    }
    __syncthreads();
    for (int i = t; i < kSlots * 3 * kH; i += kThreads)
      qkv[i / (3 * kH)][i % (3 * kH)] = part[i] + part[kSlots * 3 * kH + i] + bqkv[i % (3 * kH)];
    __syncthreads();
    // scores and softmax over the four keys: thread (head, query, key)
    if (t < 64) {
      const int h = t / 16, i = (t / 4) % 4, j = t % 4;
      float s = 0.f;
#pragma unroll 8
      for (int d = 0; d < 32; ++d) s = fmaf(qkv[i][32 * h + d], qkv[j][kH + 32 * h + d], s);
      s *= scale;
      float m = fmaxf(s, __shfl_xor(s, 1));
      m = fmaxf(m, __shfl_xor(m, 2));
      const float e = __expf(s - m);
      float l = e + __shfl_xor(e, 1);
      l += __shfl_xor(l, 2);
      prob[h][i][j] = e / l;
    }
    __syncthreads();
    // mixed[i][32 h + d] = sum_j prob[h][i][j] v[j][32 h + d]
    if (t < kSlots * kH) {
      const int i = t / kH, c = t % kH, h = c / 32;
      float a = 0.f;
#pragma unroll
      for (int j = 0; j < kSlots; ++j) a = fmaf(prob[h][i][j], qkv[j][2 * kH + c], a);
      mixed[i][c] = a;
    }
    __syncthreads();
    // output projection: column c2 of the four rows, over an eighth of the sum
    {
      float acc[kSlots] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int k = 0; k < kH / kParts; k += 4)
#pragma unroll
        for (int r = 0; r < kSlots; ++r) {
          const float4 x = *reinterpret_cast<const float4*>(&mixed[r][oct * (kH / kParts) + k]);
          acc[r] = fmaf(x.w, w2[k + 3], fmaf(x.z, w2[k + 2], fmaf(x.y, w2[k + 1], fmaf(x.x, w2[k], acc[r]))));
        }
#pragma unroll
      for (int r = 0; r < kSlots; ++r) part[(oct * kSlots + r) * kH + c2] = acc[r];
    }
    __syncthreads();
    if (t < kSlots * kH) {
      const int r = t / kH;
      float a = bo[c2];
#pragma unroll
      for (int k = 0; k < kParts; ++k) a += part[(k * kSlots + r) * kH + c2];
      rows[r * ldg + c2] += a;
    }
    __syncthreads();  // z, part and qkv are rewritten by the next position
  }
}

}  // namespace
}  // namespace mantis

using namespace mantis;

extern "C" int32_t mantis_latent_mix(float* g, int64_t ldg, int64_t n_pos, const float* wqkv_t, const float* bqkv,
                                     const float* wo_t, const float* bo, void* stream) {
  if (n_pos == 0) return MANTIS_OK;
  if (!g || !wqkv_t || !bqkv || !wo_t || !bo || n_pos < 0 || ldg < kH) return MANTIS_E_ARG;
  int dev = 0, cus = 0;
  if (hipGetDevice(&dev) != hipSuccess || hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) !=
                                              hipSuccess || cus <= 0)
    cus = 256;
  const int64_t grid = n_pos < 4 * int64_t(cus) ? n_pos : 4 * int64_t(cus);
  latent_mix_kernel<<<dim3(unsigned(grid)), dim3(kThreads), 0, as_stream(stream)>>>(
      g, ldg, n_pos, wqkv_t, bqkv, wo_t, bo, 0.17677669529663687f);
  return launched();
}

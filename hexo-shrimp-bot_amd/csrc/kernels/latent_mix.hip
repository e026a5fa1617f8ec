// Latent self-mix for gfx950: the four latent rows of each position attend
// to each other (model.py:516-526), in fp32 like the reference's mix:
//   z    = LN(g_p)                          (4 x 128; affine folded into W)
//   q|k|v = z Wqkv + bqkv                   (4 x 384)
//   a_h  = softmax(q_h k_h^T / sqrt(32)) v_h  for each of the 4 heads of 32
//   g_p += a Wo + bo
// One workgroup of 512 threads per position, at most one per CU.  The work is
// tiny (0.5 MFLOP per position); what bounds a launch is fetching the weights
// (256 KB in fp32, transposed so the threads read consecutive columns) and the
// chain of steps.  A thread requests all of its weights (one column of q|k|v
// or of the output, 128 values) at once and keeps them across its positions.
// Each projection is one fp32 FMA chain over k: the latents' last bits reach
// every later 16-bit state, and sums cut into parts moved whole evaluations by
// 9e-4.  The chains run on 4 x 4 x 1 fp32 MFMAs, half the issue time of vector
// FMAs and a quarter of their LDS reads.  Per launch, weights in L2: 5.9 us for
// one position, 11.6 for 512, 31 for 2,000 (chains of vector FMAs: 12.6, 27, 92;
// 256 threads reading 32 weights at a time: 9.6, 13.4, 34; sums in 2 and 8
// parts over 1,024 threads: 7.2, 16.8, 48).
#include "common.hpp"
#include "mfma.hpp"

namespace mantis {
namespace {

constexpr int kH = 128;
constexpr int kSlots = 4;
constexpr int kRowPitch = kH + 4;       // (the four rows' reads meet different banks)
constexpr int kQkv = 3 * kH;            // threads [0, 384): a column of q|k|v each
constexpr int kThreads = kQkv + kH;     // threads [384, 512): a column of the output each

// The four rows' products with the wavefront's 64 weight columns (w: this
// lane's), each one fp32 FMA chain over k in order: one 4 x 4 x 1 MFMA of 16
// blocks per k (rows x this lane's quad of columns; lane 4 b + i brings row
// i's value to block b, and holds its column's four sums).
__device__ __forceinline__ f32x4_t column(const float (&x)[kSlots][kRowPitch], const float (&w)[kH], int lane) {
  const float* mine = x[lane % 4];
  f32x4_t acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int k = 0; k < kH; k += 4) {
    const float4 v = *reinterpret_cast<const float4*>(mine + k);
    acc = __builtin_amdgcn_mfma_f32_4x4x1f32(v.x, w[k], acc, 0, 0, 0);
    acc = __builtin_amdgcn_mfma_f32_4x4x1f32(v.y, w[k + 1], acc, 0, 0, 0);
    acc = __builtin_amdgcn_mfma_f32_4x4x1f32(v.z, w[k + 2], acc, 0, 0, 0);
    acc = __builtin_amdgcn_mfma_f32_4x4x1f32(v.w, w[k + 3], acc, 0, 0, 0);
  }
  return acc;
}

__global__ void __launch_bounds__(kThreads)
latent_mix_kernel(float* __restrict__ g, int64_t ldg, int64_t n_pos, const float* __restrict__ wqkv_t,
                  const float* __restrict__ bqkv, const float* __restrict__ wo_t, const float* __restrict__ bo,
                  float scale) {
  __shared__ __attribute__((aligned(16))) float z[kSlots][kRowPitch];
  __shared__ float qkv[kSlots][kQkv];
  __shared__ float prob[4][kSlots][kSlots];  // [head][query][key]
  __shared__ __attribute__((aligned(16))) float mixed[kSlots][kRowPitch];
  const int t = threadIdx.x, wave = t / 64, lane = t % 64;
  // LayerNorm: wave w < 4 normalises row w, two features per lane.  A row is
  // requested before the weights and, from then on, a position ahead (loads
  // return in order: behind the weights it would wait for all of them)
  float x0 = 0.f, x1 = 0.f;
  auto request = [&](int64_t p) {
    if (wave >= kSlots || p >= n_pos) return;
    const float* row = g + (p * kSlots + wave) * ldg;
    x0 = row[lane], x1 = row[lane + 64];
  };
  request(blockIdx.x);
  // this thread's weight column (a wavefront is all of one kind)
  const bool first = t < kQkv;
  const int col = first ? t : t - kQkv, ldw = first ? kQkv : kH;
  const float* from = (first ? wqkv_t : wo_t) + col;
  float w[kH];
#pragma unroll
  for (int k = 0; k < kH; ++k) w[k] = from[k * ldw];
  const float b = first ? bqkv[col] : bo[col];
  for (int64_t p = blockIdx.x; p < n_pos; p += gridDim.x) {
    float* rows = g + p * kSlots * ldg;
    if (wave < kSlots) {
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
      request(p + gridDim.x);
    }
    __syncthreads();
    if (first) {
      const f32x4_t acc = column(z, w, lane);
#pragma unroll
      for (int r = 0; r < kSlots; ++r) qkv[r][col] = acc[r] + b;
    }
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
    {
      const int i = t / kH, c = t % kH, h = c / 32;
      float a = 0.f;
#pragma unroll
      for (int j = 0; j < kSlots; ++j) a = fmaf(prob[h][i][j], qkv[j][2 * kH + c], a);
      mixed[i][c] = a;
    }
    __syncthreads();
    if (!first) {
      const f32x4_t acc = column(mixed, w, lane);
#pragma unroll
      for (int r = 0; r < kSlots; ++r) rows[r * ldg + col] += acc[r] + b;
    }
    __syncthreads();  // z, qkv and the rows' next readers
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
  const int64_t grid = n_pos < cus ? n_pos : cus;  // one workgroup's weights fill a CU's registers
  latent_mix_kernel<<<dim3(unsigned(grid)), dim3(kThreads), 0, as_stream(stream)>>>(
      g, ldg, n_pos, wqkv_t, bqkv, wo_t, bo, 0.17677669529663687f);
  return launched();
}

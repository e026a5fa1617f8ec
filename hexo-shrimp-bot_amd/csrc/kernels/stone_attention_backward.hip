// Backward of the ragged attention on 16-bit MFMA for gfx950 (the reference's
// flash backward, attention.py:166-560, with its row statistic
// delta = sum(out * grad_out)).  With a_ij = exp(scale q_i . k_j - lse_i) over
// the live keys j < L of the live rows i < L, dp_ij = go_i . v_j and
// ds_ij = a_ij (dp_ij - delta_i):
//   dq_i = scale sum_j ds_ij k_j,  dk_j = scale sum_i ds_ij q_i,  dv_j = sum_i a_ij go_i.
//
// Two passes, each a workgroup per (position, head, 64 rows), 16 rows per
// wavefront, the other side's rows in 64-row chunks through LDS, as they are
// and transposed, the next chunk's in registers meanwhile:
//   query-major  S^T = K Q^T and dP^T = V dO^T, then dQ^T += K^T dS^T
//   key-major    S = Q K^T and dP = dO V^T, then dV^T += dO^T P, dK^T += Q^T dS
// Both keep a lane on one row of its own side, so a score fragment's value of
// row 16 tt + 4 g + t is the next product's B operand as it stands (the four
// K slots of a step are the rows 4 g + t of the lane groups g).
//
// Precision: scores and dp are exact products of 16-bit rows summed in fp32
// (16-bit MFMA); the probabilities and ds are fp32 and enter their products,
// with the rows widened, as fp32 MFMA operands.  Every sum is fp32 in a fixed
// order: two calls agree bitwise.  Rows and keys at or past L get zero
// gradients, whatever the live rows hold.
//
// Bound by the latency of a wavefront's own chain per chunk (rows, barrier,
// products, exponentials, then 32 or 64 dependent fp32 MFMAs) with two
// wavefronts per SIMD: MFMA 12-18% busy, VALU 17-18%, half of the wavefronts'
// time waiting.  192 positions of 44-124 rows, 4 heads of 32, bf16: one row per
// lane with fp32 FMAs took 74 and 152 us, these passes take 21 and 26; 16
// positions of 512-1,024 rows 390 and 611, now 64 and 105.  (Operands cut to
// bf16 pairs of 16 significant bits: 15 and 17, 40 and 55, but sums that cancel
// lose those bits and an infinite row turned zeros into NaNs.)
#include "common.hpp"
#include "mfma.hpp"

namespace mantis {
namespace {

constexpr int kTile = 64;                // rows of a workgroup, and of a chunk
constexpr int kTPitch = kTile + 8;       // 16-bit elements per transposed row
constexpr float kLog2e = 1.4426950408889634f;

struct Rows {  // one (P, A, T, HD) operand: base and element strides
  const uint16_t* p;
  int64_t sp, sa, st;
  __device__ const uint16_t* at(int64_t pos, int64_t a) const { return p + pos * sp + a * sa; }
};
struct RowsOut {
  uint16_t* p;
  int64_t sp, sa, st;
  __device__ uint16_t* row(int64_t pos, int64_t a, int64_t t) const { return p + pos * sp + a * sa + t * st; }
};

template <bool kHalf>
__device__ __forceinline__ float widen(uint32_t bits) {
  if constexpr (kHalf) return float(__builtin_bit_cast(_Float16, uint16_t(bits)));
  else return __uint_as_float(bits << 16);
}

template <bool kHalf, int HD>
struct Geom {
  static constexpr int kPitch = HD + 8;                 // 16-bit elements per staged row
  static constexpr int kKs = HD < 32 ? 1 : HD / 32;     // K steps of a product over dims
  static constexpr int kDt = HD / 16;                   // 16-dim output tiles
  static constexpr int kPieces = kTile * HD / 8;        // 16-byte pieces of a chunk
  static constexpr int kPer = kPieces < 256 ? 1 : kPieces / 256;
  // the dims of this lane in K step ks (HD = 16: lanes g >= 2 hold zeros)
  static __device__ __forceinline__ int kdim(int ks, int g) { return HD < 32 ? 8 * (g & 1) : 32 * ks + 8 * g; }
};

// A 64-row chunk of one operand: fetched to registers (zeros at or past L),
// staged as rows, as transposed rows, or both.
template <bool kHalf, int HD>
struct Chunk {
  using G = Geom<kHalf, HD>;
  uint4 reg[G::kPer];
  __device__ __forceinline__ void fetch(const uint16_t* base, int64_t st, int64_t first, int64_t L) {
#pragma unroll
    for (int r = 0; r < G::kPer; ++r) {
      const int i = int(threadIdx.x) + 256 * r;
      const int64_t row = first + i / (HD / 8);
      reg[r] = make_uint4(0u, 0u, 0u, 0u);
      if (i < G::kPieces && row < L) reg[r] = *reinterpret_cast<const uint4*>(base + row * st + 8 * (i % (HD / 8)));
    }
  }
  __device__ __forceinline__ void stage_rows(uint16_t* s) const {
#pragma unroll
    for (int r = 0; r < G::kPer; ++r) {
      const int i = int(threadIdx.x) + 256 * r;
      if (i < G::kPieces)
        *reinterpret_cast<uint4*>(s + (i / (HD / 8)) * G::kPitch + 8 * (i % (HD / 8))) = reg[r];
    }
  }
  __device__ __forceinline__ void stage_transposed(uint16_t* s) const {
#pragma unroll
    for (int r = 0; r < G::kPer; ++r) {
      const int i = int(threadIdx.x) + 256 * r;
      if (i >= G::kPieces) continue;
      uint16_t* col = s + 8 * (i % (HD / 8)) * kTPitch + i / (HD / 8);
      const uint32_t w[4] = {reg[r].x, reg[r].y, reg[r].z, reg[r].w};
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        col[2 * e * kTPitch] = uint16_t(w[e]);
        col[(2 * e + 1) * kTPitch] = uint16_t(w[e] >> 16);
      }
    }
  }
};

// this lane's row of one side as B fragments, zeros when it is not live
template <bool kHalf, int HD>
__device__ __forceinline__ void load_frags(const uint16_t* row, bool live, int g,
                                           uint4 (&u)[Geom<kHalf, HD>::kKs]) {
  using G = Geom<kHalf, HD>;
#pragma unroll
  for (int ks = 0; ks < G::kKs; ++ks) {
    u[ks] = make_uint4(0u, 0u, 0u, 0u);
    if (live && (HD >= 32 || g < 2)) u[ks] = *reinterpret_cast<const uint4*>(row + G::kdim(ks, g));
  }
}

// 4 tiles of 16 staged rows times this lane's row, those with a row below n (HD = 16: the upper K slots
// are zeros on both sides, so an infinite row meets none of them)
template <bool kHalf, int HD>
__device__ __forceinline__ void products(const uint16_t* s, int n, int l16, int g, const uint4 (&b)[Geom<kHalf, HD>::kKs],
                                         f32x4_t (&d)[4]) {
  using G = Geom<kHalf, HD>;
  using FR = Frag<kHalf>;
#pragma unroll
  for (int tt = 0; tt < 4; ++tt) {
    d[tt] = f32x4_t{0.f, 0.f, 0.f, 0.f};
    if (16 * tt >= n) continue;  // uniform
#pragma unroll
    for (int ks = 0; ks < G::kKs; ++ks) {
      uint4 a = *reinterpret_cast<const uint4*>(s + (16 * tt + l16) * G::kPitch + G::kdim(ks, g));
      if (HD < 32 && g >= 2) a = make_uint4(0u, 0u, 0u, 0u);
      d[tt] = mfma16x16x32(FR::cast(a), FR::cast(b[ks]), d[tt]);
    }
  }
}

// acc (HD dims x this lane's row) += transposed rows . x over a chunk's tiles with
// a row below n, x the 16 fp32 values of this lane (rows 16 tt + 4 g + t), on the fp32 MFMA
// (16 x 16 x 4: lane group g holds K slot g of both operands)
template <bool kHalf, int HD>
__device__ __forceinline__ void accumulate(const uint16_t* st, int n, int l16, int g, const float (&x)[4][4],
                                           f32x4_t (&acc)[Geom<kHalf, HD>::kDt]) {
#pragma unroll
  for (int tt = 0; tt < 4; ++tt) {
    if (16 * tt >= n) break;  // uniform
    uint2 a[Geom<kHalf, HD>::kDt];
#pragma unroll
    for (int dt = 0; dt < Geom<kHalf, HD>::kDt; ++dt)
      a[dt] = *reinterpret_cast<const uint2*>(st + (16 * dt + l16) * kTPitch + 16 * tt + 4 * g);
#pragma unroll
    for (int t = 0; t < 4; ++t)
#pragma unroll
      for (int dt = 0; dt < Geom<kHalf, HD>::kDt; ++dt) {
        const uint32_t w = t < 2 ? a[dt].x : a[dt].y;
        const float v = widen<kHalf>(t % 2 ? w >> 16 : w & 0xffffu);
        acc[dt] = __builtin_amdgcn_mfma_f32_16x16x4f32(v, x[tt][t], acc[dt], 0, 0, 0);
      }
  }
}

// a lane's row of HD gradients (dims 16 dt + 4 g + t), zeros when not live
template <bool kHalf, int HD>
__device__ __forceinline__ void store_row(uint16_t* row, int g, const f32x4_t (&acc)[Geom<kHalf, HD>::kDt],
                                          float scale, bool live) {
#pragma unroll
  for (int dt = 0; dt < Geom<kHalf, HD>::kDt; ++dt) {
    uint2 w = make_uint2(0u, 0u);
    if (live) {
      w.x = Frag<kHalf>::pack(acc[dt][0] * scale, acc[dt][1] * scale);
      w.y = Frag<kHalf>::pack(acc[dt][2] * scale, acc[dt][3] * scale);
    }
    *reinterpret_cast<uint2*>(row + 16 * dt + 4 * g) = w;
  }
}

template <bool kHalf, int HD>
__global__ void __launch_bounds__(256)
stone_bwd_q_kernel(Rows q, Rows k, Rows v, Rows o, Rows go, const int32_t* __restrict__ seq_lens, int heads,
                   int64_t T, const float* __restrict__ lse, float scale, float* __restrict__ delta, RowsOut dq) {
  using G = Geom<kHalf, HD>;
  __shared__ __attribute__((aligned(16))) uint16_t sk[kTile * G::kPitch], sv[kTile * G::kPitch];
  __shared__ __attribute__((aligned(16))) uint16_t skt[HD * kTPitch];
  const int64_t n_tiles = (T + kTile - 1) / kTile;
  const int64_t pa = blockIdx.x / n_tiles, tile = blockIdx.x % n_tiles;
  const int64_t pos = pa / heads, a = pa % heads;
  int64_t L = seq_lens[pos];
  L = L < 0 ? 0 : (L > T ? T : L);
  const int lane = threadIdx.x % 64, l16 = lane % 16, g = lane / 16;
  const int64_t first = tile * kTile + 16 * (threadIdx.x / 64), i = first + l16;
  const bool live = i < L;
  uint4 qf[G::kKs], gf[G::kKs], of[G::kKs];
  load_frags<kHalf, HD>(q.at(pos, a) + i * q.st, live, g, qf);
  load_frags<kHalf, HD>(go.at(pos, a) + i * go.st, live, g, gf);
  load_frags<kHalf, HD>(o.at(pos, a) + i * o.st, live, g, of);
  const float li = live ? lse[pa * T + i] : 0.f;
  float dl = 0.f;
#pragma unroll
  for (int ks = 0; ks < G::kKs; ++ks) {
    const uint32_t x[4] = {of[ks].x, of[ks].y, of[ks].z, of[ks].w}, y[4] = {gf[ks].x, gf[ks].y, gf[ks].z, gf[ks].w};
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      dl = fmaf(widen<kHalf>(x[e] & 0xffffu), widen<kHalf>(y[e] & 0xffffu), dl);
      dl = fmaf(widen<kHalf>(x[e] >> 16), widen<kHalf>(y[e] >> 16), dl);
    }
  }
  dl = sum_xor32(sum_xor16(dl));
  f32x4_t acc[G::kDt];
#pragma unroll
  for (int dt = 0; dt < G::kDt; ++dt) acc[dt] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  if (tile * kTile < L) {  // workgroup-uniform: some row of the tile is live
    const uint16_t* kp = k.at(pos, a);
    const uint16_t* vp = v.at(pos, a);
    Chunk<kHalf, HD> ck, cv;
    ck.fetch(kp, k.st, 0, L);
    cv.fetch(vp, v.st, 0, L);
    for (int64_t kb = 0; kb < L; kb += kTile) {
      __syncthreads();  // the last chunk's readers are done
      ck.stage_rows(sk);
      ck.stage_transposed(skt);
      cv.stage_rows(sv);
      __syncthreads();
      if (kb + kTile < L) {
        ck.fetch(kp, k.st, kb + kTile, L);
        cv.fetch(vp, v.st, kb + kTile, L);
      }
      if (first >= L) continue;  // wavefront-uniform: no live row here
      f32x4_t s[4], dp[4];
      const int n = int(L - kb < kTile ? L - kb : kTile);
      products<kHalf, HD>(sk, n, l16, g, qf, s);
      products<kHalf, HD>(sv, n, l16, g, gf, dp);
      const int lim = n - 4 * g;  // keys 16 tt + t below it are live
      float ds[4][4];
#pragma unroll
      for (int tt = 0; tt < 4; ++tt)
#pragma unroll
        for (int t = 0; t < 4; ++t) {
          const float al = __builtin_amdgcn_exp2f(fmaf(s[tt][t], scale, -li) * kLog2e);
          ds[tt][t] = 16 * tt + t < lim ? al * (dp[tt][t] - dl) : 0.f;
        }
      accumulate<kHalf, HD>(skt, n, l16, g, ds, acc);
    }
  }
  if (i < T) {
    store_row<kHalf, HD>(dq.row(pos, a, i), g, acc, scale, live);
    if (g == 0) delta[pa * T + i] = live ? dl : 0.f;
  }
}

template <bool kHalf, int HD>
__global__ void __launch_bounds__(256)
stone_bwd_kv_kernel(Rows q, Rows k, Rows v, Rows go, const int32_t* __restrict__ seq_lens, int heads, int64_t T,
                    const float* __restrict__ lse, float scale, const float* __restrict__ delta, RowsOut dk,
                    RowsOut dv) {
  using G = Geom<kHalf, HD>;
  __shared__ __attribute__((aligned(16))) uint16_t sq[kTile * G::kPitch], sg[kTile * G::kPitch];
  __shared__ __attribute__((aligned(16))) uint16_t sqt[HD * kTPitch], sgt[HD * kTPitch];
  __shared__ __attribute__((aligned(16))) float sl[kTile], sd[kTile];
  const int64_t n_tiles = (T + kTile - 1) / kTile;
  const int64_t pa = blockIdx.x / n_tiles, tile = blockIdx.x % n_tiles;
  const int64_t pos = pa / heads, a = pa % heads;
  int64_t L = seq_lens[pos];
  L = L < 0 ? 0 : (L > T ? T : L);
  const int lane = threadIdx.x % 64, l16 = lane % 16, g = lane / 16;
  const int64_t first = tile * kTile + 16 * (threadIdx.x / 64), j = first + l16;
  const bool live = j < L;
  uint4 kf[G::kKs], vf[G::kKs];
  load_frags<kHalf, HD>(k.at(pos, a) + j * k.st, live, g, kf);
  load_frags<kHalf, HD>(v.at(pos, a) + j * v.st, live, g, vf);
  f32x4_t ak[G::kDt], av[G::kDt];
#pragma unroll
  for (int dt = 0; dt < G::kDt; ++dt) ak[dt] = av[dt] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  if (tile * kTile < L) {  // workgroup-uniform
    const uint16_t* qp = q.at(pos, a);
    const uint16_t* gp = go.at(pos, a);
    Chunk<kHalf, HD> cq, cg;
    float rl = 0.f, rd = 0.f;
    auto fetch = [&](int64_t qb) {
      cq.fetch(qp, q.st, qb, L);
      cg.fetch(gp, go.st, qb, L);
      if (threadIdx.x < kTile) {
        const bool in = qb + threadIdx.x < L;
        rl = in ? lse[pa * T + qb + threadIdx.x] : 0.f;
        rd = in ? delta[pa * T + qb + threadIdx.x] : 0.f;
      }
    };
    fetch(0);
    for (int64_t qb = 0; qb < L; qb += kTile) {
      __syncthreads();
      cq.stage_rows(sq);
      cq.stage_transposed(sqt);
      cg.stage_rows(sg);
      cg.stage_transposed(sgt);
      if (threadIdx.x < kTile) {
        sl[threadIdx.x] = rl;
        sd[threadIdx.x] = rd;
      }
      __syncthreads();
      if (qb + kTile < L) fetch(qb + kTile);
      if (first >= L) continue;  // wavefront-uniform
      f32x4_t s[4], dp[4];
      const int n = int(L - qb < kTile ? L - qb : kTile);
      products<kHalf, HD>(sq, n, l16, g, kf, s);
      products<kHalf, HD>(sg, n, l16, g, vf, dp);
      const int lim = n - 4 * g;  // queries 16 tt + t below it are live
      float al[4][4], ds[4][4];
#pragma unroll
      for (int tt = 0; tt < 4; ++tt) {
        const float4 l4 = *reinterpret_cast<const float4*>(&sl[16 * tt + 4 * g]);
        const float4 d4 = *reinterpret_cast<const float4*>(&sd[16 * tt + 4 * g]);
        const float lv[4] = {l4.x, l4.y, l4.z, l4.w}, dv4[4] = {d4.x, d4.y, d4.z, d4.w};
#pragma unroll
        for (int t = 0; t < 4; ++t) {
          const float e = __builtin_amdgcn_exp2f(fmaf(s[tt][t], scale, -lv[t]) * kLog2e);
          al[tt][t] = 16 * tt + t < lim ? e : 0.f;
          ds[tt][t] = 16 * tt + t < lim ? e * (dp[tt][t] - dv4[t]) : 0.f;
        }
      }
      accumulate<kHalf, HD>(sgt, n, l16, g, al, av);
      accumulate<kHalf, HD>(sqt, n, l16, g, ds, ak);
    }
  }
  if (j < T) {
    store_row<kHalf, HD>(dk.row(pos, a, j), g, ak, scale, live);
    store_row<kHalf, HD>(dv.row(pos, a, j), g, av, 1.f, live);
  }
}

template <bool kHalf, int HD>
int32_t launch(const Rows& q, const Rows& k, const Rows& v, const Rows& o, const Rows& go, const int32_t* seq_lens,
               int64_t n_pos, int heads, int64_t t, const float* lse, float* delta, const RowsOut& dq,
               const RowsOut& dk, const RowsOut& dv, hipStream_t st) {
  const int64_t grid = n_pos * heads * ((t + kTile - 1) / kTile);
  if (grid > 2147483647LL) return MANTIS_E_ARG;
  const float scale = 1.f / sqrtf(float(HD));
  stone_bwd_q_kernel<kHalf, HD><<<unsigned(grid), 256, 0, st>>>(q, k, v, o, go, seq_lens, heads, t, lse, scale, delta,
                                                                dq);
  stone_bwd_kv_kernel<kHalf, HD><<<unsigned(grid), 256, 0, st>>>(q, k, v, go, seq_lens, heads, t, lse, scale, delta,
                                                                 dk, dv);
  return launched();
}

}  // namespace
}  // namespace mantis

using namespace mantis;

extern "C" int32_t mantis_stone_attention_backward(const void* q, const int64_t* qs, const void* k,
                                                   const int64_t* ks, const void* v, const int64_t* vs,
                                                   const void* out, const int64_t* os, const void* grad_out,
                                                   const int64_t* gs, const float* lse, int32_t dtype,
                                                   const int32_t* seq_lens, int64_t n_pos, int32_t heads, int64_t t,
                                                   int32_t hd, float* delta, void* dq, const int64_t* dqs, void* dk,
                                                   const int64_t* dks, void* dv, const int64_t* dvs, void* stream) {
  if (n_pos == 0 || t == 0) return MANTIS_OK;
  if (!q || !k || !v || !out || !grad_out || !lse || !seq_lens || !delta || !dq || !dk || !dv) return MANTIS_E_ARG;
  if (!qs || !ks || !vs || !os || !gs || !dqs || !dks || !dvs) return MANTIS_E_ARG;
  if ((hd != 16 && hd != 32 && hd != 64) || heads <= 0 || n_pos < 0 || t < 0) return MANTIS_E_ARG;
  if (dtype != MANTIS_BF16 && dtype != MANTIS_F16) return MANTIS_E_ARG;
  // unit dim stride and 16-byte aligned rows everywhere
  for (const int64_t* st : {qs, ks, vs, os, gs, dqs, dks, dvs}) {
    if (st[3] != 1) return MANTIS_E_ARG;
    if ((st[0] | st[1] | st[2]) % 8) return MANTIS_E_ARG;
  }
  for (const void* ptr : {q, k, v, out, grad_out, static_cast<const void*>(dq), static_cast<const void*>(dk),
                          static_cast<const void*>(dv)})
    if (!aligned16(ptr)) return MANTIS_E_ARG;
  auto rows = [](const void* ptr, const int64_t* st) {
    return Rows{static_cast<const uint16_t*>(ptr), st[0], st[1], st[2]};
  };
  auto outs = [](void* ptr, const int64_t* st) { return RowsOut{static_cast<uint16_t*>(ptr), st[0], st[1], st[2]}; };
  const Rows Q = rows(q, qs), K = rows(k, ks), V = rows(v, vs), O = rows(out, os), GO = rows(grad_out, gs);
  const RowsOut DQ = outs(dq, dqs), DK = outs(dk, dks), DV = outs(dv, dvs);
  hipStream_t st = as_stream(stream);
  const bool f16 = dtype == MANTIS_F16;
#define MANTIS_BWD(H, HD_)                                                                                    \
  return launch<H, HD_>(Q, K, V, O, GO, seq_lens, n_pos, heads, t, lse, delta, DQ, DK, DV, st)
  if (hd == 16) {
    if (f16) MANTIS_BWD(true, 16);
    MANTIS_BWD(false, 16);
  }
  if (hd == 32) {
    if (f16) MANTIS_BWD(true, 32);
    MANTIS_BWD(false, 32);
  }
  if (f16) MANTIS_BWD(true, 64);
  MANTIS_BWD(false, 64);
#undef MANTIS_BWD
}

// The production leaf evaluation as one call (MantisNet.forward,
// model.py:898-1200): the composition that mantisnet/forward.py queues launch
// by launch, here from native code over one workspace.  A Python launch costs
// 10-20 us of host time (checks, allocation, argument marshalling), 110 of
// them 1.9 ms per evaluation whatever its size; a batch below about 60
// positions computes in less than that.
//
// The host-side library steps between the launches are kernels here: the
// initial states and small per-batch tables (leaf_init_kernel), prefix sums
// (prefix_*_kernel), the latent output with the heads' position half
// (latent_out_kernel) and the value MLP (value_tail_kernel), all fp32.
#include <algorithm>
#include <initializer_list>

#include "common.hpp"

namespace mantis {
namespace {

constexpr int kBlock = 256;
constexpr int64_t kRow = 128;

// ---------------------------------------------------------------- start

struct InitArgs {
  const int64_t* stone_own;
  const int64_t* moves_idx;
  const int64_t* window_slot;
  const uint8_t* attn_valid;
  const float* stone_table;
  const float* latent_base;
  const float* token_moves;
  int64_t n_pos, max_t, max_w, n_s, n_w;
  float* sg;
  int64_t* window_pos;
  int64_t* layout_order;
  int32_t* seq_lens;
  int32_t* word;
  int32_t* flag;
  int64_t rows_blocks, window_blocks;
};

__global__ void __launch_bounds__(kBlock) leaf_init_kernel(InitArgs a) {
  int64_t b = blockIdx.x;
  if (b < a.rows_blocks) {  // [stones; latents], a float4 per thread
    if (b == 0 && threadIdx.x == 0) *a.word = 0;
    const int64_t i = b * kBlock + threadIdx.x, r = i / 32, c = i % 32;
    if (r >= a.n_s + 4 * a.n_pos) return;
    float4 x;
    if (r < a.n_s) {
      int64_t own = a.stone_own[r];
      if (own < 0 || own > 1) {
        if (c == 0) raise_flag(a.flag, MANTIS_FLAG_INDEX);
        own = 0;
      }
      x = reinterpret_cast<const float4*>(a.stone_table + own * kRow)[c];
    } else {
      const int64_t p = (r - a.n_s) / 4, j = (r - a.n_s) % 4;
      int64_t mv = a.moves_idx[p];
      if (mv < 0 || mv > 1) {
        if (c == 0) raise_flag(a.flag, MANTIS_FLAG_INDEX);
        mv = 0;
      }
      const float4 l = reinterpret_cast<const float4*>(a.latent_base + j * kRow)[c];
      const float4 t = reinterpret_cast<const float4*>(a.token_moves + mv * kRow)[c];
      x = make_float4(l.x + t.x, l.y + t.y, l.z + t.z, l.w + t.w);
    }
    reinterpret_cast<float4*>(a.sg + r * kRow)[c] = x;
    return;
  }
  b -= a.rows_blocks;
  if (b < a.window_blocks) {
    const int64_t i = b * kBlock + threadIdx.x;
    if (i >= a.n_w) return;
    const int64_t s = a.window_slot[i], q = s / a.max_w;
    a.window_pos[i] = s % a.max_w < 0 ? q - 1 : q;  // floor
    a.layout_order[i] = i;
    return;
  }
  b -= a.window_blocks;
  const int64_t p = b * (kBlock / 64) + threadIdx.x / 64;  // a wavefront per position
  if (p >= a.n_pos) return;
  int32_t n = 0;
  for (int64_t t = threadIdx.x % 64; t < a.max_t; t += 64) n += a.attn_valid[p * a.max_t + t] != 0;
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) n += __shfl_xor(n, o);
  if (threadIdx.x % 64 == 0) a.seq_lens[p] = n;
}

// ---------------------------------------------------------------- prefix sums

// Inclusive prefix sums of n small counts in two launches: the totals of 4,096
// items per workgroup, then each workgroup's scan from the sum of the totals
// before it (one launch when one workgroup holds them all).
constexpr int kPer = 16;
constexpr int64_t kSpan = kBlock * kPer;

struct Counts {  // int32 values
  const int32_t* x;
  __device__ int operator()(int64_t i) const { return x[i]; }
};
struct Covered {  // rows of a CSR that have entries
  const int64_t* ptr;
  __device__ int operator()(int64_t i) const { return ptr[i + 1] > ptr[i]; }
};

template <typename F>
__global__ void __launch_bounds__(kBlock) prefix_totals_kernel(F f, int64_t n, int64_t* __restrict__ totals) {
  __shared__ int64_t wave[kBlock / 64];
  int64_t sum = 0;
#pragma unroll
  for (int u = 0; u < kPer; ++u) {
    const int64_t i = int64_t(blockIdx.x) * kSpan + u * kBlock + threadIdx.x;
    if (i < n) sum += f(i);
  }
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) sum += __shfl_xor(sum, o);
  if (threadIdx.x % 64 == 0) wave[threadIdx.x / 64] = sum;
  __syncthreads();
  if (threadIdx.x == 0) totals[blockIdx.x] = wave[0] + wave[1] + wave[2] + wave[3];
}

template <typename F>
__global__ void __launch_bounds__(kBlock)
prefix_scan_kernel(F f, int64_t n, const int64_t* __restrict__ totals, int64_t* __restrict__ out) {
  __shared__ int64_t wave[kBlock / 64], wave2[kBlock / 64];
  const int lane = threadIdx.x % 64, w = threadIdx.x / 64;
  int64_t before = 0;
  for (int64_t b = threadIdx.x; b < blockIdx.x; b += kBlock) before += totals[b];
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) before += __shfl_xor(before, o);
  if (lane == 0) wave[w] = before;
  // this thread's kPer consecutive items
  const int64_t first = int64_t(blockIdx.x) * kSpan + int64_t(threadIdx.x) * kPer;
  int c[kPer], own = 0;
#pragma unroll
  for (int u = 0; u < kPer; ++u) {
    c[u] = first + u < n ? f(first + u) : 0;
    own += c[u];
  }
  int64_t inc = own;
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    const int64_t v = __shfl_up(inc, o);
    if (lane >= o) inc += v;
  }
  if (lane == 63) wave2[w] = inc;
  __syncthreads();
  int64_t run = wave[0] + wave[1] + wave[2] + wave[3] + inc - own;
  for (int k = 0; k < w; ++k) run += wave2[k];
#pragma unroll
  for (int u = 0; u < kPer; ++u) {
    run += c[u];
    if (first + u < n) out[first + u] = run;
  }
}

template <typename F>
void prefix(F f, int64_t n, int64_t* totals, int64_t* out, hipStream_t s) {
  const unsigned blocks = unsigned((n + kSpan - 1) / kSpan);
  if (blocks > 1) prefix_totals_kernel<F><<<blocks, kBlock, 0, s>>>(f, n, totals);
  prefix_scan_kernel<F><<<blocks, kBlock, 0, s>>>(f, n, totals, out);
}

__global__ void zero_i64_kernel(int64_t* p) { *p = 0; }

// ---------------------------------------------------------------- outputs

// Per position: the four latent rows through ln_out, their mean (the position's
// output row) and the heads' position half W g (256 outputs, W transposed).
// A workgroup per position: a chain of L2 round trips for the weights, 16 loads
// in flight.
__global__ void __launch_bounds__(256)
latent_out_kernel(const float* __restrict__ g, const float* __restrict__ gamma, const float* __restrict__ beta,
                  const float* __restrict__ wt, float* __restrict__ g_out, float* __restrict__ g_half) {
  __shared__ float rows[4][kRow];
  __shared__ float mean_row[kRow];
  const int64_t p = blockIdx.x;
  const int r = threadIdx.x / 64, lane = threadIdx.x % 64;
  const float2 x = reinterpret_cast<const float2*>(g + (4 * p + r) * kRow)[lane];
  float s = x.x + x.y;
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) s += __shfl_xor(s, o);
  const float mu = s * (1.f / 128.f), dx = x.x - mu, dy = x.y - mu;
  float v = dx * dx + dy * dy;
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) v += __shfl_xor(v, o);
  const float rstd = rsqrtf(v * (1.f / 128.f) + 1e-5f);
  rows[r][2 * lane] = dx * rstd * gamma[2 * lane] + beta[2 * lane];
  rows[r][2 * lane + 1] = dy * rstd * gamma[2 * lane + 1] + beta[2 * lane + 1];
  __syncthreads();
  if (threadIdx.x < kRow) {
    const int c = threadIdx.x;
    const float m = ((rows[0][c] + rows[1][c]) + (rows[2][c] + rows[3][c])) * 0.25f;
    mean_row[c] = m;
    g_out[p * kRow + c] = m;
  }
  __syncthreads();
  float acc[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll 4
  for (int k = 0; k < int(kRow); k += 4)
#pragma unroll
    for (int u = 0; u < 4; ++u) acc[u] = fmaf(wt[(k + u) * 256 + threadIdx.x], mean_row[k + u], acc[u]);
  g_half[p * 256 + threadIdx.x] = (acc[0] + acc[1]) + (acc[2] + acc[3]);
}

// The value MLP of kPosV positions per workgroup: hidden = relu(W0 r + b0) (512
// -> 128), logits = W2 hidden + b2, their softmax and its mean over the bins.
// The inner dimension of each product is cut over the 8 groups of 128 threads
// (one thread per output), so a weight load serves the positions and the chain
// per thread is 64 loads, 16 in flight.
constexpr int kPosV = 4;
__global__ void __launch_bounds__(1024)
value_tail_kernel(const float* __restrict__ read, int64_t n_pos, const float* __restrict__ w0,
                  const float* __restrict__ b0, const float* __restrict__ w2, const float* __restrict__ b2, int n_bins,
                  const float* __restrict__ bins, float* __restrict__ value, float* __restrict__ dist,
                  float* __restrict__ logits) {
  constexpr int kParts = 8;
  __shared__ float in[kPosV][512];
  __shared__ float part[kParts][kPosV][kRow];
  __shared__ float hid[kPosV][kRow];
  const int64_t p0 = int64_t(blockIdx.x) * kPosV;
  const int o = threadIdx.x % 128, g = threadIdx.x / 128;
  for (int i = threadIdx.x; i < kPosV * 512; i += 1024)
    in[i / 512][i % 512] = p0 + i / 512 < n_pos ? read[p0 * 512 + i] : 0.f;
  __syncthreads();
  float acc[kPosV] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll 16
  for (int k = g * 64; k < g * 64 + 64; ++k) {
    const float w = w0[k * 128 + o];
#pragma unroll
    for (int j = 0; j < kPosV; ++j) acc[j] = fmaf(w, in[j][k], acc[j]);
  }
#pragma unroll
  for (int j = 0; j < kPosV; ++j) part[g][j][o] = acc[j];
  __syncthreads();
  if (g < kPosV) {
    float s = b0[o];
#pragma unroll
    for (int k = 0; k < kParts; ++k) s += part[k][g][o];
    hid[g][o] = s < 0.f ? 0.f : s;  // (a NaN stays one: fmaxf would answer 0)
  }
  __syncthreads();
#pragma unroll
  for (int j = 0; j < kPosV; ++j) acc[j] = 0.f;
  if (o < n_bins) {
#pragma unroll
    for (int k = 0; k < 16; ++k) {
      const float w = w2[(g * 16 + k) * n_bins + o];
#pragma unroll
      for (int j = 0; j < kPosV; ++j) acc[j] = fmaf(w, hid[j][g * 16 + k], acc[j]);
    }
  }
#pragma unroll
  for (int j = 0; j < kPosV; ++j) part[g][j][o] = acc[j];
  __syncthreads();
  // a wavefront per position: bins lane and lane + 64
  const int j = threadIdx.x / 64, lane = threadIdx.x % 64;
  if (j >= kPosV || p0 + j >= n_pos) return;
  float x[2], m = -INFINITY;
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    const int c = lane + 64 * h;
    x[h] = -INFINITY;
    if (c < n_bins) {
      float s = b2[c];
#pragma unroll
      for (int k = 0; k < kParts; ++k) s += part[k][j][c];
      x[h] = s;
      logits[(p0 + j) * n_bins + c] = s;
    }
    m = fmaxf(m, x[h]);
  }
#pragma unroll
  for (int d = 1; d < 64; d <<= 1) m = fmaxf(m, __shfl_xor(m, d));
  float e[2], sum = 0.f;
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    e[h] = lane + 64 * h < n_bins ? expf(x[h] - m) : 0.f;
    sum += e[h];
  }
#pragma unroll
  for (int d = 1; d < 64; d <<= 1) sum += __shfl_xor(sum, d);
  float mean = 0.f;
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    const int c = lane + 64 * h;
    if (c < n_bins) {
      const float q = e[h] / sum;
      dist[(p0 + j) * n_bins + c] = q;
      mean = fmaf(q, bins[c], mean);
    }
  }
#pragma unroll
  for (int d = 1; d < 64; d <<= 1) mean += __shfl_xor(mean, d);
  if (lane == 0) value[p0 + j] = mean;
}

// ---------------------------------------------------------------- workspace

struct Carve {  // 256-byte aligned pieces of the workspace
  char* base;
  int64_t used = 0;
  template <typename T>
  T* take(int64_t n) {
    T* p = base ? reinterpret_cast<T*>(base + used) : nullptr;
    used += (n * int64_t(sizeof(T)) + 255) / 256 * 256;
    return p;
  }
};

typedef _Float16 half;

struct Space {
  // plan
  int64_t *window_pos, *layout_order, *inc_win_ptr, *inc_stone_ptr, *run_window, *run_class, *layout_offsets, *cell_ptr,
      *radius_ptr, *radius_class, *rank, *totals, *cov_rows, *wcell, *wclass, *win_ptr, *attn_src, *attn_back;
  int32_t *seq_lens, *cell_order, *schedule;
  char* key_ws;
  // rows
  half *w, *c, *x_s, *agg_w, *cr_kv, *rad_kv, *wr_kv, *wp, *qkv, *attn, *qx, *kvb, *pre;
  float *sg, *sw_all, *agg_s, *read, *lread_ws, *vread, *vread_ws, *g_out, *g_half;
  int64_t n_schedule, bytes;

  Space(void* ws, const mantis_leaf_batch& b, int64_t n_blocks) {
    Carve k{static_cast<char*>(ws)};
    const int64_t p = b.n_pos, slots = p * b.max_t, sg_rows = b.n_s + 4 * p;
    window_pos = k.take<int64_t>(b.n_w);
    layout_order = k.take<int64_t>(b.n_w);
    inc_win_ptr = k.take<int64_t>(b.n_w + 1);
    inc_stone_ptr = k.take<int64_t>(b.n_s + 1);
    run_window = k.take<int64_t>(b.n_inc);
    run_class = k.take<int64_t>(b.n_inc);
    layout_offsets = k.take<int64_t>(p + 1);
    cell_ptr = k.take<int64_t>(b.n_c + 1);
    radius_ptr = k.take<int64_t>(b.n_c + 1);
    radius_class = k.take<int64_t>(b.n_rad);
    rank = k.take<int64_t>(b.n_c);
    totals = k.take<int64_t>((std::max(b.n_c, b.n_s) + kSpan - 1) / kSpan);
    cov_rows = k.take<int64_t>(b.n_cov);
    wcell = k.take<int64_t>(b.n_dec);
    wclass = k.take<int64_t>(b.n_dec);
    win_ptr = k.take<int64_t>(b.n_w + 1);
    attn_src = k.take<int64_t>(slots);
    attn_back = k.take<int64_t>(sg_rows);
    seq_lens = k.take<int32_t>(p);
    cell_order = k.take<int32_t>(b.n_c);
    // (as ops.stone_attention_schedule: one 128-query tile needs no order)
    n_schedule = b.max_t > 128 ? mantis_stone_attention_schedule_len(p, 4, b.max_t) : 0;
    schedule = k.take<int32_t>(n_schedule);
    key_ws = k.take<char>(mantis_stable_key_order_workspace(b.n_inc, b.n_s));
    w = k.take<half>(b.n_w * kRow);
    c = k.take<half>(b.n_c * kRow);
    x_s = k.take<half>(b.n_s * kRow);
    agg_w = k.take<half>(b.n_w * kRow);
    cr_kv = k.take<half>(b.n_w * 2 * kRow);
    rad_kv = k.take<half>(b.n_s * 2 * kRow);
    wr_kv = k.take<half>(b.n_cov * 2 * kRow);
    wp = k.take<half>(b.n_w * kRow);
    qkv = k.take<half>(slots * 3 * kRow);
    attn = k.take<half>(slots * kRow);
    qx = k.take<half>(4 * p * 4 * kRow);
    kvb = k.take<half>(4 * p * 2 * kRow);
    pre = k.take<half>(b.n_w * kRow);
    sg = k.take<float>(sg_rows * kRow);
    sw_all = k.take<float>(b.n_s * n_blocks * kRow);
    agg_s = k.take<float>(b.n_s * kRow);
    read = k.take<float>(4 * p * kRow);
    lread_ws = k.take<float>(mantis_latent_read_x_workspace(p) / 4);
    vread = k.take<float>(4 * p * kRow);
    vread_ws = k.take<float>(mantis_value_read_workspace(p) / 4);
    g_out = k.take<float>(p * kRow);
    g_half = k.take<float>(p * 2 * kRow);
    bytes = k.used;
  }
};

bool sizes_ok(const mantis_leaf_batch& b) {
  for (int64_t n : {b.n_pos, b.max_w, b.n_s, b.n_w, b.n_c, b.n_cov, b.n_inc, b.n_rad, b.n_dec})
    if (n < 1 || n > 2147483647LL) return false;
  return b.max_t >= 4 && b.max_t <= 2048 && b.n_pos * b.max_t <= 2147483647LL;
}

using Ptrs = std::initializer_list<const void*>;
bool all_set(Ptrs ps) { return std::all_of(ps.begin(), ps.end(), [](const void* p) { return p != nullptr; }); }
bool all_aligned(Ptrs ps) { return std::all_of(ps.begin(), ps.end(), [](const void* p) { return aligned16(p); }); }

// What the launches below read without a check of their own, and what the
// entry points they call would refuse once launches before them are queued.
// (The biases of the row projections may be null, as those entries take them.)
bool batch_ok(const mantis_leaf_batch& b) {
  return all_set({b.stone_own, b.window_feat, b.moves_idx, b.inc_stone, b.inc_window, b.inc_class, b.stone_slot,
                  b.window_slot, b.legal_offsets, b.cell_pos, b.cell_nearest, b.radius_src, b.radius_dst,
                  b.radius_orbit, b.radius_own, b.radius_on_axis, b.dec_cell, b.dec_window, b.dec_class, b.act_class,
                  b.act_rev, b.act_empty, b.attn_valid});
}

bool block_ok(const mantis_leaf_block& B) {
  return all_set({B.u_w, B.mlp_w1_w, B.mlp_w2_w, B.mlp_w3_w, B.cr_kv_w, B.cr_q_w, B.cr_q_b, B.cr_o_w, B.cr_o_b,
                  B.cr_bias, B.rad_kv_w, B.rad_q_w, B.rad_q_b, B.rad_o_w, B.rad_o_b, B.radius_bias, B.wr_kv_w,
                  B.wr_q_w, B.wr_q_b, B.wr_o_w, B.wr_o_b, B.wr_bias, B.wproj_w, B.wproj_b, B.mlp_s1_w, B.mlp_s2_w,
                  B.mlp_s3_w, B.qkv_w, B.attn_o_w, B.lq_read_x_w, B.lread_v_w, B.lread_v_b, B.lo_read_w, B.mix_qkv_wt,
                  B.mix_qkv_b, B.mix_o_wt, B.mix_o_b, B.lkv_bcast_w, B.bcast_q_w, B.bcast_q_b, B.lo_bcast_w,
                  B.lo_bcast_b, B.ffn1_w, B.ffn2_w}) &&
         (B.cr_vcls == nullptr) == (B.rad_vcls == nullptr) &&
         all_aligned({B.u_w, B.u_b, B.mlp_w1_w, B.mlp_w1_b, B.mlp_w2_w, B.ws_tab, B.mlp_w3_w, B.mlp_w3_b, B.cr_kv_w,
                      B.cr_kv_b, B.cr_q_w, B.cr_q_b, B.cr_o_w, B.cr_o_b, B.cr_vcls, B.rad_kv_w, B.rad_kv_b, B.rad_q_w,
                      B.rad_q_b, B.rad_o_w, B.rad_o_b, B.rad_vcls, B.wr_kv_w, B.wr_kv_b, B.wr_q_w, B.wr_q_b, B.wr_o_w,
                      B.wr_o_b, B.wproj_w, B.wproj_b, B.mlp_s1_w, B.mlp_s1_b, B.mlp_s2_w, B.mlp_s3_w, B.mlp_s3_b,
                      B.qkv_w, B.qkv_b, B.attn_o_w, B.attn_o_b, B.lq_read_x_w, B.lq_read_x_b, B.lread_v_w, B.lo_read_w,
                      B.lo_read_b, B.lkv_bcast_w, B.lkv_bcast_b, B.bcast_q_w, B.bcast_q_b, B.lo_bcast_w, B.lo_bcast_b,
                      B.ffn1_w, B.ffn1_b, B.ffn2_w, B.ffn2_b});
}

bool model_ok(const mantis_leaf_model& M, bool full) {
  if (M.n_blocks < 1 || !M.blocks) return false;
  for (int64_t i = 0; i < M.n_blocks; ++i)
    if (!block_ok(M.blocks[i])) return false;
  if (full && (M.n_bins < 1 || M.n_bins > 128 ||
               !all_set({M.ln_value_w, M.ln_value_b, M.value_queries, M.mlp_v0_wt, M.mlp_v0_b, M.mlp_v2_wt, M.mlp_v2_b})))
    return false;
  for (int64_t n : {M.n_patterns, M.n_init, M.n_occ, M.n_dec_classes, M.n_rad_classes, M.n_act})
    if (n < 1) return false;
  return all_set({M.window_table, M.cell_table, M.stone_table, M.latent_base, M.token_moves, M.sw_all, M.ln_out_w,
                  M.ln_out_b, M.act_proj_w, M.head1_w, M.head1_b, M.head2_w, M.head3_w, M.head3_b, M.act_table,
                  M.empty_rows, M.head_tab, M.glin_wt}) &&
         all_aligned({M.window_table, M.cell_table, M.stone_table, M.latent_base, M.token_moves, M.act_proj_w,
                      M.act_proj_b, M.head1_w, M.head1_b, M.head2_w, M.head3_w, M.head3_b, M.act_table, M.empty_rows,
                      M.head_tab});
}

}  // namespace
}  // namespace mantis

using namespace mantis;

extern "C" {

int32_t mantis_latent_out(const float* g, int64_t n_pos, const float* gamma, const float* beta, const float* glin_wt,
                          float* g_out, float* g_half, void* stream) {
  if (n_pos == 0) return MANTIS_OK;
  if (!g || !gamma || !beta || !glin_wt || !g_out || !g_half || n_pos < 0 || n_pos > 2147483647LL || !aligned16(g))
    return MANTIS_E_ARG;
  latent_out_kernel<<<unsigned(n_pos), 256, 0, as_stream(stream)>>>(g, gamma, beta, glin_wt, g_out, g_half);
  return launched();
}

int32_t mantis_value_tail(const float* read, int64_t n_pos, const float* w0_t, const float* b0, const float* w2_t,
                          const float* b2, int64_t n_bins, const float* bin_centers, float* value, float* dist,
                          float* logits, void* stream) {
  if (n_pos == 0) return MANTIS_OK;
  if (!read || !w0_t || !b0 || !w2_t || !b2 || !bin_centers || !value || !dist || !logits || n_pos < 0 ||
      n_pos > 2147483647LL || n_bins < 1 || n_bins > 128)
    return MANTIS_E_ARG;
  value_tail_kernel<<<unsigned((n_pos + kPosV - 1) / kPosV), 1024, 0, as_stream(stream)>>>(
      read, n_pos, w0_t, b0, w2_t, b2, int(n_bins), bin_centers, value, dist, logits);
  return launched();
}

int64_t mantis_leaf_workspace(const mantis_leaf_batch* batch, int64_t n_blocks) {
  if (!batch || n_blocks < 1 || !sizes_ok(*batch)) return -1;
  return Space(nullptr, *batch, n_blocks).bytes;
}

int32_t mantis_leaf_forward(const mantis_leaf_model* model, const mantis_leaf_batch* batch,
                            const mantis_leaf_out* out, float mass_floor, void* workspace, int64_t workspace_bytes,
                            int32_t* noncanonical, int32_t* err_flag, uint32_t* tile_counters, void* stream) {
  if (!model || !batch || !out || !workspace || !noncanonical || !tile_counters) return MANTIS_E_ARG;
  const mantis_leaf_model& M = *model;
  const mantis_leaf_batch& b = *batch;
  const bool full = out->value != nullptr;
  if (!sizes_ok(b) || !batch_ok(b) || !model_ok(M, full) || !out->rows || !aligned16(out->rows)) return MANTIS_E_ARG;
  if (full && !all_set({out->policy, out->q_values, out->q_score, out->dist, out->logits, out->bin_centers}))
    return MANTIS_E_ARG;
  const Space S(workspace, b, M.n_blocks);
  if (workspace_bytes < S.bytes || (reinterpret_cast<uintptr_t>(workspace) & 255u)) return MANTIS_E_ARG;
  hipStream_t st = as_stream(stream);
  int32_t rc = MANTIS_OK;
  // every launch below runs only while the ones before it were accepted
#define MANTIS_DO(call)                 \
  do {                                  \
    if (rc == MANTIS_OK) rc = (call);   \
  } while (0)
  const int64_t p = b.n_pos, n_sg = b.n_s + 4 * p, slots = p * b.max_t;
  float* const s = S.sg;
  float* const g = S.sg + b.n_s * kRow;
  auto linear = [&](const void* x, int32_t xdt, int64_t ldx, const int64_t* rows, int64_t n_x, int64_t m, int ln,
                    const void* w1, const float* b1, int32_t n1, int32_t mode, void* to, int64_t ldo) {
    return mantis_fused_linear(x, xdt, ldx, rows, n_x, m, ln, nullptr, 0, 0, w1, nullptr, b1, n1, nullptr, 0, nullptr,
                               nullptr, 0, 0, nullptr, nullptr, 0, mode, to, ldo, err_flag, stream);
  };
  constexpr int32_t kF16 = MANTIS_F16, kF32 = MANTIS_F32;
  constexpr int32_t kOut16 = 0, kAdd32 = 2, kAdd16 = 3, kFrom16 = 4;  // fused_linear out_mode

  // ---- the index plan and the initial rows
  InitArgs ia{b.stone_own, b.moves_idx, b.window_slot, b.attn_valid, M.stone_table, M.latent_base, M.token_moves,
              p, b.max_t, b.max_w, b.n_s, b.n_w, S.sg, S.window_pos, S.layout_order, S.seq_lens, noncanonical,
              err_flag, (n_sg * 32 + kBlock - 1) / kBlock, (b.n_w + kBlock - 1) / kBlock};
  const int64_t init_blocks = ia.rows_blocks + ia.window_blocks + (p + 3) / 4;
  if (init_blocks > 2147483647LL) return MANTIS_E_ARG;
  leaf_init_kernel<<<unsigned(init_blocks), kBlock, 0, st>>>(ia);
  MANTIS_DO(launched());
  MANTIS_DO(mantis_runs_to_ptr(b.inc_window, b.n_inc, b.n_w, S.inc_win_ptr, err_flag, stream));
  const mantis_leaf_block& B0 = M.blocks[0];
  auto windows_from_stones = [&](const mantis_leaf_block& B, bool first) {  // windows <- stones
    MANTIS_DO(linear(s, kF32, kRow, nullptr, b.n_s, b.n_s, 1, B.u_w, B.u_b, 128, kOut16, S.x_s, kRow));
    MANTIS_DO(mantis_run_reduce(S.x_s, kF16, b.n_s, kRow, kRow, b.inc_stone, b.n_inc, S.inc_win_ptr, b.n_w, S.agg_w,
                                kF16, err_flag, stream));
    MANTIS_DO(mantis_fused_linear(first ? M.window_table : S.w, kF16, kRow, first ? b.window_feat : nullptr,
                                  first ? M.n_patterns : b.n_w, b.n_w, 1, S.agg_w, kF16, kRow, B.mlp_w1_w, B.mlp_w2_w,
                                  B.mlp_w1_b, 128, nullptr, 0, B.ws_tab, b.window_feat, M.n_patterns, 1, B.mlp_w3_w,
                                  B.mlp_w3_b, 128, first ? kFrom16 : kAdd16, S.w, kRow, err_flag, stream));
  };
  windows_from_stones(B0, true);  // the first large launches before the rest of the plan
  MANTIS_DO(mantis_plan_check(b.dec_cell, b.dec_window, b.n_dec, b.act_rev, b.radius_dst, b.n_rad, b.window_slot,
                              b.n_w, b.max_w, noncanonical, stream));
  MANTIS_DO(mantis_stable_key_count(b.inc_stone, b.n_inc, b.n_s, S.key_ws, err_flag, stream));
  if (rc != MANTIS_OK) return rc;
  zero_i64_kernel<<<1, 1, 0, st>>>(S.inc_stone_ptr);
  prefix(Counts{reinterpret_cast<const int32_t*>(S.key_ws)}, b.n_s, S.totals, S.inc_stone_ptr + 1, st);
  MANTIS_DO(mantis_stable_key_order(b.inc_stone, b.inc_window, b.inc_class, b.n_inc, b.n_s, S.inc_stone_ptr,
                                    S.run_window, S.run_class, S.key_ws, stream));
  MANTIS_DO(mantis_run_reduce(M.sw_all, kF32, M.n_occ, M.n_blocks * kRow, M.n_blocks * kRow, S.run_class, b.n_inc,
                              S.inc_stone_ptr, b.n_s, S.sw_all, kF32, err_flag, stream));
  MANTIS_DO(mantis_runs_to_ptr(S.window_pos, b.n_w, p, S.layout_offsets, err_flag, stream));
  MANTIS_DO(mantis_runs_to_ptr(b.dec_cell, b.n_dec, b.n_c, S.cell_ptr, err_flag, stream));
  MANTIS_DO(mantis_runs_to_ptr(b.radius_dst, b.n_rad, b.n_c, S.radius_ptr, err_flag, stream));
  MANTIS_DO(mantis_radius_class(b.radius_orbit, b.radius_own, b.radius_on_axis, b.n_rad, S.radius_class, stream));
  MANTIS_DO(mantis_segment_order(b.legal_offsets, p, S.cell_ptr, S.radius_ptr, b.n_c, S.cell_order, err_flag,
                                 stream));
  if (rc != MANTIS_OK) return rc;
  prefix(Covered{S.cell_ptr}, b.n_c, S.totals, S.rank, st);
  MANTIS_DO(mantis_window_view(b.act_rev, b.dec_cell, b.dec_class, b.dec_window, b.n_dec, b.n_w, b.n_c, S.cell_ptr,
                               S.rank, b.n_cov, S.cov_rows, S.wcell, S.wclass, S.win_ptr, err_flag, stream));
  MANTIS_DO(mantis_attention_slots(b.stone_slot, b.n_s, p, b.max_t, S.attn_src, S.attn_back, err_flag, stream));
  if (S.n_schedule > 0)
    MANTIS_DO(mantis_stone_attention_schedule(S.seq_lens, p, 4, b.max_t, S.schedule, stream));

  // ---- the trunk
  for (int64_t i = 0; i < M.n_blocks; ++i) {
    const mantis_leaf_block& B = M.blocks[i];
    const bool last = i + 1 == M.n_blocks;
    if (i > 0) windows_from_stones(B, false);
    // the cell stage: cells <- windows, cells <- stones, then windows <- cells
    // with the stones' value projection of the rows it updates
    MANTIS_DO(linear(S.w, kF16, kRow, nullptr, b.n_w, b.n_w, 1, B.cr_kv_w, B.cr_kv_b, 256, kOut16, S.cr_kv, 256));
    MANTIS_DO(linear(s, kF32, kRow, nullptr, b.n_s, b.n_s, 1, B.rad_kv_w, B.rad_kv_b, 256, kOut16, S.rad_kv, 256));
    const mantis_substage cells[2] = {
        {B.cr_q_w, B.cr_q_b, S.cr_kv, S.cr_kv + kRow, 256, 256, b.n_w, B.cr_bias, M.n_dec_classes, B.cr_vcls,
         S.cell_ptr, b.dec_window, b.dec_class, b.n_dec, B.cr_o_w, B.cr_o_b},
        {B.rad_q_w, B.rad_q_b, S.rad_kv, S.rad_kv + kRow, 256, 256, b.n_s, B.radius_bias, M.n_rad_classes, B.rad_vcls,
         S.radius_ptr, b.radius_src, S.radius_class, b.n_rad, B.rad_o_w, B.rad_o_b}};
    if (i == 0)
      MANTIS_DO(mantis_attention_substages_init(S.c, kF16, kRow, b.n_c, S.cell_order, cells, 2, M.cell_table, kRow,
                                                M.n_init, b.cell_nearest, M.n_init - 1, err_flag, tile_counters,
                                                stream));
    else
      MANTIS_DO(mantis_attention_substages(S.c, kF16, kRow, b.n_c, S.cell_order, cells, 2, err_flag, tile_counters,
                                           stream));
    MANTIS_DO(linear(S.c, kF16, kRow, S.cov_rows, b.n_c, b.n_cov, 1, B.wr_kv_w, B.wr_kv_b, 256, kOut16, S.wr_kv,
                     256));
    const mantis_substage windows = {B.wr_q_w, B.wr_q_b, S.wr_kv, S.wr_kv + kRow, 256, 256, b.n_cov, B.wr_bias,
                                     M.n_dec_classes, nullptr, S.win_ptr, S.wcell, S.wclass, b.n_dec, B.wr_o_w,
                                     B.wr_o_b};
    MANTIS_DO(mantis_attention_substage_project(S.w, kF16, kRow, b.n_w, nullptr, &windows, B.wproj_w, B.wproj_b, S.wp,
                                                kRow, err_flag, tile_counters, stream));
    // stones <- windows
    MANTIS_DO(mantis_run_reduce(S.wp, kF16, b.n_w, kRow, kRow, S.run_window, b.n_inc, S.inc_stone_ptr, b.n_s, S.agg_s,
                                kF32, err_flag, stream));
    MANTIS_DO(mantis_fused_linear(s, kF32, kRow, nullptr, b.n_s, b.n_s, 1, S.agg_s, kF32, kRow, B.mlp_s1_w,
                                  B.mlp_s2_w, B.mlp_s1_b, 128, S.sw_all + i * kRow, M.n_blocks * kRow, nullptr,
                                  nullptr, 0, 1, B.mlp_s3_w, B.mlp_s3_b, 128, kAdd32, s, kRow, err_flag, stream));
    // attention over [latents; stones]
    MANTIS_DO(linear(S.sg, kF32, kRow, S.attn_src, n_sg, slots, 1, B.qkv_w, B.qkv_b, 384, kOut16, S.qkv, 384));
    if (!last) {
      const int64_t in[4] = {b.max_t * 384, 32, 384, 1}, to[4] = {b.max_t * kRow, 32, kRow, 1};
      MANTIS_DO(mantis_stone_attention(S.qkv, in, S.qkv + kRow, in, S.qkv + 2 * kRow, in, kF16, S.seq_lens, p, 4,
                                       b.max_t, 32, S.attn, to, nullptr, S.n_schedule > 0 ? S.schedule : nullptr,
                                       stream));
      MANTIS_DO(linear(S.attn, kF16, kRow, S.attn_back, slots, n_sg, 0, B.attn_o_w, B.attn_o_b, 128, kAdd32, S.sg,
                       kRow));
    } else {
      MANTIS_DO(mantis_latent_attend(S.qkv, kF16, 384, b.attn_valid, p, b.max_t, S.read, stream));
      MANTIS_DO(linear(S.read, kF32, kRow, nullptr, 4 * p, 4 * p, 0, B.attn_o_w, B.attn_o_b, 128, kAdd32, g, kRow));
    }
    // the window-latent cycle
    MANTIS_DO(linear(g, kF32, kRow, nullptr, 4 * p, 4 * p, 1, B.lq_read_x_w, B.lq_read_x_b, 512, kOut16, S.qx, 512));
    MANTIS_DO(mantis_latent_read_x(S.qx, 512, S.w, kRow, S.layout_offsets, nullptr, p, b.n_w, B.lread_v_w,
                                   B.lread_v_b, S.read, S.lread_ws, err_flag, stream));
    MANTIS_DO(linear(S.read, kF32, kRow, nullptr, 4 * p, 4 * p, 0, B.lo_read_w, B.lo_read_b, 128, kAdd32, g, kRow));
    MANTIS_DO(mantis_latent_mix(g, kRow, p, B.mix_qkv_wt, B.mix_qkv_b, B.mix_o_wt, B.mix_o_b, stream));
    MANTIS_DO(linear(g, kF32, kRow, nullptr, 4 * p, 4 * p, 1, B.lkv_bcast_w, B.lkv_bcast_b, 256, kOut16, S.kvb, 256));
    MANTIS_DO(mantis_latent_broadcast_project_residual(B.bcast_q_w, B.bcast_q_b, S.kvb, 256, S.window_pos, p, b.n_w,
                                                       B.lo_bcast_w, B.lo_bcast_b, S.w, kRow, err_flag, stream));
    // FFN (latents only in the last block)
    const int64_t m = last ? 4 * p : n_sg;
    float* const t = last ? g : S.sg;
    MANTIS_DO(mantis_fused_linear(t, kF32, kRow, nullptr, m, m, 1, nullptr, 0, 0, B.ffn1_w, nullptr, B.ffn1_b, 256,
                                  nullptr, 0, nullptr, nullptr, 0, 1, B.ffn2_w, B.ffn2_b, 128, kAdd32, t, kRow,
                                  err_flag, stream));
  }

  // ---- the heads
  MANTIS_DO(mantis_latent_out(g, p, M.ln_out_w, M.ln_out_b, M.glin_wt, S.g_out, S.g_half, stream));
  if (full) {
    MANTIS_DO(mantis_value_read(S.g_out, S.w, kF16, b.n_w, S.layout_offsets, S.layout_order, p, M.ln_out_w,
                                M.ln_out_b, M.ln_value_w, M.ln_value_b, M.value_queries, 4, S.vread, S.vread_ws,
                                err_flag, stream));
    MANTIS_DO(mantis_value_tail(S.vread, p, M.mlp_v0_wt, M.mlp_v0_b, M.mlp_v2_wt, M.mlp_v2_b, M.n_bins,
                                out->bin_centers, out->value, out->dist, out->logits, stream));
  }
  MANTIS_DO(linear(S.w, kF16, kRow, nullptr, b.n_w, b.n_w, 1, M.act_proj_w, M.act_proj_b, 128, kOut16, S.pre, kRow));
  MANTIS_DO(mantis_cell_heads(S.c, kF16, 1, 0, kRow, b.n_c, S.cell_order, M.head1_w, M.head1_b, M.head2_w, M.head3_w,
                              M.head3_b, S.pre, b.n_w, M.act_table, M.n_act, M.empty_rows, b.act_empty, nullptr,
                              M.head_tab, M.n_dec_classes, S.g_half, p, b.cell_pos, S.cell_ptr, b.dec_window,
                              b.act_class, b.dec_class, b.n_dec, out->rows, err_flag, tile_counters, stream));
  if (full)
    MANTIS_DO(mantis_compose_q_rows(out->rows, 4, b.legal_offsets, p, b.n_c, mass_floor, out->policy, out->q_values,
                                    out->q_score, stream));
#undef MANTIS_DO
  return rc;
}

}  // extern "C"

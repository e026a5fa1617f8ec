// Sliced reductions over unbounded runs (class-major entry lists, where one
// class can own most of the entries): every run is cut into slices of at
// most kSlice entries, each slice is summed into a partial row by its own
// lane group, and slice_merge sums each run's partials, a workgroup per run
// and 32 columns or, of many short runs, per 8 runs.  The slice tables come
// from two small kernels: an exclusive scan of the slice counts (slice_ptr,
// one per run) and the first entry of every slice (slice_edge).
// Deterministic: fixed slice bounds, fixed orders.
#pragma once

#include "common.hpp"
#include "gather.hpp"

namespace mantis {
namespace {

// Run entries per partial row: the longest chain of a lane group (and of fp32
// additions: at 128 the sums of 1,200 entries were 1.6 times as far from
// float64), against the partial rows that the merge reads back.
constexpr int64_t kSlice = 64;

// slice_ptr[k] = first slice of class k: the exclusive prefix sum of
// ceil(len_k / kSlice) over the classes (one workgroup, chunks of 1024).
__global__ void __launch_bounds__(1024)
slice_scan_kernel(const int64_t* __restrict__ cls_ptr, int64_t n_cls, int64_t n_edges,
                  int64_t* __restrict__ slice_ptr) {
  __shared__ int64_t part[1024 / 64];
  const int t = threadIdx.x, lane = t % 64, wave = t / 64;
  int64_t carry = 0;
  for (int64_t k0 = 0; k0 < n_cls; k0 += 1024) {
    const int64_t k = k0 + t;
    int64_t n = 0;
    if (k < n_cls) {
      int64_t a, b;
      segment(cls_ptr, k, n_edges, a, b);
      n = (b - a + kSlice - 1) / kSlice;
    }
    // inclusive scan within the wave, then across the 16 waves
    int64_t v = n;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
      const int64_t u = __shfl_up(v, o, 64);
      if (lane >= o) v += u;
    }
    if (lane == 63) part[wave] = v;
    __syncthreads();
    int64_t before = carry;
    for (int w = 0; w < wave; ++w) before += part[w];
    int64_t total = carry;
    for (int w = 0; w < 1024 / 64; ++w) total += part[w];
    if (k < n_cls) slice_ptr[k] = before + v - n;
    __syncthreads();  // part is rewritten by the next chunk
    carry = total;
  }
  if (t == 0) slice_ptr[n_cls] = carry;
}

// slice_edge[s] = first class-ordered entry of slice s, for s in
// [0, n_slices]; slices past the last class's take the end of the runs, so
// their runs are empty.
__global__ void slice_edges_kernel(const int64_t* __restrict__ cls_ptr, const int64_t* __restrict__ slice_ptr,
                                   int64_t n_cls, int64_t n_edges, int64_t n_slices,
                                   int64_t* __restrict__ slice_edge) {
  const int64_t s = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
  if (s > n_slices) return;
  int64_t endc = cls_ptr[n_cls];
  endc = endc < 0 ? 0 : (endc > n_edges ? n_edges : endc);
  if (s >= slice_ptr[n_cls]) {
    slice_edge[s] = endc;
    return;
  }
  // the class k with slice_ptr[k] <= s < slice_ptr[k + 1]
  int64_t lo = 0, hi = n_cls;  // slice_ptr[lo] <= s < slice_ptr[hi]
  while (hi - lo > 1) {
    const int64_t mid = (lo + hi) / 2;
    if (slice_ptr[mid] <= s) lo = mid;
    else hi = mid;
  }
  int64_t a, b;
  segment(cls_ptr, lo, n_edges, a, b);
  slice_edge[s] = a + (s - slice_ptr[lo]) * kSlice;
}

// partial[s] = sum of values[gather[j]] over the entries j of slice s, columns
// 128 blockIdx.y .. (16 lanes per slice and chunk, h a multiple of 8): 16
// indices per load, kLook raw rows in flight from clamped indices (a load under
// a condition or converted at once is waited for before the next).  Bound by
// the latency of the gathered rows while slices are few: the class sums of a
// training step over 96 positions took 63.6 us with four conditional loads,
// 59.3 with these.
template <typename Tin>
__global__ void __launch_bounds__(256)
slice_sum_kernel(const Tin* __restrict__ values, int64_t n_src, int64_t ld, int64_t h,
                 const int64_t* __restrict__ gather, int64_t n_entries, const int64_t* __restrict__ slice_edge,
                 int64_t n_slices, float* __restrict__ partial, int32_t* flag) {
  constexpr int kLook = 8;
  const int64_t s = int64_t(blockIdx.x) * (256 / kGroup) + threadIdx.x / kGroup;
  const int lane = threadIdx.x % kGroup;
  if (s >= n_slices) return;
  const int64_t c0 = int64_t(blockIdx.y) * (kGroup * 8) + lane * 8;
  const bool mine = c0 < h;  // a lane past the width reads the first columns and stores nothing
  const Tin* col = values + (mine ? c0 : 0);
  int64_t st, en;
  segment(slice_edge, s, n_entries, st, en);
  float acc[8] = {0, 0, 0, 0, 0, 0, 0, 0};
  for (int64_t base = st; base < en; base += kGroup) {
    const int cnt = int(en - base < kGroup ? en - base : kGroup);
    const int64_t g = gather[base + (lane < cnt ? lane : cnt - 1)];
    const bool in = g >= 0 && g < n_src;
    if (lane < cnt && !in) raise_flag(flag, MANTIS_FLAG_INDEX);
    const int32_t row = in ? int32_t(g) : -1;  // n_src fits int32 (host check)
    if (n_src <= 0) continue;  // no row to read: every entry is flagged
    for (int j = 0; j < cnt; j += kLook) {
      Chunk8<Tin> x[kLook];
      int32_t r[kLook];
#pragma unroll
      for (int u = 0; u < kLook; ++u) {  // (an entry out of range reads row 0)
        r[u] = __shfl(row, j + u < cnt ? j + u : cnt - 1, kGroup);
        x[u].load(col + int64_t(r[u] < 0 ? 0 : r[u]) * ld);
      }
#pragma unroll
      for (int u = 0; u < kLook; ++u)
        if (j + u < cnt && r[u] >= 0)  // uniform over the group
#pragma unroll
          for (int i = 0; i < 8; ++i) acc[i] += x[u][i];
    }
  }
  if (mine) store8(partial + s * h + c0, acc);
}

// out[k] = sum of the partial rows of run k (slice_ptr[k] .. slice_ptr[k+1])
// over 32 columns by a workgroup: 8 row groups, 8 rows in flight each, then the
// groups by halves.  (A run of 10^5 entries has about 10^3 partial rows; summed
// one after another by one lane group they were 170 us of every class gradient
// at 64-96 positions, here under 20.)
constexpr int kMergeCols = 32;
constexpr int kMergeGroups = 256 / kMergeCols;
template <typename To>
__device__ __forceinline__ void merge_run(const float* __restrict__ partial, int64_t h, int64_t st, int64_t en,
                                          int64_t c, int g, float (&red)[kMergeGroups][kMergeCols], To* to) {
  const int col = threadIdx.x % kMergeCols;
  float acc = 0.f;
  if (c < h) {
    for (int64_t s = st + g; s < en; s += 8 * kMergeGroups) {
      float x[8];
#pragma unroll
      for (int u = 0; u < 8; ++u) {
        const int64_t r = s + u * kMergeGroups;
        x[u] = partial[(r < en ? r : s) * h + c];
      }
#pragma unroll
      for (int u = 0; u < 8; ++u) acc += s + u * kMergeGroups < en ? x[u] : 0.f;
    }
  }
  red[g][col] = acc;
  __syncthreads();
#pragma unroll
  for (int o = kMergeGroups / 2; o > 0; o >>= 1) {
    if (g < o) red[g][col] += red[g + o][col];
    __syncthreads();
  }
  if (g == 0 && c < h) from_f32(*to, red[0][col]);
}

// a workgroup per run and 32 columns
template <typename To>
__global__ void __launch_bounds__(256)
slice_merge_kernel(const float* __restrict__ partial, int64_t h, const int64_t* __restrict__ slice_ptr,
                   int64_t n_slices, To* __restrict__ out) {
  __shared__ float red[kMergeGroups][kMergeCols];
  const int64_t k = blockIdx.x, c = int64_t(blockIdx.y) * kMergeCols + threadIdx.x % kMergeCols;
  int64_t st, en;
  segment(slice_ptr, k, n_slices, st, en);
  merge_run(partial, h, st, en, c, int(threadIdx.x / kMergeCols), red, out + k * h + (c < h ? c : 0));
}

// a workgroup per kManyRuns runs: a row group sums a run of up to kShort rows
// by itself, in order, four columns per lane; the workgroup shares the longer ones
constexpr int kManyRuns = kMergeGroups;
constexpr int kShort = 8;
template <typename To>
__global__ void __launch_bounds__(256)
slice_merge_many_kernel(const float* __restrict__ partial, int64_t h, const int64_t* __restrict__ slice_ptr,
                        int64_t n_slices, int64_t n_runs, To* __restrict__ out) {
  __shared__ float red[kMergeGroups][kMergeCols];
  __shared__ uint32_t longer;
  const int col = threadIdx.x % kMergeCols, g = threadIdx.x / kMergeCols;
  const int64_t first = int64_t(blockIdx.x) * kManyRuns;
  if (threadIdx.x == 0) longer = 0;
  __syncthreads();
  if (const int64_t k = first + g; k < n_runs) {
    int64_t st, en;
    segment(slice_ptr, k, n_slices, st, en);
    if (en - st > kShort) {
      if (col == 0) atomicOr(&longer, 1u << g);
    } else {
      for (int64_t c0 = col; c0 < h; c0 += 4 * kMergeCols) {
        int64_t c[4];
        float acc[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int q = 0; q < 4; ++q) c[q] = c0 + q * kMergeCols < h ? c0 + q * kMergeCols : c0;
        for (int64_t s = st; s < en; s += 2) {
          float x[2][4];
#pragma unroll
          for (int u = 0; u < 2; ++u)
#pragma unroll
            for (int q = 0; q < 4; ++q) x[u][q] = partial[(s + u < en ? s + u : s) * h + c[q]];
#pragma unroll
          for (int q = 0; q < 4; ++q) {
            acc[q] += x[0][q];
            if (s + 1 < en) acc[q] += x[1][q];
          }
        }
#pragma unroll
        for (int q = 0; q < 4; ++q)
          if (c0 + q * kMergeCols < h) from_f32(out[k * h + c[q]], acc[q]);
      }
    }
  }
  __syncthreads();
  for (uint32_t todo = longer; todo != 0; todo &= todo - 1) {  // uniform
    const int64_t k = first + __ffs(int(todo)) - 1;
    int64_t st, en;
    segment(slice_ptr, k, n_slices, st, en);
    for (int64_t c = col; c - col < h; c += kMergeCols) {
      merge_run(partial, h, st, en, c, g, red, out + k * h + (c < h ? c : 0));
      __syncthreads();  // red is the next columns'
    }
  }
}

// A workgroup per run and 32 columns for up to 2,048 runs (the class
// vocabularies, a few of whose classes own most entries: shared by eight runs'
// workgroups, the long runs of 1,458 classes at 96 positions made a training
// step's class sums 606 us instead of 436) and for long runs; past that, with at
// most 8 partial rows per run on average, 8 runs each: class sums of 20,000
// entries over 4,000 classes take 20 us instead of 27, of 100,000 over 20,000 57
// instead of 95, of 200,000 over 100,000 214 instead of 405 (a lane group per run,
// as before the merge: 24, 63, 217).
template <typename To>
int32_t slice_merge(const float* partial, int64_t h, const int64_t* slice_ptr, int64_t n_slices, int64_t n_runs,
                    To* out, hipStream_t s) {
  if (n_runs > 2048 && n_slices <= kShort * n_runs) {
    slice_merge_many_kernel<To><<<unsigned((n_runs + kManyRuns - 1) / kManyRuns), 256, 0, s>>>(
        partial, h, slice_ptr, n_slices, n_runs, out);
    return launched();
  }
  const dim3 grid{unsigned(n_runs), unsigned((h + kMergeCols - 1) / kMergeCols)};
  slice_merge_kernel<To><<<grid, 256, 0, s>>>(partial, h, slice_ptr, n_slices, out);
  return launched();
}

inline int32_t slice_merge(const float* partial, int64_t h, const int64_t* slice_ptr, int64_t n_slices,
                           int64_t n_runs, void* out, int32_t out_dtype, hipStream_t s) {
  switch (out_dtype) {
    case MANTIS_F32: return slice_merge(partial, h, slice_ptr, n_slices, n_runs, static_cast<float*>(out), s);
    case MANTIS_BF16: return slice_merge(partial, h, slice_ptr, n_slices, n_runs, static_cast<uint16_t*>(out), s);
    case MANTIS_F16: return slice_merge(partial, h, slice_ptr, n_slices, n_runs, static_cast<_Float16*>(out), s);
    default: return MANTIS_E_ARG;
  }
}

inline int64_t align256(int64_t n) { return (n + 255) / 256 * 256; }

// Workspace carve-up of the sliced class reduction: the slice tables and
// the slice partials, each 256-byte aligned.
struct SliceLayout {
  int64_t slice_ptr, slice_edge, partial, total, n_slices;
};

SliceLayout slice_layout(int64_t n_entries, int64_t n_cls, int64_t h) {
  SliceLayout L;
  L.n_slices = (n_entries + kSlice - 1) / kSlice + n_cls;  // >= sum_k ceil(len_k / kSlice)
  L.slice_ptr = 0;
  L.slice_edge = L.slice_ptr + align256((n_cls + 1) * 8);
  L.partial = L.slice_edge + align256((L.n_slices + 1) * 8);
  L.total = L.partial + align256(L.n_slices * h * 4);
  return L;
}

}  // namespace
}  // namespace mantis

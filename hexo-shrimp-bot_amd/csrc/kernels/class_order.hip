// Stable class-major order of an entry list whose keys are few (class ids):
// the class gradients' counterpart of argsort(key, stable) + gather + CSR, in
// three launches for up to 2,048 keys.
//
//   count    each wavefront counts the keys of its tile of 512 entries in LDS
//   scan     per key, the exclusive prefix over the tiles (16 keys x 64 tile
//            segments per workgroup), and the key totals
//   scatter  each workgroup scans the key totals, and each wavefront walks its
//            tile in order, 64 entries at a time: an entry's place is its
//            key's running count plus the lanes below it with the same key
//            (found by one ballot per key bit)
//
// A wavefront requests its tile's entries before it uses the first (a tile of
// 1,024 that loaded 64 at a time took a memory latency for each).
//
// Bound by latency at these sizes (10^5-10^6 entries).  The action rows of 96
// positions (622,000 entries): a comparison merge sort of 64-bit keys 200 us in
// 15 launches, these three 32 us (count 5.7, scan 13.5, scatter 12.9; with the
// tiles of 1,024: 11 + 9 + 21).
#include "common.hpp"

namespace mantis {
namespace {

constexpr int kMaxKeys = 2048;
constexpr int kTile = 512;  // entries of a wavefront
constexpr int kSteps = kTile / 64;
constexpr int kWaves = 4;

__global__ void __launch_bounds__(64 * kWaves)
class_count_kernel(const int64_t* __restrict__ key, int64_t n, int n_keys, int64_t n_tiles,
                   int32_t* __restrict__ hist, int32_t* flag) {
  __shared__ int32_t count[kWaves][kMaxKeys];
  const int lane = threadIdx.x % 64, wave = threadIdx.x / 64;
  for (int k = threadIdx.x; k < kWaves * kMaxKeys; k += 64 * kWaves) count[k / kMaxKeys][k % kMaxKeys] = 0;
  __syncthreads();
  const int64_t tile = int64_t(blockIdx.x) * kWaves + wave;
  int64_t k[kSteps];
#pragma unroll
  for (int i = 0; i < kSteps; ++i) {  // (n > 0: a grid of no tiles is not launched)
    const int64_t e = tile * kTile + i * 64 + lane;
    k[i] = key[e < n ? e : n - 1];
  }
#pragma unroll
  for (int i = 0; i < kSteps; ++i) {
    if (tile * kTile + i * 64 + lane >= n) continue;
    if (k[i] >= 0 && k[i] < n_keys) atomicAdd(&count[wave][k[i]], 1);
    else raise_flag(flag, MANTIS_FLAG_INDEX);
  }
  __syncthreads();
  if (tile < n_tiles)
    for (int k = lane; k < n_keys; k += 64) hist[tile * n_keys + k] = count[wave][k];
}

constexpr int kScanKeys = 16, kScanSegs = 64;
__global__ void __launch_bounds__(kScanKeys * kScanSegs)
class_scan_kernel(int32_t* __restrict__ hist, int n_keys, int64_t n_tiles, int32_t* __restrict__ total) {
  __shared__ int32_t part[kScanSegs][kScanKeys + 1];
  const int kk = threadIdx.x % kScanKeys, seg = threadIdx.x / kScanKeys;
  const int k = blockIdx.x * kScanKeys + kk;
  const int64_t per = (n_tiles + kScanSegs - 1) / kScanSegs;
  const int64_t t0 = seg * per, t1 = t0 + per < n_tiles ? t0 + per : n_tiles;
  int32_t sum = 0;
  if (k < n_keys) {
#pragma unroll 8
    for (int64_t t = t0; t < t1; ++t) sum += hist[t * n_keys + k];
  }
  part[seg][kk] = sum;
  __syncthreads();
  int32_t run = 0;
#pragma unroll 8
  for (int s = 0; s < seg; ++s) run += part[s][kk];
  if (k >= n_keys) return;
  if (seg == kScanSegs - 1) total[k] = run + sum;
  constexpr int kAhead = 8;  // counts read before the first of them is overwritten
  for (int64_t t = t0; t < t1; t += kAhead) {
    int32_t c[kAhead];
#pragma unroll
    for (int u = 0; u < kAhead; ++u) c[u] = hist[(t + u < t1 ? t + u : t1 - 1) * n_keys + k];
#pragma unroll
    for (int u = 0; u < kAhead; ++u) {
      if (t + u < t1) hist[(t + u) * n_keys + k] = run;
      run += c[u];
    }
  }
}

__global__ void __launch_bounds__(64 * kWaves)
class_scatter_kernel(const int64_t* __restrict__ key, const int64_t* __restrict__ col, int64_t n, int n_keys,
                     int bits, int64_t n_tiles, const int32_t* __restrict__ hist, const int32_t* __restrict__ total,
                     int64_t* __restrict__ ptr, int64_t* __restrict__ out) {
  constexpr int kPer = kMaxKeys / (64 * kWaves);  // keys per thread
  __shared__ int32_t start[kMaxKeys];
  __shared__ int32_t next[kWaves][kMaxKeys];
  __shared__ int32_t wave_sum[kWaves];
  const int lane = threadIdx.x % 64, wave = threadIdx.x / 64;
  const int64_t tile = int64_t(blockIdx.x) * kWaves + wave;
  int64_t k64[kSteps], v[kSteps];
#pragma unroll
  for (int i = 0; i < kSteps; ++i) {
    const int64_t e = tile * kTile + i * 64 + lane;
    k64[i] = e < n ? key[e] : -1;
    v[i] = e < n ? (col ? col[e] : e) : 0;
  }
  // exclusive scan of the key totals: thread t owns keys kPer t ..
  int32_t c[kPer], own = 0;
#pragma unroll
  for (int j = 0; j < kPer; ++j) {
    const int k = threadIdx.x * kPer + j;
    c[j] = k < n_keys ? total[k] : 0;
    own += c[j];
  }
  int32_t inc = own;
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    const int32_t v = __shfl_up(inc, o);
    if (lane >= o) inc += v;
  }
  if (lane == 63) wave_sum[wave] = inc;
  __syncthreads();
  int32_t run = inc - own;
  for (int w = 0; w < wave; ++w) run += wave_sum[w];
#pragma unroll
  for (int j = 0; j < kPer; ++j) {
    start[threadIdx.x * kPer + j] = run;
    run += c[j];
  }
  __syncthreads();
  if (blockIdx.x == 0) {
    for (int k = threadIdx.x; k < n_keys; k += 64 * kWaves) ptr[k] = start[k];
    if (threadIdx.x == 64 * kWaves - 1) ptr[n_keys] = run;  // the last thread's running sum: all entries
  }
  if (tile >= n_tiles) return;  // (no barrier below)
  int32_t* mine = next[wave];
  for (int k = lane; k < n_keys; k += 64) mine[k] = start[k] + hist[tile * n_keys + k];
#pragma unroll
  for (int i = 0; i < kSteps; ++i) {
    // other lanes' counts: keep the reads of this step after the writes before it
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    const bool ok = k64[i] >= 0 && k64[i] < n_keys;
    const int k = ok ? int(k64[i]) : 0;
    uint64_t same = __ballot(ok);
    for (int b = 0; b < bits; ++b) {
      const uint64_t set = __ballot((k >> b) & 1);
      same &= (k >> b) & 1 ? set : ~set;
    }
    if (ok) {
      const int below = __popcll(same & ((uint64_t(1) << lane) - 1));
      const int32_t at = mine[k] + below;
      // every lane of the key has read the count (one wavefront, LDS in order)
      if (below == 0) mine[k] = at + __popcll(same);
      out[at] = v[i];
    }
  }
}

int64_t n_tiles_of(int64_t n) { return (n + kTile - 1) / kTile; }

}  // namespace
}  // namespace mantis

using namespace mantis;

extern "C" {

int64_t mantis_class_order_workspace(int64_t n_entries, int64_t n_keys) {
  if (n_entries < 0 || n_keys <= 0 || n_keys > kMaxKeys || n_entries > 2147483647LL - kTile) return -1;
  return (n_tiles_of(n_entries) + 1) * n_keys * int64_t(sizeof(int32_t));
}

int32_t mantis_class_order(const int64_t* key, const int64_t* col, int64_t n_entries, int64_t n_keys, int64_t* ptr,
                           int64_t* out, void* workspace, int64_t workspace_bytes, int32_t* err_flag, void* stream) {
  const int64_t need = mantis_class_order_workspace(n_entries, n_keys);
  if (need < 0 || !ptr || (n_entries > 0 && (!key || !out)) || !workspace || workspace_bytes < need ||
      !aligned16(workspace))
    return MANTIS_E_ARG;
  const int64_t n_tiles = n_tiles_of(n_entries);
  int32_t* hist = static_cast<int32_t*>(workspace);
  int32_t* total = hist + n_tiles * n_keys;
  int bits = 0;
  while ((int64_t(1) << bits) < n_keys) ++bits;
  hipStream_t s = as_stream(stream);
  const unsigned grid = unsigned((n_tiles + kWaves - 1) / kWaves);
  if (grid > 0)
    class_count_kernel<<<grid, 64 * kWaves, 0, s>>>(key, n_entries, int(n_keys), n_tiles, hist, err_flag);
  class_scan_kernel<<<unsigned((n_keys + kScanKeys - 1) / kScanKeys), kScanKeys * kScanSegs, 0, s>>>(
      hist, int(n_keys), n_tiles, total);
  class_scatter_kernel<<<grid > 0 ? grid : 1, 64 * kWaves, 0, s>>>(key, col, n_entries, int(n_keys), bits, n_tiles,
                                                                 hist, total, ptr, out);
  return launched();
}

}  // extern "C"

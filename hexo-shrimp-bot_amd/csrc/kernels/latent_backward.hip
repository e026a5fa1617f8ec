// Backward of the window-latent read and broadcast for gfx950
// (window_latents.py:132-230, 503-551, 589-715): four latent rows per
// position against that position's windows, 4 heads x 32 dims.
//
//   read       latent queries over window keys and values:
//              dq (latents), dk and dv (windows)
//   broadcast  window queries over latent keys and values:
//              dq (windows), dk and dv (latents)
//
// Both are bound by the window rows, which one pass reads and writes once:
// a position's four latent rows (and the gradient sums of those rows) stay in
// registers while its windows stream by, 16 lanes per window, the next
// window's rows requested while the current one computes.  The softmax terms
// are recomputed from the forward's m and l; in the read, delta of a latent
// row is grad . out (the flash form), in the broadcast it is a window's own
// four-term sum, so neither needs a pass of its own.  A position's windows
// are split over workgroups (about kPerSplit windows each); a second launch
// adds the splits' partial sums in split order.  fp32 sums in a fixed order,
// no atomics: two calls agree bitwise.
//
// What bounds the passes is the wavefronts in flight: the broadcast's keeps four
// latent rows' keys, values and two sums (256 VGPRs, one wavefront per SIMD, TD
// 45% and VALU 38% busy), the read's half of that (174, two; TD 69%, VALU 49%).
//
// (128 positions of 40-120 stones, 169k windows, bf16: forward and backward of
// the read and the broadcast together 4,810 -> 336 us; before, each operator
// ran two passes of 1.1 ms over a materialised edge list.)
#include "common.hpp"
#include "gather.hpp"

namespace mantis {
namespace {

constexpr int kBlock = 256;
constexpr int kGroups = kBlock / kGroup;
constexpr int kRow = 128;
constexpr int kHeads = 4;
constexpr int kSlots = 4;
// windows per workgroup: enough that the latent rows and the partial sums
// (4 KB) are small beside them, few enough that one position of 1,300
// windows already fills 20 workgroups
constexpr int64_t kPerSplit = 64;
constexpr int64_t kMaxSplits = 64;

int64_t n_splits(int64_t n_pos, int64_t n_w) {
  const int64_t s = n_pos > 0 ? (n_w + n_pos * kPerSplit - 1) / (n_pos * kPerSplit) : 1;
  return s < 1 ? 1 : (s > kMaxSplits ? kMaxSplits : s);
}

struct LatArgs {
  const void* q;
  const void* k;
  const void* v;
  int64_t ldq, ldk, ldv;
  const int64_t* pos;      // (n_w,) position of each window
  const int64_t* offsets;  // (n_pos + 1,)
  const int64_t* order;    // (n_w,) windows, position-major
  int64_t n_pos, n_w;
  const float* go;   // grad of the output rows, 128 wide
  const float* out;  // the forward's output (read only)
  const float* m;
  const float* l;
  float* partial;  // (n_pos, splits, 512 or 1024)
  int32_t* mark;   // (n_w,) the order entry that wrote a window's rows
  void* dq;
  void* dk;
  void* dv;
  float scale;
  int32_t splits;
  int32_t* flag;
};

__device__ __forceinline__ float dot8(const float (&a)[8], const float (&b)[8]) {
  float d = 0.f;
#pragma unroll
  for (int i = 0; i < 8; ++i) d = fmaf(a[i], b[i], d);
  return d;
}

// the windows order[a .. b) of split `s` of position p
__device__ __forceinline__ void split_range(const LatArgs& a, int64_t p, int s, int64_t& lo, int64_t& hi) {
  int64_t st, en;
  segment(a.offsets, p, a.n_w, st, en);
  const int64_t per = (en - st + a.splits - 1) / a.splits;
  lo = st + per * s;
  lo = lo < en ? lo : en;
  hi = lo + per < en ? lo + per : en;
}

// Sum kN lane values over the workgroup's 16 groups into `to` (kN * 16 wide:
// value j, then the lane's 8 features).  Groups of a wavefront by lane swaps,
// then the four wavefronts in order.
template <int kSets>
__device__ __forceinline__ void store_partial(float (&acc)[kSets][8], float* to) {
  __shared__ float red[kBlock / 64][kSets * kRow];
  const int lane = threadIdx.x % kGroup, wave = threadIdx.x / 64;
#pragma unroll
  for (int j = 0; j < kSets; ++j)
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const float x = sum_xor32(sum_xor16(acc[j][i]));
      if ((threadIdx.x & 63) < kGroup) red[wave][j * kRow + 8 * lane + i] = x;
    }
  __syncthreads();
  for (int i = threadIdx.x; i < kSets * kRow; i += kBlock)
    to[i] = ((red[0][i] + red[1][i]) + red[2][i]) + red[3][i];
}

// ---------------------------------------------------------------- read

// a position's latent rows, this lane's 8 features and head
template <typename T>
struct ReadLatents {
  float q[kSlots][8], g[kSlots][8], mm[kSlots], inv[kSlots], delta[kSlots];
  // `entries`: the position's run of the order is not empty.  A row of such a
  // position without a positive l had a score of NaN or +-inf (its output may
  // be 0 then): delta, the sum of alpha dalpha, is NaN, and so are the row's
  // dq and its share of dk.
  __device__ __forceinline__ void load(const LatArgs& a, int64_t p, int lane, bool entries) {
    const int h = lane >> 2;
#pragma unroll
    for (int j = 0; j < kSlots; ++j) {
      const int64_t r = kSlots * p + j;
      float o[8];
      load8(static_cast<const T*>(a.q) + r * a.ldq + 8 * lane, q[j]);
      load8(a.go + r * kRow + 8 * lane, g[j]);
      load8(a.out + r * kRow + 8 * lane, o);
      delta[j] = head_sum(dot8(g[j], o));
      mm[j] = a.m[r * kHeads + h];
      const float ll = a.l[r * kHeads + h];
      inv[j] = ll > 0.f ? 1.f / ll : 0.f;
      if (entries && !(ll > 0.f)) delta[j] = __builtin_nanf("");
    }
  }
  // one window: its dk, dv, and ds per slot
  __device__ __forceinline__ void window(const LatArgs& a, const float (&k)[8], const float (&v)[8], float (&dk)[8],
                                         float (&dv)[8], float (&ds)[kSlots]) const {
#pragma unroll
    for (int i = 0; i < 8; ++i) dk[i] = dv[i] = 0.f;
#pragma unroll
    for (int j = 0; j < kSlots; ++j) {
      const float sd = head_sum(dot8(q[j], k)), dd = head_sum(dot8(g[j], v));
      const float al = inv[j] > 0.f ? expf(sd * a.scale - mm[j]) * inv[j] : 0.f;
      ds[j] = al * (dd - delta[j]);
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        dv[i] = fmaf(al, g[j][i], dv[i]);
        dk[i] = fmaf(ds[j] * a.scale, q[j][i], dk[i]);
      }
    }
  }
};

template <typename T>
__global__ void __launch_bounds__(kBlock)
latent_read_bwd_kernel(LatArgs a) {
  const int64_t p = blockIdx.x / a.splits;
  const int lane = threadIdx.x % kGroup;
  ReadLatents<T> L;
  L.load(a, p, lane, true);  // (used for the windows of the run only)
  int64_t lo, hi;
  split_range(a, p, int(blockIdx.x % a.splits), lo, hi);
  float acc[kSlots][8];
#pragma unroll
  for (int j = 0; j < kSlots; ++j)
#pragma unroll
    for (int i = 0; i < 8; ++i) acc[j][i] = 0.f;
  const T* kb = static_cast<const T*>(a.k);
  const T* vb = static_cast<const T*>(a.v);
  auto entry = [&](int64_t i) { return i < hi ? a.order[i] : int64_t(-1); };
  auto clamped = [&](int64_t w) { return w >= 0 && w < a.n_w ? w : int64_t(0); };
  int64_t i = lo + threadIdx.x / kGroup;
  if (i < hi) {  // (then n_w > 0: row 0 exists)
    int64_t w0 = entry(i), w1 = entry(i + kGroups);
    Chunk8<T> k0, v0, k1, v1;
    k0.load(kb + clamped(w0) * a.ldk + 8 * lane);
    v0.load(vb + clamped(w0) * a.ldv + 8 * lane);
    int64_t p0 = a.pos[clamped(w0)], p1;
    for (; i < hi; i += kGroups) {
      const int64_t w2 = entry(i + 2 * kGroups);
      k1.load(kb + clamped(w1) * a.ldk + 8 * lane);
      v1.load(vb + clamped(w1) * a.ldv + 8 * lane);
      p1 = a.pos[clamped(w1)];
      if (w0 >= 0 && w0 < a.n_w) {  // uniform over the 16 lanes
        float k[8], v[8], dk[8], dv[8], ds[kSlots];
#pragma unroll
        for (int e = 0; e < 8; ++e) k[e] = k0[e], v[e] = v0[e];
        L.window(a, k, v, dk, dv, ds);
#pragma unroll
        for (int j = 0; j < kSlots; ++j)
#pragma unroll
          for (int e = 0; e < 8; ++e) acc[j][e] = fmaf(ds[j], k[e], acc[j][e]);
        if (p0 == p) {
          store8(static_cast<T*>(a.dk) + w0 * kRow + 8 * lane, dk);
          store8(static_cast<T*>(a.dv) + w0 * kRow + 8 * lane, dv);
          if (lane == 0) a.mark[w0] = int32_t(i);
        }
      } else if (lane == 0) {
        raise_flag(a.flag, MANTIS_FLAG_INDEX);
      }
      w0 = w1, w1 = w2, k0 = k1, v0 = v1, p0 = p1;
    }
  }
  store_partial<kSlots>(acc, a.partial + int64_t(blockIdx.x) * kSlots * kRow);
}

// ---------------------------------------------------------------- broadcast

template <typename T>
struct CastLatents {
  float k[kSlots][8], v[kSlots][8];
  __device__ __forceinline__ void load(const LatArgs& a, int64_t p, int lane) {
#pragma unroll
    for (int j = 0; j < kSlots; ++j) {
      load8(static_cast<const T*>(a.k) + (kSlots * p + j) * a.ldk + 8 * lane, k[j]);
      load8(static_cast<const T*>(a.v) + (kSlots * p + j) * a.ldv + 8 * lane, v[j]);
    }
  }
  // alpha and dalpha of one window, and its delta: NaN, as its terms are, for
  // a window without a positive l (its scores hold a NaN or +-inf)
  __device__ __forceinline__ float terms(const LatArgs& a, const float (&q)[8], const float (&g)[8], float mm,
                                         float ll, float (&al)[kSlots], float (&dd)[kSlots]) const {
    const float inv = ll > 0.f ? 1.f / ll : 0.f;
    float delta = 0.f;
#pragma unroll
    for (int j = 0; j < kSlots; ++j) {
      const float sd = head_sum(dot8(q, k[j]));
      dd[j] = head_sum(dot8(g, v[j]));
      al[j] = inv > 0.f ? expf(sd * a.scale - mm) * inv : 0.f;
      delta = fmaf(al[j], dd[j], delta);
    }
    return inv > 0.f ? delta : __builtin_nanf("");
  }
  __device__ __forceinline__ void store_dq(const LatArgs& a, int64_t w, int lane, const float (&ds)[kSlots]) const {
    float d[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) d[i] = 0.f;
#pragma unroll
    for (int j = 0; j < kSlots; ++j)
#pragma unroll
      for (int i = 0; i < 8; ++i) d[i] = fmaf(ds[j] * a.scale, k[j][i], d[i]);
    store8(static_cast<T*>(a.dq) + w * kRow + 8 * lane, d);
  }
};

template <typename T>
__global__ void __launch_bounds__(kBlock)
latent_broadcast_bwd_kernel(LatArgs a) {
  const int64_t p = blockIdx.x / a.splits;
  const int lane = threadIdx.x % kGroup, h = lane >> 2;
  CastLatents<T> L;
  L.load(a, p, lane);
  int64_t lo, hi;
  split_range(a, p, int(blockIdx.x % a.splits), lo, hi);
  float acc[2 * kSlots][8];  // dk, dv of the four latents
#pragma unroll
  for (int j = 0; j < 2 * kSlots; ++j)
#pragma unroll
    for (int i = 0; i < 8; ++i) acc[j][i] = 0.f;
  const T* qb = static_cast<const T*>(a.q);
  auto entry = [&](int64_t i) { return i < hi ? a.order[i] : int64_t(-1); };
  auto clamped = [&](int64_t w) { return w >= 0 && w < a.n_w ? w : int64_t(0); };
  int64_t i = lo + threadIdx.x / kGroup;
  if (i < hi) {
    int64_t w0 = entry(i), w1 = entry(i + kGroups);
    Chunk8<T> q0, q1;
    Chunk8<float> g0, g1;
    float m0, l0, m1, l1;
    int64_t p0, p1;
    auto fetch = [&](int64_t w, Chunk8<T>& q, Chunk8<float>& g, float& m, float& l, int64_t& pw) {
      const int64_t r = clamped(w);
      q.load(qb + r * a.ldq + 8 * lane);
      g.load(a.go + r * kRow + 8 * lane);
      m = a.m[r * kHeads + h];
      l = a.l[r * kHeads + h];
      pw = a.pos[r];
    };
    fetch(w0, q0, g0, m0, l0, p0);
    for (; i < hi; i += kGroups) {
      const int64_t w2 = entry(i + 2 * kGroups);
      fetch(w1, q1, g1, m1, l1, p1);
      if (w0 >= 0 && w0 < a.n_w) {
        float q[8], g[8], al[kSlots], dd[kSlots], ds[kSlots];
#pragma unroll
        for (int e = 0; e < 8; ++e) q[e] = q0[e], g[e] = g0[e];
        float delta = L.terms(a, q, g, m0, l0, al, dd);
        if (p0 != p) {
          // the order names a window of another position: its delta is over
          // its own position's latents
          delta = 0.f;
          if (p0 >= 0 && p0 < a.n_pos) {
            CastLatents<T> own;
            own.load(a, p0, lane);
            float al2[kSlots], dd2[kSlots];
            delta = own.terms(a, q, g, m0, l0, al2, dd2);
          }
        }
#pragma unroll
        for (int j = 0; j < kSlots; ++j) {
          ds[j] = al[j] * (dd[j] - delta);
#pragma unroll
          for (int e = 0; e < 8; ++e) {
            acc[j][e] = fmaf(ds[j], q[e], acc[j][e]);
            acc[kSlots + j][e] = fmaf(al[j], g[e], acc[kSlots + j][e]);
          }
        }
        if (p0 == p) {
          L.store_dq(a, w0, lane, ds);
          if (lane == 0) a.mark[w0] = int32_t(i);
        }
      } else if (lane == 0) {
        raise_flag(a.flag, MANTIS_FLAG_INDEX);
      }
      w0 = w1, w1 = w2, q0 = q1, g0 = g1, m0 = m1, l0 = l1, p0 = p1;
    }
  }
  store_partial<2 * kSlots>(acc, a.partial + int64_t(blockIdx.x) * 2 * kSlots * kRow);
}

// ---------------------------------------------------------------- finish

// Blocks [0, n_pos * kParts): the splits' partial sums of a position's latent
// rows, a column per thread and kAhead splits in flight, added in split order
// (one workgroup per position, a split after the other, was 21 and 11.6 us of
// a launch at 128 positions of 21 splits).
// The others: 256 windows each, which the first launch has written if the
// layout is window_latent_layout's; a window that its position's run of the
// order does not name (mark holds no entry of that run naming it) gets its
// rows here, from its own position.
template <bool kRead>
constexpr int kPartialWidth = (kRead ? 1 : 2) * kSlots * kRow;
template <bool kRead>
constexpr int kParts = kPartialWidth<kRead> / kBlock;
constexpr int kAhead = 8;
template <typename T, bool kRead>
__global__ void __launch_bounds__(kBlock)
latent_bwd_finish_kernel(LatArgs a) {
  constexpr int kWidth = kPartialWidth<kRead>;
  const int64_t n_sums = a.n_pos * kParts<kRead>;
  if (int64_t(blockIdx.x) < n_sums) {
    const int64_t p = blockIdx.x / kParts<kRead>;
    const int c = int(blockIdx.x % kParts<kRead>) * kBlock + threadIdx.x;
    const float* from = a.partial + p * a.splits * kWidth + c;
    float x = 0.f;
    for (int s = 0; s < a.splits; s += kAhead) {
      float y[kAhead];
#pragma unroll
      for (int u = 0; u < kAhead; ++u) y[u] = from[int64_t(s + u < a.splits ? s + u : a.splits - 1) * kWidth];
#pragma unroll
      for (int u = 0; u < kAhead; ++u)
        if (s + u < a.splits) x += y[u];
    }
    // dq or dk: times the score scale; dv: as summed
    const bool second = c >= kSlots * kRow;
    T* to = static_cast<T*>(kRead ? a.dq : second ? a.dv : a.dk);
    from_f32(to[p * kSlots * kRow + c % (kSlots * kRow)], second ? x : x * a.scale);
    return;
  }
  const int lane = threadIdx.x % kGroup;
  const int64_t first = (int64_t(blockIdx.x) - n_sums) * kBlock + threadIdx.x / kGroup * kGroup;
  const int64_t mine = first + lane;
  bool miss = false;
  if (mine < a.n_w) {
    const int64_t p = a.pos[mine];
    miss = true;
    if (p >= 0 && p < a.n_pos) {
      int64_t st, en;
      segment(a.offsets, p, a.n_w, st, en);
      const int64_t i = a.mark[mine];
      miss = !(i >= st && i < en && a.order[i] == mine);
    } else {
      raise_flag(a.flag, MANTIS_FLAG_INDEX);
    }
  }
  const uint64_t all = __ballot(miss);
  uint32_t todo = uint32_t(all >> (threadIdx.x & 48)) & 0xffffu;  // this group's 16 windows
  while (todo) {
    const int64_t w = first + __ffs(int(todo)) - 1;
    todo &= todo - 1;
    const int64_t p = a.pos[w];
    const bool ok = p >= 0 && p < a.n_pos;
    float zero[8] = {0, 0, 0, 0, 0, 0, 0, 0};
    if constexpr (kRead) {
      float k[8], v[8], dk[8], dv[8], ds[kSlots];
      if (ok) {
        ReadLatents<T> L;
        int64_t st, en;
        segment(a.offsets, p, a.n_w, st, en);
        L.load(a, p, lane, en > st);
        load8(static_cast<const T*>(a.k) + w * a.ldk + 8 * lane, k);
        load8(static_cast<const T*>(a.v) + w * a.ldv + 8 * lane, v);
        L.window(a, k, v, dk, dv, ds);
      }
      store8(static_cast<T*>(a.dk) + w * kRow + 8 * lane, ok ? dk : zero);
      store8(static_cast<T*>(a.dv) + w * kRow + 8 * lane, ok ? dv : zero);
    } else {
      if (!ok) {
        store8(static_cast<T*>(a.dq) + w * kRow + 8 * lane, zero);
        continue;
      }
      float q[8], g[8], al[kSlots], dd[kSlots], ds[kSlots];
      CastLatents<T> L;
      L.load(a, p, lane);
      load8(static_cast<const T*>(a.q) + w * a.ldq + 8 * lane, q);
      load8(a.go + w * kRow + 8 * lane, g);
      const float delta = L.terms(a, q, g, a.m[w * kHeads + (lane >> 2)], a.l[w * kHeads + (lane >> 2)], al, dd);
#pragma unroll
      for (int j = 0; j < kSlots; ++j) ds[j] = al[j] * (dd[j] - delta);
      L.store_dq(a, w, lane, ds);
    }
  }
}

int64_t partial_bytes(int64_t n_pos, int64_t n_w) {
  return n_pos * n_splits(n_pos, n_w) * 2 * kSlots * kRow * int64_t(sizeof(float));
}

template <bool kRead>
int32_t backward(LatArgs a, int32_t dtype, void* workspace, int64_t workspace_bytes, void* stream) {
  if (a.n_pos < 0 || a.n_w < 0 || a.n_w > 2147483647LL - kBlock) return MANTIS_E_ARG;
  if (a.n_pos == 0 && a.n_w == 0) return MANTIS_OK;
  const int64_t lat = a.n_pos, win = a.n_w;
  if ((lat > 0 && (!a.offsets || !a.partial)) || (win > 0 && (!a.order || !a.pos))) return MANTIS_E_ARG;
  const int64_t nq = kRead ? lat : win, nk = kRead ? win : lat;
  if (nq > 0 && (!a.q || !a.go || !a.m || !a.l || !a.dq || (kRead && !a.out))) return MANTIS_E_ARG;
  if (nk > 0 && (!a.k || !a.v || !a.dk || !a.dv)) return MANTIS_E_ARG;
  for (int64_t ld : {a.ldq, a.ldk, a.ldv})
    if (ld < kRow || ld % 8) return MANTIS_E_ARG;
  for (const void* p : {a.q, a.k, a.v, static_cast<const void*>(a.go), static_cast<const void*>(a.out),
                        static_cast<const void*>(a.dq), static_cast<const void*>(a.dk),
                        static_cast<const void*>(a.dv)})
    if (p && !aligned16(p)) return MANTIS_E_ARG;
  if (!workspace || !aligned16(workspace) || workspace_bytes < partial_bytes(lat, win) + win * 4) return MANTIS_E_ARG;
  a.splits = int32_t(n_splits(lat, win));
  const int64_t grid = lat * a.splits, finish = lat * kParts<kRead> + (win + kBlock - 1) / kBlock;
  if (grid > 2147483647LL || finish > 2147483647LL) return MANTIS_E_ARG;
  a.mark = reinterpret_cast<int32_t*>(static_cast<char*>(workspace) + partial_bytes(lat, win));
  a.scale = 0.17677669529663687f;  // 1 / sqrt(32)
  hipStream_t s = as_stream(stream);
  auto run = [&](auto t) {
    using T = decltype(t);
    if (grid > 0) {
      if constexpr (kRead) latent_read_bwd_kernel<T><<<unsigned(grid), kBlock, 0, s>>>(a);
      else latent_broadcast_bwd_kernel<T><<<unsigned(grid), kBlock, 0, s>>>(a);
    }
    latent_bwd_finish_kernel<T, kRead><<<unsigned(finish), kBlock, 0, s>>>(a);
  };
  switch (dtype) {
    case MANTIS_F32: run(float{}); break;
    case MANTIS_BF16: run(uint16_t{}); break;
    case MANTIS_F16: run(_Float16{}); break;
    default: return MANTIS_E_ARG;
  }
  return launched();
}

}  // namespace
}  // namespace mantis

using namespace mantis;

extern "C" {

int64_t mantis_latent_backward_workspace(int64_t n_pos, int64_t n_w) {
  if (n_pos < 0 || n_w < 0) return -1;
  return partial_bytes(n_pos, n_w) + n_w * 4;
}

int32_t mantis_latent_read_backward(const void* q, const void* k, const void* v, int32_t dtype, int64_t ldq,
                                    int64_t ldk, int64_t ldv, const int64_t* window_pos, const int64_t* offsets,
                                    const int64_t* order, int64_t n_pos, int64_t n_w, const float* grad_out,
                                    const float* out, const float* m, const float* l, void* workspace,
                                    int64_t workspace_bytes, void* dq, void* dk, void* dv, int32_t* err_flag,
                                    void* stream) {
  return backward<true>({q, k, v, ldq, ldk, ldv, window_pos, offsets, order, n_pos, n_w, grad_out, out, m, l,
                         static_cast<float*>(workspace), nullptr, dq, dk, dv, 0.f, 1, err_flag},
                        dtype, workspace, workspace_bytes, stream);
}

int32_t mantis_latent_broadcast_backward(const void* q, const void* k, const void* v, int32_t dtype, int64_t ldq,
                                         int64_t ldk, int64_t ldv, const int64_t* window_pos, const int64_t* offsets,
                                         const int64_t* order, int64_t n_pos, int64_t n_w, const float* grad_out,
                                         const float* m, const float* l, void* workspace, int64_t workspace_bytes,
                                         void* dq, void* dk, void* dv, int32_t* err_flag, void* stream) {
  return backward<false>({q, k, v, ldq, ldk, ldv, window_pos, offsets, order, n_pos, n_w, grad_out, nullptr, m, l,
                          static_cast<float*>(workspace), nullptr, dq, dk, dv, 0.f, 1, err_flag},
                         dtype, workspace, workspace_bytes, stream);
}

}  // extern "C"

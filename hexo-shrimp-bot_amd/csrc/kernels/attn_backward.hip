// Backward kernels for gfx950 of the segment-attention and row-encoder
// operators (the reference's register_autograd pairs):
//
//  * typed segment attention (cell_attention / cell_attention_plain,
//    python/mantisnet/mantisnet/cell_latents.py:570-621, 680-797).  With
//      score_e = scale q[qid_e] . k[src_e] + bias[cls_e]
//      alpha_e = exp(score_e - m[qid_e]) / l[qid_e]        (the forward's softmax)
//      dalpha_e = go[qid_e] . (v[src_e] + vcls[cls_e])
//      delta_q = sum_e alpha_e dalpha_e,   dscore_e = alpha_e (dalpha_e - delta_q)
//    the gradients are dq = scale sum_e dscore_e k[src_e],
//    dk = scale sum_e dscore_e q[qid_e], dv = sum_e alpha_e go[qid_e],
//    dbias[cls] = sum_e dscore_e and dvcls[cls] = sum_e alpha_e go[qid_e].
//    A query-major pass forms delta, dq and the per-edge (alpha, dalpha); a
//    source-major pass recomputes each edge's score for dk and dv; the class
//    sums are sliced reductions over the class-major edge list.
//  * the action-row encoder (row_encoder.py:115-413): with
//    mask_e = pre[window_e] + table[class_e] > 0 the gradients are
//    dpre[w] = sum_e mask_e go[cell_e] over the window's entries and
//    dtable[c] = sum_e mask_e go[cell_e] over the class's entries.
//
// Geometry: 16 lanes per row of 4 heads x 32 (a lane owns 8 consecutive
// features, a head is 4 adjacent lanes), the entries of a row loaded 16 at a
// time, every sum in fp32 in a fixed order: no atomics, and two calls agree
// bitwise.
#include "common.hpp"
#include "gather.hpp"
#include "slices.hpp"

#include <type_traits>

namespace mantis {
namespace {

constexpr int kBlock = 256;
constexpr int kGroupsPerBlock = kBlock / kGroup;
constexpr int kRow = 128;
constexpr int kHeads = 4;

inline unsigned grid_rows(int64_t rows) { return unsigned((rows + kGroupsPerBlock - 1) / kGroupsPerBlock); }

struct AttnBwd {
  const void* q;
  const void* k;
  const void* v;
  int64_t ldq, ldk, ldv;
  int64_t n_q, n_k;
  const float* bias;  // (4, n_classes) or null
  int64_t n_classes;
  const void* vcls;  // (n_classes, 128) or null
  const float* go;   // (n_q, ldgo) fp32
  int64_t ldgo;
  const float* m;  // (n_q, 4)
  const float* l;  // (n_q, 4)
  float* delta;    // (n_q, 4)
  float4* stats;   // (n_q, 4): m, 1 / l (0 for a row without entries), delta
  float scale;
  int32_t* flag;
};

// x, or zeros: a row that is not to count must not bring its infinities in
template <typename T>
__device__ __forceinline__ void keep(Chunk8<T>& x, bool ok) {
  if constexpr (std::is_same_v<T, float>) {
#pragma unroll
    for (int i = 0; i < 8; ++i) x.f[i] = ok ? x.f[i] : 0.f;
  } else {
    x.u.x = ok ? x.u.x : 0u, x.u.y = ok ? x.u.y : 0u, x.u.z = ok ? x.u.z : 0u, x.u.w = ok ? x.u.w : 0u;
  }
}

// Query-major pass: 16 lanes per query row; up to 16 of its entries are loaded
// at once, one per lane, and shared by shuffles, so the rows of kB entries are
// in flight together and their score chains (two head sums and an exponential)
// run side by side.  Bound by the gathered rows' path (TD 75-88% busy, half of it
// stalled on L1 misses, VALU 52-57%) and the chain pointers -> indices -> rows:
// two entries per step, so that four wavefronts fit a SIMD, three with fp32 class
// values (64 positions, bf16, 1,075,000 / 416,000 / 416,000 entries: 138 / 112 / 43
// us; four entries and a branch per entry 144 / 114 / 42; four side by side,
// three wavefronts, 143 / 113 / 51; without the q and gradient rows of queries
// that have no entry 144 / 114 / 43).  With alpha_e, alpha and dalpha of every
// entry are kept for the class sums; with finish the lane that wrote them
// turns dalpha into dscore (callers without qid, whose class pass cannot look
// delta up).
template <typename T, typename Tv, bool kVcls>
__global__ void __launch_bounds__(kBlock)
attn_bwd_q_kernel(AttnBwd a, const int64_t* __restrict__ seg_ptr, const int64_t* __restrict__ src,
                  const int64_t* __restrict__ cls, int64_t n_entries, T* __restrict__ dq,
                  float* __restrict__ alpha_e, float* __restrict__ dalpha_e, bool finish) {
  constexpr int kB = 2;
  const int64_t row = int64_t(blockIdx.x) * kGroupsPerBlock + threadIdx.x / kGroup;
  const int lane = threadIdx.x % kGroup;
  if (row >= a.n_q) return;
  const int h = lane >> 2;
  const int64_t c0 = 8 * lane;
  const T* kb = static_cast<const T*>(a.k) + c0;
  const T* vb = static_cast<const T*>(a.v) + c0;
  const Tv* cb = static_cast<const Tv*>(a.vcls) + c0;
  int64_t st, en;
  segment(seg_ptr, row, n_entries, st, en);
  float qv[8], gv[8];
  load8(static_cast<const T*>(a.q) + row * a.ldq + c0, qv);
  load8(a.go + row * a.ldgo + c0, gv);
  const float mm = a.m[row * kHeads + h], ll = a.l[row * kHeads + h];
  const float inv = ll > 0.f ? 1.f / ll : 0.f;
  const float* bias = a.bias + h * a.n_classes;  // (read only if a.bias)
  float A[8] = {0, 0, 0, 0, 0, 0, 0, 0}, B[8] = {0, 0, 0, 0, 0, 0, 0, 0};
  float delta = 0.f;
  for (int64_t base = st; base < en; base += kGroup) {
    const int cnt = int(en - base < kGroup ? en - base : kGroup);
    const int64_t mine = base + (lane < cnt ? lane : cnt - 1);
    const int64_t s = src[mine], c = cls ? cls[mine] : 0;
    const bool good = s >= 0 && s < a.n_k && c >= 0 && (!cls || c < a.n_classes);
    if (!good && lane < cnt) raise_flag(a.flag, MANTIS_FLAG_INDEX);
    const int32_t c_in = good ? int32_t(c) : -1;
    // the entry's row offsets once, by its lane: 64-bit products are 16 cycles each
    const int64_t k_at = good ? s * a.ldk : 0, v_at = good ? s * a.ldv : 0;
    if (a.n_k <= 0) {  // no row to read: every entry is flagged
      if (alpha_e && (lane & 3) == 0)
        for (int64_t e = base; e < base + cnt; ++e) alpha_e[e * kHeads + h] = dalpha_e[e * kHeads + h] = 0.f;
      continue;
    }
    for (int j = 0; j < cnt; j += kB) {
      Chunk8<T> xk[kB], xv[kB];
      Chunk8<Tv> xc[kB];
      float bs[kB], sd[kB], dd[kB];
      bool ok[kB];
#pragma unroll
      for (int u = 0; u < kB; ++u) {  // (an entry that is not ok reads row 0)
        const int from = j + u < cnt ? j + u : cnt - 1;
        const int32_t cu = __shfl(c_in, from, kGroup);
        ok[u] = cu >= 0 && j + u < cnt;
        xk[u].load(kb + __shfl(k_at, from, kGroup));
        xv[u].load(vb + __shfl(v_at, from, kGroup));
        const uint32_t co = cu < 0 ? 0u : uint32_t(cu);
        if constexpr (kVcls) xc[u].load(cb + int64_t(co) * kRow);
        bs[u] = a.bias ? bias[co] : 0.f;
      }
      // without a branch between them the entries' chains run side by side
#pragma unroll
      for (int u = 0; u < kB; ++u) {
        sd[u] = dd[u] = 0.f;
        keep(xk[u], ok[u]);
#pragma unroll
        for (int i = 0; i < 8; ++i) {
          float vv = xv[u][i];
          if constexpr (kVcls) vv += xc[u][i];
          sd[u] = fmaf(qv[i], xk[u][i], sd[u]);
          dd[u] = fmaf(gv[i], vv, dd[u]);
        }
      }
#pragma unroll
      for (int u = 0; u < kB; ++u) {
        sd[u] = head_sum(sd[u]);
        dd[u] = head_sum(dd[u]);
      }
#pragma unroll
      for (int u = 0; u < kB; ++u) {
        const float al = ok[u] ? expf(sd[u] * a.scale + bs[u] - mm) * inv : 0.f;
        const float da = ok[u] ? dd[u] : 0.f, ad = al * da;
        delta = fmaf(al, da, delta);
#pragma unroll
        for (int i = 0; i < 8; ++i) {
          A[i] = fmaf(ad, xk[u][i], A[i]);
          B[i] = fmaf(al, xk[u][i], B[i]);
        }
        if (alpha_e && (lane & 3) == 0 && j + u < cnt) {
          const int64_t e = base + j + u;
          alpha_e[e * kHeads + h] = al;
          dalpha_e[e * kHeads + h] = da;
        }
      }
    }
  }
  float d[8];
#pragma unroll
  for (int i = 0; i < 8; ++i) d[i] = a.scale * (A[i] - delta * B[i]);
  store8(dq + row * kRow + c0, d);
  if ((lane & 3) == 0) {
    // (apart too: the class pass reads 16 bytes of it per entry, not 64)
    a.delta[row * kHeads + h] = delta;
    a.stats[row * kHeads + h] = make_float4(mm, inv, delta, 0.f);
    // this lane wrote these entries above: dscore = alpha (dalpha - delta)
    if (finish)
      for (int64_t e = st; e < en; ++e)
        dalpha_e[e * kHeads + h] = alpha_e[e * kHeads + h] * (dalpha_e[e * kHeads + h] - delta);
  }
}

// Source-major pass: kG lane groups per source row, each taking every kG-th
// chunk of 16 entries, their sums added in group order.  One group for short
// runs (windows and cells: about five entries); a stone's run of 200 radius
// entries left 5,000 groups each walking its own chain, a quarter of a
// launch's lanes, so long runs get 4 groups (a wavefront) or 16 (a workgroup).
// The query pass leaves m, 1 / l and delta of a query's head side by side: one
// 16-byte load per entry instead of three and no division (64 positions, bf16:
// 118.6 / 54.8 -> 113.3 / 51 us; 80 for the pass without class values, as before).
template <typename T, typename Tv, bool kVcls, int kG>
__global__ void __launch_bounds__(kBlock)
attn_bwd_kv_kernel(AttnBwd a, const int64_t* __restrict__ sseg_ptr, const int64_t* __restrict__ sqid,
                   const int64_t* __restrict__ scls, int64_t n_entries, T* __restrict__ dk, T* __restrict__ dv) {
  static_assert(kG == 1 || kG == 4 || kG == kGroupsPerBlock);
  constexpr int kB = 2;
  const int group = threadIdx.x / kGroup;
  const int64_t row = int64_t(blockIdx.x) * (kGroupsPerBlock / kG) + group / kG;
  const int lane = threadIdx.x % kGroup;
  if (row >= a.n_k) return;  // uniform over the groups of a row
  const int h = lane >> 2;
  const int64_t c0 = 8 * lane;
  const T* qb = static_cast<const T*>(a.q) + c0;
  const float* gb = a.go + c0;
  const Tv* cb = static_cast<const Tv*>(a.vcls) + c0;
  int64_t st, en;
  segment(sseg_ptr, row, n_entries, st, en);
  float kv[8], vv[8];
  load8(static_cast<const T*>(a.k) + row * a.ldk + c0, kv);
  load8(static_cast<const T*>(a.v) + row * a.ldv + c0, vv);
  const float* bias = a.bias + h * a.n_classes;  // (read only if a.bias)
  float gk[8] = {0, 0, 0, 0, 0, 0, 0, 0}, gvv[8] = {0, 0, 0, 0, 0, 0, 0, 0};
  for (int64_t base = st + int64_t(group % kG) * kGroup; base < en; base += kG * kGroup) {
    const int cnt = int(en - base < kGroup ? en - base : kGroup);
    const int64_t mine = base + (lane < cnt ? lane : cnt - 1);
    const int64_t qi = sqid[mine], c = scls ? scls[mine] : 0;
    const bool good = qi >= 0 && qi < a.n_q && c >= 0 && (!scls || c < a.n_classes);
    if (!good && lane < cnt) raise_flag(a.flag, MANTIS_FLAG_INDEX);
    const int32_t c_in = good ? int32_t(c) : -1;
    const int64_t q_in = good ? qi : 0, q_at = q_in * a.ldq, g_at = q_in * a.ldgo;
    if (a.n_q <= 0) continue;  // no row to read: every entry is flagged
    for (int j = 0; j < cnt; j += kB) {
      Chunk8<T> xq[kB];
      Chunk8<float> xg[kB];
      Chunk8<Tv> xc[kB];
      float4 st4[kB];
      float bs[kB], sd[kB], dd[kB];
      bool ok[kB];
#pragma unroll
      for (int u = 0; u < kB; ++u) {  // (an entry that is not ok reads row 0)
        const int from = j + u < cnt ? j + u : cnt - 1;
        const int32_t cu = __shfl(c_in, from, kGroup);
        ok[u] = cu >= 0 && j + u < cnt;
        xq[u].load(qb + __shfl(q_at, from, kGroup));
        xg[u].load(gb + __shfl(g_at, from, kGroup));
        st4[u] = a.stats[__shfl(q_in, from, kGroup) * kHeads + h];
        const uint32_t co = cu < 0 ? 0u : uint32_t(cu);
        if constexpr (kVcls) xc[u].load(cb + int64_t(co) * kRow);
        bs[u] = a.bias ? bias[co] : 0.f;
      }
#pragma unroll
      for (int u = 0; u < kB; ++u) {
        sd[u] = dd[u] = 0.f;
        keep(xq[u], ok[u]);
        keep(xg[u], ok[u]);
#pragma unroll
        for (int i = 0; i < 8; ++i) {
          float ve = vv[i];
          if constexpr (kVcls) ve += xc[u][i];
          sd[u] = fmaf(xq[u][i], kv[i], sd[u]);
          dd[u] = fmaf(xg[u][i], ve, dd[u]);
        }
      }
#pragma unroll
      for (int u = 0; u < kB; ++u) {
        sd[u] = head_sum(sd[u]);
        dd[u] = head_sum(dd[u]);
      }
#pragma unroll
      for (int u = 0; u < kB; ++u) {
        const float al = ok[u] && st4[u].y > 0.f ? expf(sd[u] * a.scale + bs[u] - st4[u].x) * st4[u].y : 0.f;
        const float ds = ok[u] ? al * (dd[u] - st4[u].z) * a.scale : 0.f;
#pragma unroll
        for (int i = 0; i < 8; ++i) {
          gk[i] = fmaf(ds, xq[u][i], gk[i]);
          gvv[i] = fmaf(al, xg[u][i], gvv[i]);
        }
      }
    }
  }
  if constexpr (kG > 1) {
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      gk[i] = sum_xor32(sum_xor16(gk[i]));
      gvv[i] = sum_xor32(sum_xor16(gvv[i]));
    }
  }
  if constexpr (kG == kGroupsPerBlock) {  // one row per workgroup: the wavefronts in order
    __shared__ float red[kBlock / 64][2][kRow];
    if ((threadIdx.x & 63) < kGroup)
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        red[threadIdx.x / 64][0][c0 + i] = gk[i];
        red[threadIdx.x / 64][1][c0 + i] = gvv[i];
      }
    __syncthreads();
    if (threadIdx.x < kGroup)
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        gk[i] = ((red[0][0][c0 + i] + red[1][0][c0 + i]) + red[2][0][c0 + i]) + red[3][0][c0 + i];
        gvv[i] = ((red[0][1][c0 + i] + red[1][1][c0 + i]) + red[2][1][c0 + i]) + red[3][1][c0 + i];
      }
  }
  if (group % kG == 0) {
    store8(dk + row * kRow + c0, gk);
    store8(dv + row * kRow + c0, gvv);
  }
}

// Class slices: partial4[s] = sum over the class-major entries j of slice s of
// dscore[E], E = cedge[j] (a query-major edge), and with kV partial[s] = sum
// of alpha[E, head] * go[qid[E]].  dscore = alpha (dalpha - delta[qid]), or
// with qid null dalpha_e already holds it.  16 entries per index load; the gradient
// rows of kLook entries in flight from clamped indices (a load under a
// condition is waited for before the next), the scores one entry per lane.
// Bound by the latency of the gathered gradient rows (TD 67-80% busy, most of it
// stalled on L1 misses, 10-16% L2 hits, VALU 8%): with eight rows in
// flight 147 and 53.5 us for 1,075,000 and 416,000 entries (four conditional
// ones: 156 and 55.6), 22 and 19 for 193,000 and 74,000 (33 and 31).
template <bool kV>
__global__ void __launch_bounds__(kBlock)
class_slice_kernel(const float* __restrict__ alpha_e, const float* __restrict__ dalpha_e,
                   const float* __restrict__ delta, const float* __restrict__ go, int64_t ldgo, const int64_t* __restrict__ qid, int64_t n_q,
                   const int64_t* __restrict__ cedge, int64_t n_edges, const int64_t* __restrict__ slice_edge,
                   int64_t n_slices, float* __restrict__ partial, float* __restrict__ partial4, int32_t* flag) {
  constexpr int kLook = 8;
  const int64_t s = int64_t(blockIdx.x) * kGroupsPerBlock + threadIdx.x / kGroup;
  const int lane = threadIdx.x % kGroup;
  if (s >= n_slices) return;
  const int h = lane >> 2;
  const int64_t c0 = 8 * lane;
  int64_t st, en;
  segment(slice_edge, s, n_edges, st, en);
  float acc[8] = {0, 0, 0, 0, 0, 0, 0, 0};
  float4 d4 = make_float4(0.f, 0.f, 0.f, 0.f);
  for (int64_t base = st; base < en; base += kGroup) {
    const int cnt = int(en - base < kGroup ? en - base : kGroup);
    const int64_t E = cedge[base + (lane < cnt ? lane : cnt - 1)];
    bool ok = E >= 0 && E < n_edges;
    int64_t qi = 0;
    if (qid) {
      qi = ok ? qid[E] : -1;
      ok = qi >= 0 && qi < n_q;
    }
    if (!ok && lane < cnt) raise_flag(flag, MANTIS_FLAG_INDEX);
    if (ok && lane < cnt) {
      float4 d = *reinterpret_cast<const float4*>(dalpha_e + E * kHeads);
      if (qid) {
        const float4 al = *reinterpret_cast<const float4*>(alpha_e + E * kHeads);
        const float4 dl = *reinterpret_cast<const float4*>(delta + qi * kHeads);
        d.x = al.x * (d.x - dl.x), d.y = al.y * (d.y - dl.y);
        d.z = al.z * (d.z - dl.z), d.w = al.w * (d.w - dl.w);
      }
      d4.x += d.x, d4.y += d.y, d4.z += d.z, d4.w += d.w;
    }
    if constexpr (kV) {
      const int64_t row = ok ? qi : -1;
      for (int j = 0; j < cnt && n_q > 0; j += kLook) {
        Chunk8<float> gv[kLook];
        float al[kLook];
        bool use[kLook];
#pragma unroll
        for (int u = 0; u < kLook; ++u) {  // (an entry out of range reads row 0 and edge 0)
          const int from = j + u < cnt ? j + u : cnt - 1;
          const int64_t r = __shfl(row, from, kGroup), e = __shfl(E, from, kGroup);
          use[u] = j + u < cnt && r >= 0;
          gv[u].load(go + (r >= 0 ? r : 0) * ldgo + c0);
          al[u] = alpha_e[(r >= 0 ? e : 0) * kHeads + h];
        }
#pragma unroll
        for (int u = 0; u < kLook; ++u)
          if (use[u])  // uniform over the group
#pragma unroll
            for (int i = 0; i < 8; ++i) acc[i] = fmaf(al[u], gv[u][i], acc[i]);
      }
    }
  }
  if constexpr (kV) store8(partial + s * kRow + c0, acc);
  d4.x = row16_sum(d4.x), d4.y = row16_sum(d4.y), d4.z = row16_sum(d4.z), d4.w = row16_sum(d4.w);
  if (lane == 0) *reinterpret_cast<float4*>(partial4 + s * kHeads) = d4;
}

// Row-encoder gradient runs: out[d] = sum over j in [ptr[d], ptr[d+1]) of
// mask_E * go[cell_E], E = perm[j] (an entry of the cell-major decoder list).
// 16 entries per index load, the rows of kLook entries in flight.
template <typename Tp, typename Tt, typename To>
__global__ void __launch_bounds__(kBlock)
row_mask_kernel(const Tp* __restrict__ pre, int64_t ldp, int64_t n_w, const Tt* __restrict__ table, int64_t n_cls,
                const float* __restrict__ go, int64_t n_cells, const int64_t* __restrict__ edge_window,
                const int64_t* __restrict__ edge_class, const int64_t* __restrict__ edge_cell, int64_t n_edges,
                const int64_t* __restrict__ ptr, const int64_t* __restrict__ perm, int64_t n_dest,
                To* __restrict__ out, int32_t* flag) {
  constexpr int kLook = 4;
  const int64_t d = int64_t(blockIdx.x) * kGroupsPerBlock + threadIdx.x / kGroup;
  const int lane = threadIdx.x % kGroup;
  if (d >= n_dest) return;
  const int64_t c0 = 8 * lane;
  int64_t st, en;
  segment(ptr, d, n_edges, st, en);
  float acc[8] = {0, 0, 0, 0, 0, 0, 0, 0};
  for (int64_t base = st; base < en; base += kGroup) {
    const int cnt = int(en - base < kGroup ? en - base : kGroup);
    const int64_t E = perm[base + (lane < cnt ? lane : cnt - 1)];
    const bool in = E >= 0 && E < n_edges;
    const int64_t w = in ? edge_window[E] : -1, c = in ? edge_class[E] : -1, cell = in ? edge_cell[E] : -1;
    const bool good = w >= 0 && w < n_w && c >= 0 && c < n_cls && cell >= 0 && cell < n_cells;
    if (!good && lane < cnt) raise_flag(flag, MANTIS_FLAG_INDEX);
    for (int j = 0; j < cnt; j += kLook) {
      Chunk8<Tp> pv[kLook];
      Chunk8<Tt> tv[kLook];
      Chunk8<float> gv[kLook];
      bool use[kLook];
#pragma unroll
      for (int u = 0; u < kLook; ++u) {
        const int from = j + u < cnt ? j + u : cnt - 1;
        const int64_t wu = __shfl(w, from, kGroup), cu = __shfl(c, from, kGroup), du = __shfl(cell, from, kGroup);
        use[u] = __shfl(int(good), from, kGroup) != 0 && j + u < cnt;
        if (use[u]) {  // uniform over the group
          pv[u].load(pre + wu * ldp + c0);
          tv[u].load(table + cu * kRow + c0);
          gv[u].load(go + du * kRow + c0);
        }
      }
#pragma unroll
      for (int u = 0; u < kLook; ++u)
        if (use[u])
#pragma unroll
          for (int i = 0; i < 8; ++i) acc[i] += (pv[u][i] + tv[u][i] > 0.f) ? gv[u][i] : 0.f;
    }
  }
  store8(out + d * kRow + c0, acc);
}

template <typename F>
bool with_type(int32_t dtype, F&& fn) {
  switch (dtype) {
    case MANTIS_F32: fn(float{}); return true;
    case MANTIS_BF16: fn(uint16_t{}); return true;
    case MANTIS_F16: fn(_Float16{}); return true;
    default: return false;
  }
}

// Workspace of the attention backward: delta, the packed row terms, per-edge alpha and dalpha,
// the class slice tables and the two kinds of partial rows.
struct AttnLayout {
  int64_t delta, stats, alpha, dalpha, slices, total;
};

// (untyped edges, n_classes == 0, need no per-edge terms)
AttnLayout attn_layout(int64_t n_q, int64_t n_edges, int64_t n_classes) {
  AttnLayout L;
  L.delta = 0;
  L.stats = L.delta + align256(n_q * kHeads * 4);
  L.alpha = L.stats + align256(n_q * kHeads * 16);
  if (n_classes == 0) {
    L.dalpha = L.slices = L.total = L.alpha;
    return L;
  }
  L.dalpha = L.alpha + align256(n_edges * kHeads * 4);
  L.slices = L.dalpha + align256(n_edges * kHeads * 4);
  // slice tables + 128-wide partials, then 4-wide partials
  const SliceLayout S = slice_layout(n_edges, n_classes, kRow);
  L.total = L.slices + S.total + align256(S.n_slices * kHeads * 4);
  return L;
}

}  // namespace
}  // namespace mantis

using namespace mantis;

extern "C" {

int64_t mantis_attention_backward_workspace(int64_t n_q, int64_t n_entries, int64_t n_classes) {
  // n_classes = 0: untyped edges (no bias / class values)
  if (n_q < 0 || n_entries < 0 || n_classes < 0) return -1;
  return attn_layout(n_q, n_entries, n_classes).total;
}

int32_t mantis_attention_backward(const void* q, const void* k, const void* v, int32_t dtype, int64_t ldq, int64_t ldk,
                                  int64_t ldv, int64_t n_q, int64_t n_k, const float* bias, int64_t n_classes,
                                  const void* vcls, int32_t vcls_dtype, const float* grad_out, int64_t ldgo,
                                  const float* m, const float* l, const int64_t* seg_ptr, const int64_t* src,
                                  const int64_t* cls, const int64_t* qid, int64_t n_entries, const int64_t* sseg_ptr,
                                  const int64_t* sqid, const int64_t* scls, const int64_t* cptr,
                                  const int64_t* cedge_q, void* workspace, int64_t workspace_bytes, void* dq,
                                  void* dk, void* dv, float* dbias_t, void* dvcls, int32_t* err_flag, void* stream) {
  if (n_q < 0 || n_k < 0 || n_entries < 0 || n_classes < 0) return MANTIS_E_ARG;
  if ((n_q > 0 && (!q || !grad_out || !m || !l || !dq || !seg_ptr)) || (n_k > 0 && (!k || !v || !dk || !dv || !sseg_ptr)))
    return MANTIS_E_ARG;
  if (n_entries > 0 && (!src || !sqid)) return MANTIS_E_ARG;
  if (ldq < kRow || ldk < kRow || ldv < kRow || ldgo < kRow || ldq % 8 || ldk % 8 || ldv % 8 || ldgo % 4)
    return MANTIS_E_ARG;
  const bool typed = bias != nullptr;  // class-typed edges: cls, scls and the class views
  if (typed && (n_classes <= 0 || (n_entries > 0 && (!cls || !scls)) || !cptr || (n_entries > 0 && !cedge_q) ||
                !dbias_t))
    return MANTIS_E_ARG;
  if (vcls && (!typed || !dvcls || (n_entries > 0 && !qid))) return MANTIS_E_ARG;
  for (const void* p : {q, k, v, static_cast<const void*>(grad_out), vcls, static_cast<const void*>(dq),
                        static_cast<const void*>(dk), static_cast<const void*>(dv), static_cast<const void*>(dvcls)})
    if (p && !aligned16(p)) return MANTIS_E_ARG;
  const AttnLayout L = attn_layout(n_q, n_entries, n_classes);
  if (!workspace || workspace_bytes < L.total || !aligned16(workspace)) return MANTIS_E_ARG;
  char* ws = static_cast<char*>(workspace);
  AttnBwd a{q, k, v, ldq, ldk, ldv, n_q, n_k, bias, n_classes, vcls, grad_out, ldgo, m, l,
            reinterpret_cast<float*>(ws + L.delta), reinterpret_cast<float4*>(ws + L.stats), 0.17677669529663687f, err_flag};
  // per-edge softmax terms: kept for the class sums of typed edges only
  float* alpha_e = typed ? reinterpret_cast<float*>(ws + L.alpha) : nullptr;
  float* dalpha_e = typed ? reinterpret_cast<float*>(ws + L.dalpha) : nullptr;
  hipStream_t s = as_stream(stream);
  bool ok_v = true;
  const bool ok = with_type(dtype, [&](auto t) {
    using T = decltype(t);
    auto run = [&](auto tv) {
      using Tv = decltype(tv);
      auto passes = [&](auto with_vcls) {
        constexpr bool kV = decltype(with_vcls)::value;
        if (n_q > 0)
          attn_bwd_q_kernel<T, Tv, kV><<<grid_rows(n_q), kBlock, 0, s>>>(
              a, seg_ptr, src, typed ? cls : nullptr, n_entries, static_cast<T*>(dq), alpha_e, dalpha_e,
              typed && !qid);
        if (n_k == 0) return;
        auto kv = [&](auto groups) {
          constexpr int kG = decltype(groups)::value;
          attn_bwd_kv_kernel<T, Tv, kV, kG><<<grid_rows(n_k * kG), kBlock, 0, s>>>(
              a, sseg_ptr, sqid, typed ? scls : nullptr, n_entries, static_cast<T*>(dk), static_cast<T*>(dv));
        };
        // a mean run of one chunk of 16 entries per group of the row
        if (n_entries < 16 * n_k) kv(std::integral_constant<int, 1>{});
        else if (n_entries < 64 * n_k) kv(std::integral_constant<int, 4>{});
        else kv(std::integral_constant<int, kGroupsPerBlock>{});
      };
      if (vcls) passes(std::true_type{});
      else passes(std::false_type{});
    };
    if (!vcls) run(float{});
    else ok_v = with_type(vcls_dtype, run);
  });
  if (!ok || !ok_v) return MANTIS_E_ARG;
  int32_t st = launched();
  if (st != MANTIS_OK || !typed) return st;
  // class sums over the class-major view: slice tables once, then dbias
  // (4-wide rows of dscore) and dvcls (alpha-weighted gradient rows)
  const SliceLayout S = slice_layout(n_entries, n_classes, kRow);
  char* sl = ws + L.slices;
  int64_t* slice_ptr = reinterpret_cast<int64_t*>(sl + S.slice_ptr);
  int64_t* slice_edge = reinterpret_cast<int64_t*>(sl + S.slice_edge);
  float* partial = reinterpret_cast<float*>(sl + S.partial);
  float* partial4 = reinterpret_cast<float*>(sl + S.total);
  slice_scan_kernel<<<1, 1024, 0, s>>>(cptr, n_classes, n_entries, slice_ptr);
  if ((st = launched()) != MANTIS_OK) return st;
  slice_edges_kernel<<<unsigned((S.n_slices + 1 + 255) / 256), 256, 0, s>>>(cptr, slice_ptr, n_classes, n_entries,
                                                                             S.n_slices, slice_edge);
  if ((st = launched()) != MANTIS_OK) return st;
  auto slices = vcls ? class_slice_kernel<true> : class_slice_kernel<false>;
  slices<<<grid_rows(S.n_slices), kBlock, 0, s>>>(alpha_e, dalpha_e, a.delta, grad_out, ldgo, qid, n_q, cedge_q, n_entries,
                                                  slice_edge, S.n_slices, partial, partial4, err_flag);
  if ((st = launched()) != MANTIS_OK) return st;
  st = slice_merge(partial4, kHeads, slice_ptr, S.n_slices, n_classes, dbias_t, s);
  if (st != MANTIS_OK || !vcls) return st;
  return slice_merge(partial, kRow, slice_ptr, S.n_slices, n_classes, dvcls, vcls_dtype, s);
}

int64_t mantis_row_encode_backward_workspace(int64_t n_entries, int64_t n_classes) {
  if (n_entries < 0 || n_classes < 0) return -1;
  return slice_layout(n_entries, n_classes, kRow).total;
}

int32_t mantis_row_encode_backward(const void* pre, int32_t pre_dtype, int64_t ldp, int64_t n_w, const void* table,
                                   int32_t table_dtype, int64_t n_cls, const float* grad_out, int64_t n_cells,
                                   const int64_t* edge_window, const int64_t* edge_class, const int64_t* edge_cell,
                                   int64_t n_entries, const int64_t* win_ptr, const int64_t* edge_rev,
                                   const int64_t* cls_ptr, const int64_t* cls_order, void* workspace,
                                   int64_t workspace_bytes, void* dpre, void* dtable, int32_t* err_flag,
                                   void* stream) {
  if (n_w < 0 || n_cls < 0 || n_cells < 0 || n_entries < 0 || ldp < kRow || ldp % 8) return MANTIS_E_ARG;
  if ((n_w > 0 && (!pre || !dpre || !win_ptr)) || (n_cls > 0 && (!table || !dtable || !cls_ptr))) return MANTIS_E_ARG;
  if (n_entries > 0 && (!edge_window || !edge_class || !edge_cell || !edge_rev || !cls_order || !grad_out))
    return MANTIS_E_ARG;
  for (const void* p : {pre, table, static_cast<const void*>(grad_out), static_cast<const void*>(dpre),
                        static_cast<const void*>(dtable)})
    if (p && !aligned16(p)) return MANTIS_E_ARG;
  const SliceLayout S = slice_layout(n_entries, n_cls, kRow);
  if (n_cls > 0 && (!workspace || workspace_bytes < S.total || !aligned16(workspace))) return MANTIS_E_ARG;
  hipStream_t s = as_stream(stream);
  int32_t st = MANTIS_OK;
  bool ok_t = true, ok_o = true;
  const bool ok_p = with_type(pre_dtype, [&](auto tp) {
    using Tp = decltype(tp);
    ok_t = with_type(table_dtype, [&](auto tt) {
      using Tt = decltype(tt);
      // dpre over the window-major entries (edge_rev), in pre's dtype
      if (n_w > 0)
        row_mask_kernel<Tp, Tt, Tp><<<grid_rows(n_w), kBlock, 0, s>>>(
            static_cast<const Tp*>(pre), ldp, n_w, static_cast<const Tt*>(table), n_cls, grad_out, n_cells,
            edge_window, edge_class, edge_cell, n_entries, win_ptr, edge_rev, n_w, static_cast<Tp*>(dpre), err_flag);
      if (n_cls == 0) return;
      // dtable: slices of the class-major entries, then each class's slices
      char* ws = static_cast<char*>(workspace);
      int64_t* slice_ptr = reinterpret_cast<int64_t*>(ws + S.slice_ptr);
      int64_t* slice_edge = reinterpret_cast<int64_t*>(ws + S.slice_edge);
      float* partial = reinterpret_cast<float*>(ws + S.partial);
      slice_scan_kernel<<<1, 1024, 0, s>>>(cls_ptr, n_cls, n_entries, slice_ptr);
      slice_edges_kernel<<<unsigned((S.n_slices + 1 + 255) / 256), 256, 0, s>>>(cls_ptr, slice_ptr, n_cls, n_entries,
                                                                                 S.n_slices, slice_edge);
      row_mask_kernel<Tp, Tt, float><<<grid_rows(S.n_slices), kBlock, 0, s>>>(
          static_cast<const Tp*>(pre), ldp, n_w, static_cast<const Tt*>(table), n_cls, grad_out, n_cells,
          edge_window, edge_class, edge_cell, n_entries, slice_edge, cls_order, S.n_slices, partial, err_flag);
      if ((st = launched()) != MANTIS_OK) return;
      st = slice_merge(partial, kRow, slice_ptr, S.n_slices, n_cls, dtable, table_dtype, s);
      ok_o = st != MANTIS_E_ARG;
    });
  });
  if (!ok_p || !ok_t || !ok_o) return MANTIS_E_ARG;
  if (st != MANTIS_OK) return st;
  return launched();
}

}  // extern "C"

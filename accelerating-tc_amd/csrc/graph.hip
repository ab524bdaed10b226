// Device graph: upload, simplification, orientation (ID / degree / A-direction
// / k-core), A-order relabelling and oriented-CSR construction, all in HBM.
//
// Layout in HBM (one graph):
//   src, dst   : uint32[m_raw]   raw records as read from the edge file
//   rowptr     : uint32[n+1]     oriented CSR offsets
//   col        : uint32[m+]      oriented CSR targets, ascending per row
//   esrc       : uint32[m+]      source of each CSR edge (edge-centric kernels)
//   vkey       : int32[n]        A-direction priority or core number
#include <algorithm>
#include <cmath>
#include <cstdio>
#include <cstring>

#include "engine.h"
#include "internal.h"

namespace tcx {
namespace {

constexpr int TB = 256;

inline unsigned grid_for(uint64_t n, int tb = TB) {
  uint64_t b = (n + tb - 1) / tb;
  if (b < 1) b = 1;
  if (b > (1u << 20)) b = 1u << 20;
  return (unsigned)b;
}

__device__ inline uint64_t gtid() { return (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; }
__device__ inline uint64_t gstride() { return (uint64_t)gridDim.x * blockDim.x; }

__global__ void k_fill_u32(uint32_t* p, uint32_t v, uint64_t n) {
  for (uint64_t i = gtid(); i < n; i += gstride()) p[i] = v;
}
__global__ void k_fill_i32(int32_t* p, int32_t v, uint64_t n) {
  for (uint64_t i = gtid(); i < n; i += gstride()) p[i] = v;
}

// Degree over the raw records (duplicates and self-loops counted),
// Hu/preTC.cu:119-123, Bisson/preTC.cu:65-76, tricount_gpu.cu:37-47.
// (prune) flag[v] = deg[v] <= 1, Hu/preTC.cu:139-144.
__global__ void k_low_degree_flag(const uint32_t* deg, uint32_t n, uint32_t* flag) {
  for (uint64_t v = gtid(); v < n; v += gstride()) flag[v] = deg[v] <= 1 ? 1u : 0u;
}

// Orient one raw record into a packed (src<<32 | dst) key; self-loops and
// pruned endpoints become the sentinel (n_out << 32), which sorts last.
// tie (optional, TC_ORIENT_DEGREE): equal degrees compare tie[] before ids.
__global__ void k_orient_keys(const uint32_t* __restrict__ s, const uint32_t* __restrict__ d,
                              uint64_t m, const uint32_t* __restrict__ deg, int mode,
                              const uint32_t* __restrict__ pruned_before, uint32_t n_out,
                              const uint32_t* __restrict__ tie, int shift,
                              uint64_t* __restrict__ keys) {
  const uint64_t sentinel = (uint64_t)n_out << shift;
  for (uint64_t i = gtid(); i < m; i += gstride()) {
    uint32_t a = s[i], b = d[i];
    bool swap;
    if (mode == TC_ORIENT_ID) {
      swap = a < b;  // src = larger id (Fox/preTC.cu:94-98)
    } else if (mode == TC_ORIENT_DEGREE) {
      uint32_t da = deg[a], db = deg[b];
      if (tie && da == db && tie[a] != tie[b]) swap = tie[a] > tie[b];
      else swap = da > db || (da == db && a < b);  // Hu/preTC.cu:129
    } else {
      uint32_t da = deg[a], db = deg[b];
      swap = da > db || (da == db && a > b);  // tricount_gpu.cu:76
    }
    uint32_t os = swap ? b : a, od = swap ? a : b;
    uint64_t key;
    if (os == od) {
      key = sentinel;
    } else if (pruned_before) {
      if (deg[os] <= 1 || deg[od] <= 1) key = sentinel;  // Hu/preTC.cu:151-160
      else key = ((uint64_t)(os - pruned_before[os]) << shift) | (od - pruned_before[od]);
    } else {
      key = ((uint64_t)os << shift) | od;
    }
    keys[i] = key;
  }
}

// Canonical simple-edge key (min<<32 | max); self-loops -> sentinel.
__global__ void k_simple_keys(const uint32_t* __restrict__ s, const uint32_t* __restrict__ d,
                              uint64_t m, uint32_t n, uint64_t* __restrict__ keys) {
  for (uint64_t i = gtid(); i < m; i += gstride()) {
    uint32_t a = s[i], b = d[i];
    uint32_t lo = a < b ? a : b, hi = a < b ? b : a;
    keys[i] = a == b ? ((uint64_t)n << 32) : (((uint64_t)lo << 32) | hi);
  }
}

// Both directions of every non-loop record (A-direction-seri.cpp:215-221).
__global__ void k_sym_keys(const uint32_t* __restrict__ s, const uint32_t* __restrict__ d,
                           uint64_t m, uint32_t n, int shift, uint64_t* __restrict__ keys) {
  for (uint64_t i = gtid(); i < m; i += gstride()) {
    uint32_t a = s[i], b = d[i];
    if (a == b) {
      keys[2 * i] = (uint64_t)n << shift;
      keys[2 * i + 1] = (uint64_t)n << shift;
    } else {
      keys[2 * i] = ((uint64_t)a << shift) | b;
      keys[2 * i + 1] = ((uint64_t)b << shift) | a;
    }
  }
}

__global__ void k_unzip(const uint64_t* __restrict__ keys, uint64_t m, uint32_t* __restrict__ s,
                        uint32_t* __restrict__ d) {
  for (uint64_t i = gtid(); i < m; i += gstride()) {
    uint64_t k = keys[i];
    s[i] = (uint32_t)(k >> 32);
    d[i] = (uint32_t)k;
  }
}

// Row offsets + targets + sources from keys sorted by (src,dst); one thread
// per key plus one for the tail (tricount_gpu.cu:127-137 builds the same
// offsets from a sorted first-endpoint array).
// col (and esrc) from sorted (src << 32 | dst) keys; rowptr comes from
// dev::k_rowptr_search, so runs of empty rows cost nothing extra.
__global__ void k_csr_cols(const uint64_t* __restrict__ keys, uint64_t m,
                           uint32_t* __restrict__ col, uint32_t* __restrict__ esrc) {
  for (uint64_t i = gtid(); i < m; i += gstride()) {
    const uint64_t k = keys[i];
    col[i] = (uint32_t)k;
    if (esrc) esrc[i] = (uint32_t)(k >> 32);
  }
}

__device__ inline unsigned long long wave_sum_u64(unsigned long long v) {
  for (int off = 32; off > 0; off >>= 1) v += __shfl_down(v, off, 64);
  return v;
}

// acc[0] += sum d+^2, acc[1] += sum d- d+ (d+ of every entry's target),
// acc[2] = max d+.  One workgroup a CU with one atomic per figure: atomics on
// three words of a line serialise at about 14 ns, and were all of the time with
// one per wave (n = 2^21: 1.16 ms) or eight workgroups a CU (n = 2^18, 3.8 * 10^6
// entries: 84 us).
constexpr uint32_t kStatThreads = 1024, kStatWaves = kStatThreads / 64;

__global__ __launch_bounds__(kStatThreads) void k_csr_stats(const uint32_t* __restrict__ rowptr,
                                                            const uint32_t* __restrict__ col,
                                                            uint32_t n, uint64_t m,
                                                            unsigned long long* acc) {
  __shared__ unsigned long long red[3][kStatWaves];
  unsigned long long s1 = 0, s2 = 0, mx = 0;
  for (uint64_t v = gtid(); v < n; v += gstride()) {
    const uint64_t d = rowptr[v + 1] - rowptr[v];
    s1 += d * d;
    mx = d > mx ? d : mx;
  }
  for (uint64_t e0 = gtid(); e0 < m; e0 += 4 * gstride()) {
    uint32_t v[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) v[i] = e0 + i * gstride() < m ? col[e0 + i * gstride()] : dev::kEmpty;
#pragma unroll
    for (int i = 0; i < 4; ++i) s2 += v[i] != dev::kEmpty ? rowptr[v[i] + 1] - rowptr[v[i]] : 0u;
  }
  s1 = wave_sum_u64(s1);
  s2 = wave_sum_u64(s2);
  for (int off = 32; off > 0; off >>= 1) {
    const unsigned long long o = __shfl_down(mx, off, 64);
    mx = o > mx ? o : mx;
  }
  if ((threadIdx.x & 63) == 0) {
    red[0][threadIdx.x >> 6] = s1;
    red[1][threadIdx.x >> 6] = s2;
    red[2][threadIdx.x >> 6] = mx;
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    for (uint32_t w = 1; w < kStatWaves; ++w) {
      s1 += red[0][w];
      s2 += red[1][w];
      mx = max(mx, red[2][w]);
    }
    atomicAdd(acc + 0, s1);
    atomicAdd(acc + 1, s2);
    atomicMax(acc + 2, mx);
  }
}

__global__ void k_row_degrees(const uint32_t* __restrict__ rp, uint32_t n,
                              uint32_t* __restrict__ deg) {
  for (uint64_t v = gtid(); v < n; v += gstride()) deg[v] = rp[v + 1] - rp[v];
}

// ---- A-direction peel (edge_directing/A-direction-seri.cpp:35-153) --------
//
// The serial peel assigns a vertex the label of the frontier level during
// which its runtime degree first drops to the threshold, so processing one
// whole level in parallel reproduces its labels exactly.  Runtime degrees
// start at twice the simple degree (each neighbour is listed twice, :44-73)
// and each peeled neighbour removes 2.
__global__ void k_adir_init(const uint32_t* __restrict__ rp, uint32_t n, int32_t* rtd,
                            int32_t* prio) {
  for (uint64_t v = gtid(); v < n; v += gstride()) {
    rtd[v] = 2 * (int32_t)(rp[v + 1] - rp[v]);
    prio[v] = -1;
  }
}

// Vertices collected by one wave in LDS on their way to a list: the list's
// counter takes one atomic per 64 of them or more (atomics on one word are
// serialised, about 14 ns each, and were most of a peel level's time).
struct Collect {
  uint32_t* buf;    // 128 words
  uint32_t* list;
  uint32_t* count;
  uint32_t held;    // wave-uniform

  __device__ void flush() {
    if (!held) return;
    const uint32_t lane = threadIdx.x & 63;
    uint32_t at = 0;
    if (lane == 0) at = atomicAdd(count, held);
    at = __shfl(at, 0, 64);
    dev::wave_sync();
    for (uint32_t i = lane; i < held; i += 64) list[at + i] = buf[i];
    dev::wave_sync();
    held = 0;
  }
  // every lane of the wave calls it
  __device__ void add(bool take, uint32_t v) {
    const uint64_t mask = dev::lanes(take);
    if (!mask) return;
    if (take) buf[dev::lanes_below(mask, held)] = v;
    held = dev::uniform(held + (uint32_t)__popcll(mask));
    if (held >= 64) flush();
  }
};

// frontier = the unpeeled vertices within the threshold, labelled
__global__ __launch_bounds__(256) void k_adir_scan(uint32_t n, const int32_t* __restrict__ rtd,
                                                   int32_t* prio, float t, int32_t label,
                                                   uint32_t* frontier, uint32_t* fcount) {
  __shared__ uint32_t buf[4][128];
  Collect out{buf[threadIdx.x >> 6], frontier, fcount, 0u};
  for (uint64_t v0 = gtid() & ~63ull; v0 < n; v0 += gstride()) {
    const uint64_t v = v0 + (threadIdx.x & 63);
    const bool take = v < n && prio[v] == -1 && (float)rtd[v] <= t;
    if (take) prio[v] = label;
    out.add(take, (uint32_t)v);
  }
  out.flush();
}

// What a peeled vertex does to its neighbours, A-direction: a peeled neighbour
// takes 2 from the runtime degree (it is listed twice in allEdges); a vertex
// is peeled when its degree first reaches the threshold, which makes the
// labels independent of the order of the frontier.
struct AdirStep {
  int32_t* rtd;
  int32_t* prio;
  float t;
  int32_t label;
  __device__ void next_level() { ++label; }
  __device__ bool live(uint32_t y) const {
    return __hip_atomic_load(prio + y, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == -1;
  }
  __device__ bool take(uint32_t y) const {
    const int32_t old = atomicSub(rtd + y, 2);
    if (!((float)old > t && (float)(old - 2) <= t)) return false;
    prio[y] = label;
    return true;
  }
};

// One level: step for every unpeeled neighbour y (live) of every frontier
// vertex; the ones it takes form the next frontier (order free).  A wave takes per
// (1 .. 64) frontier vertices and walks their neighbours back to back, 64 at a
// time, each lane finding its vertex by a search over the prefix of the
// lengths in LDS: with a wave per vertex most lanes idled on the short rows
// that make up the early levels.  Rows of kLongRow entries or more are set
// aside in pieces of that length (`big`: bounds) for k_peel_big, so no wave is
// left with a hub.
constexpr uint32_t kLongRow = 2048;

// Four neighbours of each lane (kEmpty: none), their loads and atomics in
// flight together.
template <class Step>
__device__ inline void peel4(const uint32_t (&y)[4], const Step& step, Collect& out) {
  bool live[4], take[4];
#pragma unroll
  for (int u = 0; u < 4; ++u) live[u] = y[u] != dev::kEmpty && step.live(y[u]);
#pragma unroll
  for (int u = 0; u < 4; ++u) take[u] = live[u] && step.take(y[u]);
#pragma unroll
  for (int u = 0; u < 4; ++u) out.add(take[u], y[u]);
}

template <class Step>
__global__ __launch_bounds__(256) void k_peel_expand(const uint32_t* __restrict__ frontier,
                                                     uint32_t fsize, uint32_t per,
                                                     const uint32_t* __restrict__ rp,
                                                     const uint32_t* __restrict__ col, Step step,
                                                     uint32_t* next, uint32_t* ncount, uint2* big,
                                                     uint32_t* nbig) {
  __shared__ uint32_t pre[4][64], at[4][64], buf[4][128];
  const uint32_t lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  const uint64_t wave = gtid() >> 6, nwaves = gstride() >> 6;
  Collect out{buf[wv], next, ncount, 0u};
  for (uint64_t f = wave * per; f < fsize; f += nwaves * per) {
    uint32_t b = 0, len = 0;
    if (lane < per && f + lane < fsize) {
      const uint32_t v = frontier[f + lane];
      b = rp[v];
      len = rp[v + 1] - b;
    }
    uint64_t lng = dev::lanes(len >= kLongRow);
    while (lng) {
      const uint32_t j = (uint32_t)__builtin_ctzll(lng);
      lng &= lng - 1;
      const uint32_t vb = __shfl(b, j, 64), vl = __shfl(len, j, 64);
      const uint32_t pieces = (vl + kLongRow - 1) / kLongRow;
      uint32_t p0 = 0;
      if (lane == 0) p0 = atomicAdd(nbig, pieces);
      p0 = __shfl(p0, 0, 64);
      for (uint32_t i = lane; i < pieces; i += 64)
        big[p0 + i] = make_uint2(vb + i * kLongRow, vb + min(vl, (i + 1) * kLongRow));
      if (lane == j) len = 0;
    }
    const uint32_t incl = dev::wave_incl_scan_dpp(len), total = __shfl(incl, 63, 64);
    pre[wv][lane] = incl - len;
    at[wv][lane] = b;
    dev::wave_sync();
    for (uint32_t i0 = 0; i0 < total; i0 += 256) {
      uint32_t y[4];
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const uint32_t i = i0 + 64 * u + lane, j = dev::seg64(pre[wv], i);
        y[u] = i < total ? col[at[wv][j] + (i - pre[wv][j])] : dev::kEmpty;
      }
      peel4(y, step, out);
    }
    dev::wave_sync();
  }
  out.flush();
}

template <class Step>
__global__ __launch_bounds__(256) void k_peel_big(const uint2* __restrict__ big, uint32_t nbig,
                                                  const uint32_t* __restrict__ col, Step step,
                                                  uint32_t* next, uint32_t* ncount) {
  __shared__ uint32_t buf[4][128];
  const uint32_t lane = threadIdx.x & 63;
  Collect out{buf[threadIdx.x >> 6], next, ncount, 0u};
  for (uint64_t k = gtid() >> 6; k < nbig; k += gstride() >> 6) {
    const uint2 r = big[k];
    for (uint32_t i0 = r.x; i0 < r.y; i0 += 256) {
      uint32_t y[4];
#pragma unroll
      for (int u = 0; u < 4; ++u) y[u] = i0 + 64 * u + lane < r.y ? col[i0 + 64 * u + lane] : dev::kEmpty;
      peel4(y, step, out);
    }
  }
  out.flush();
}

// Levels of few vertices and neighbours, one after the other in one workgroup,
// while they stay so: st = (vertices taken in all, levels, vertices of the last
// frontier, whether it is in b).  Most levels are like this, and a launch, a
// copy and a wait for each cost about 20 us; at most kSmallArcs neighbours keep a
// level here shorter than that.  k-core of R-MAT-14, 16, 20 (2^18, 2^19, 2^24
// records): 6.5 -> 4.8, 8.4 -> 6.1, 30.7 -> 25.5 ms, A-direction 1.35 -> 1.08,
// 2.09 -> 1.88, 7.76 -> 7.61.  kSmallLevels bounds a launch, a level of which takes
// 2 to 10 us, to some 20 ms at most (a path has a level for every two vertices);
// the host goes on from the frontier that it leaves.
constexpr uint32_t kSmallThreads = 1024, kSmallFrontier = 1024, kSmallArcs = 8192;
constexpr uint32_t kSmallLevels = 2048;

template <class Step>
__global__ __launch_bounds__(kSmallThreads) void k_peel_small(uint32_t* __restrict__ a,
                                                              uint32_t* __restrict__ b,
                                                              uint32_t fsize,
                                                              const uint32_t* __restrict__ rp,
                                                              const uint32_t* __restrict__ col,
                                                              Step step, uint32_t* st) {
  constexpr uint32_t kWaves = kSmallThreads / 64;
  __shared__ uint32_t pre[kSmallFrontier], at[kSmallFrontier];
  __shared__ uint32_t buf[kWaves][128], wsum[kWaves], s_next;
  const uint32_t tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
  uint32_t fs = fsize, taken = 0, levels = 0;  // the same in every thread
  uint32_t *F = a, *N = b;
  while (fs && fs <= kSmallFrontier && levels < kSmallLevels) {
    // row bounds and the prefix of the lengths
    uint32_t len = 0;
    if (tid < fs) {
      const uint32_t v = F[tid], r = rp[v];
      at[tid] = r;
      len = rp[v + 1] - r;
    }
    const uint32_t incl = dev::wave_incl_scan_dpp(len);
    if (lane == 63) wsum[wv] = incl;
    if (tid == 0) s_next = 0;
    __syncthreads();
    uint32_t before = 0, total = 0;
    for (uint32_t w = 0; w < kWaves; ++w) {
      before += w < wv ? wsum[w] : 0u;
      total += wsum[w];
    }
    if (tid < fs) pre[tid] = before + incl - len;
    __syncthreads();
    if (total > kSmallArcs) break;
    Collect out{buf[wv], N, &s_next, 0u};
    for (uint32_t i0 = 0; i0 < total; i0 += 4 * kSmallThreads) {
      uint32_t y[4];
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const uint32_t i = i0 + u * kSmallThreads + tid;
        uint32_t lo = 0, n = fs;  // last vertex whose arcs begin at or before i
        while (n > 1) {
          const uint32_t half = n >> 1;
          if (pre[lo + half] <= i) lo += half;
          n -= half;
        }
        y[u] = i < total ? col[at[lo] + (i - pre[lo])] : dev::kEmpty;
      }
      peel4(y, step, out);
    }
    out.flush();
    __syncthreads();  // the counter, and N's entries for the workgroup's next reads
    fs = s_next;
    __syncthreads();
    taken += fs;
    ++levels;
    step.next_level();
    uint32_t* t = F;
    F = N;
    N = t;
  }
  if (tid == 0) {
    st[0] = taken;
    st[1] = levels;
    st[2] = fs;
    st[3] = F == b;
  }
}

// ---- Bisson/A-direction.cpp degree record ----------------------------------
// Bisson's peel (Bisson/A-direction.cpp:43-163) records degreeRecord[v] =
// runTimeDegree[v] when the scan peels v (:96), but a cascade push writes the
// slot of the pushing frontier element's INDEX, not of the pushed vertex
// (:118 writes degreeRecord[i]).  The record therefore depends on the serial
// frontier order, which these kernels rebuild: a round's first frontier is
// ascending ids (:91-98); the next frontier lists pushed vertices in the order
// of their crossing decrement, i.e. by (pusher index p, position e of the
// vertex in the pusher's allEdges list).  allEdges[x] (:75-80 over the (i,
// nbr) pairs of :253-258) is [N(x) below x] + [N(x)] + [N(x) above x], so a
// neighbour y of rank r in N(x), with L neighbours below x, sits at
// e1 = r, e2 = L + r when y < x and at e1 = L + r, e2 = deg(x) + r when y > x.

__global__ void k_adir_scan_flags(uint32_t n, const int32_t* __restrict__ rtd,
                                  const int32_t* __restrict__ prio, float t,
                                  uint8_t* __restrict__ flags) {
  for (uint64_t v = gtid(); v < n; v += gstride())
    flags[v] = (prio[v] == -1 && (float)rtd[v] <= t) ? 1 : 0;
}

__global__ void k_adir_mark_scan(const uint32_t* __restrict__ F, uint32_t fs,
                                 const int32_t* __restrict__ rtd, int32_t* __restrict__ prio,
                                 int32_t label, int32_t* __restrict__ rec) {
  for (uint64_t i = gtid(); i < fs; i += gstride()) {
    const uint32_t v = F[i];
    prio[v] = label;
    rec[v] = rtd[v];
  }
}

// One event (y << 32 | p) per frontier element p and unpeeled neighbour y
// (each stands for y's two entries in allEdges[F[p]]); rtd[y] -= 2.
__global__ void k_adir_events(const uint32_t* __restrict__ F, uint32_t fs,
                              const uint32_t* __restrict__ rp, const uint32_t* __restrict__ col,
                              int32_t* rtd, const int32_t* __restrict__ prio,
                              uint64_t* __restrict__ ev, unsigned long long* ecount) {
  const uint32_t lane = threadIdx.x & 63;
  const uint64_t wave = gtid() >> 6, nwaves = gstride() >> 6;
  for (uint64_t p = wave; p < fs; p += nwaves) {
    const uint32_t x = F[p], b = rp[x], e = rp[x + 1];
    for (uint32_t base = b; base < e; base += 64) {
      const uint32_t i = base + lane;
      const uint32_t y = i < e ? col[i] : 0;
      const bool live = i < e && prio[y] == -1;
      const uint64_t mask = __ballot(live);
      unsigned long long at = 0;
      if (lane == 0 && mask) at = atomicAdd(ecount, (unsigned long long)__popcll(mask));
      at = __shfl(at, 0, 64);
      if (live) {
        atomicSub(rtd + y, 2);
        ev[at + __popcll(mask & ((1ull << lane) - 1))] = ((uint64_t)y << 32) | p;
      }
    }
  }
}

__device__ inline uint32_t lower_bound_u32(const uint32_t* a, uint32_t lo, uint32_t hi,
                                           uint32_t v) {
  while (lo < hi) {
    const uint32_t mid = lo + ((hi - lo) >> 1);
    if (a[mid] < v) lo = mid + 1;
    else hi = mid;
  }
  return lo;
}

// Over the events sorted by (y, p): y's k-th decrement (k = its runtime
// degree at the level's start - floor(t)) peels it, if it has that many.
// The j = ceil(k/2)-th pusher p* made it, at e1 (k odd) or e2; slot p* of
// the record takes floor(t) (the runtime degree right after the crossing).
// Pushed vertices go out with the key (p* << 32 | e*) of the next order.
__global__ void k_adir_cross(const uint64_t* __restrict__ ev, uint64_t E,
                             const uint32_t* __restrict__ F, const uint32_t* __restrict__ rp,
                             const uint32_t* __restrict__ col, const int32_t* __restrict__ rtd,
                             int32_t* __restrict__ prio, int32_t tfloor, int32_t label,
                             int32_t* __restrict__ rec, uint64_t* __restrict__ nkey,
                             uint32_t* __restrict__ nid, uint32_t* ncount) {
  for (uint64_t i = gtid(); i < E; i += gstride()) {
    const uint32_t y = (uint32_t)(ev[i] >> 32);
    if (i > 0 && (uint32_t)(ev[i - 1] >> 32) == y) continue;
    uint64_t lo = i, hi = E;  // first event of a larger y
    const uint64_t bound = ((uint64_t)y + 1) << 32;
    while (lo < hi) {
      const uint64_t mid = lo + ((hi - lo) >> 1);
      if (ev[mid] < bound) lo = mid + 1;
      else hi = mid;
    }
    const int64_t cy = (int64_t)(lo - i);
    const int64_t k = (int64_t)rtd[y] + 2 * cy - tfloor;
    if (k < 1 || k > 2 * cy) continue;
    const uint32_t p = (uint32_t)ev[i + (uint64_t)((k + 1) / 2) - 1];
    const uint32_t x = F[p], b = rp[x], e = rp[x + 1];
    const uint32_t r = lower_bound_u32(col, b, e, y) - b;
    const uint32_t L = lower_bound_u32(col, b, e, x) - b;
    const uint32_t e1 = y < x ? r : L + r;
    const uint32_t e2 = y < x ? L + r : (e - b) + r;
    prio[y] = label;
    rec[p] = tfloor;
    const uint32_t at = atomicAdd(ncount, 1u);
    nkey[at] = ((uint64_t)p << 32) | ((k & 1) ? e1 : e2);
    nid[at] = y;
  }
}

// One atomic per workgroup (launched with a few hundred).
__global__ __launch_bounds__(256) void k_min_unpeeled(uint32_t n, const int32_t* __restrict__ val,
                                                      const int32_t* __restrict__ state,
                                                      int32_t* out) {
  __shared__ int32_t red[4];
  int32_t mn = INT32_MAX;
  for (uint64_t v = gtid(); v < n; v += gstride())
    if (state[v] == -1 && val[v] < mn) mn = val[v];
  for (int off = 32; off > 0; off >>= 1) {
    int32_t o = __shfl_down(mn, off, 64);
    mn = o < mn ? o : mn;
  }
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = mn;
  __syncthreads();
  if (threadIdx.x == 0) {
    mn = min(min(red[0], red[1]), min(red[2], red[3]));
    if (mn != INT32_MAX) atomicMin(out, mn);
  }
}

// ---- k-core (edge_directing/kcore_direction.cpp:91-126) --------------------
// Level-synchronous peel: at level k every vertex whose remaining degree is
// <= k is removed with core number k; core numbers are order-independent.
__global__ void k_core_init(const uint32_t* __restrict__ rp, uint32_t n, int32_t* deg,
                            int32_t* core) {
  for (uint64_t v = gtid(); v < n; v += gstride()) {
    deg[v] = (int32_t)(rp[v + 1] - rp[v]);
    core[v] = -1;
  }
}

// `step` (optional) receives the index of the frontier that removes each
// vertex: every frontier is one step, numbered over the whole peel.
__global__ __launch_bounds__(256) void k_core_scan(uint32_t n, const int32_t* __restrict__ deg,
                                                   int32_t* core, int32_t k, uint32_t* frontier,
                                                   uint32_t* fcount, int32_t* step, int32_t t) {
  __shared__ uint32_t buf[4][128];
  Collect out{buf[threadIdx.x >> 6], frontier, fcount, 0u};
  for (uint64_t v0 = gtid() & ~63ull; v0 < n; v0 += gstride()) {
    const uint64_t v = v0 + (threadIdx.x & 63);
    const bool take = v < n && core[v] == -1 && deg[v] <= k;
    if (take) {
      core[v] = k;
      if (step) step[v] = t;
    }
    out.add(take, (uint32_t)v);
  }
  out.flush();
}

struct CoreStep {
  int32_t* deg;
  int32_t* core;
  int32_t k;
  int32_t* step;
  int32_t t;
  __device__ void next_level() { ++t; }
  __device__ bool live(uint32_t y) const {
    return __hip_atomic_load(core + y, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == -1;
  }
  __device__ bool take(uint32_t y) const {
    if (atomicSub(deg + y, 1) != k + 1) return false;
    core[y] = k;
    if (step) step[y] = t;
    return true;
  }
};

// keep[e] for a sorted symmetric key list: ADIR (mode 2), or KCORE (mode 3)
// and DEGENERACY (mode 5), whose keys both point up from the lower (key, id).
// tie (optional, A-direction): equal priorities compare tie[] before ids.
__global__ void k_sym_keep(const uint64_t* __restrict__ keys, uint64_t m2,
                           const int32_t* __restrict__ key, int mode,
                           const uint32_t* __restrict__ tie, uint8_t* keep) {
  for (uint64_t e = gtid(); e < m2; e += gstride()) {
    uint64_t kk = keys[e];
    uint32_t i = (uint32_t)(kk >> 32), j = (uint32_t)kk;
    int32_t pi = key[i], pj = key[j];
    bool k;
    if (tie && pi == pj && tie[i] != tie[j])
      k = tie[i] < tie[j];
    else if (mode == TC_ORIENT_ADIR || mode == TC_ORIENT_ADIR_OMP)
      k = pj > pi || (pj == pi && i < j);  // A-direction-seri.cpp:259-261, A-direction.cpp:266-268
    else k = pi < pj || (pi == pj && i < j);                         // kcore_direction.cpp:137-138
    keep[e] = k ? 1 : 0;
  }
}

// Tie keys of learned orientation ties: a vertex's forced out-degree (the
// neighbours strictly above it in the primary order: higher A-direction
// priority, or higher degree), ascending or (desc) descending.
__global__ void k_forced_sym(const uint32_t* __restrict__ rp, const uint32_t* __restrict__ col,
                             uint32_t n, const int32_t* __restrict__ key, int desc,
                             uint32_t* __restrict__ tie) {
  for (uint64_t v = gtid(); v < n; v += gstride()) {
    uint32_t h = 0;
    for (uint32_t e = rp[v]; e < rp[v + 1]; ++e) h += key[col[e]] > key[v];
    tie[v] = desc ? ~h : h;
  }
}

// over raw records (every record counts, as the degree does)
__global__ void k_forced_raw(const uint32_t* __restrict__ s, const uint32_t* __restrict__ d,
                             uint64_t m, const uint32_t* __restrict__ deg, uint32_t* h) {
  for (uint64_t i = gtid(); i < m; i += gstride()) {
    const uint32_t a = s[i], b = d[i];
    if (a == b) continue;
    if (deg[b] > deg[a]) atomicAdd(h + a, 1u);
    else if (deg[a] > deg[b]) atomicAdd(h + b, 1u);
  }
}

__global__ void k_tie_flip(uint32_t* __restrict__ h, uint32_t n) {
  for (uint64_t v = gtid(); v < n; v += gstride()) h[v] = ~h[v];
}

// A-direction cost function sum_v |d+(v) - avg| (verification.cpp:43-45's
// f_lp over the oriented CSR): per-block partial sums over a fixed grid, so
// the host's ordered sum of the partials is deterministic.
__global__ __launch_bounds__(256) void k_adir_cost(const uint32_t* __restrict__ rp, uint32_t n,
                                                   double avg, double* __restrict__ partial) {
  __shared__ double red[4];
  double acc = 0;
  for (uint64_t v = gtid(); v < n; v += gstride()) acc += fabs((double)(rp[v + 1] - rp[v]) - avg);
  for (int off = 32; off > 0; off >>= 1) acc += __shfl_xor(acc, off, 64);
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = acc;
  __syncthreads();
  if (threadIdx.x == 0) partial[blockIdx.x] = ((red[0] + red[1]) + red[2]) + red[3];
}

// A-order helpers: oriented out-degree over raw records (A-order.cpp:88-99)
// and the relabelled "reordered" records (:219-228).
__global__ void k_aorder_outdeg(const uint32_t* __restrict__ s, const uint32_t* __restrict__ d,
                                uint64_t m, const uint32_t* __restrict__ deg, uint32_t* rtd) {
  for (uint64_t i = gtid(); i < m; i += gstride()) {
    uint32_t a = s[i], b = d[i];
    bool swap = deg[a] > deg[b] || (deg[a] == deg[b] && a < b);
    atomicAdd(rtd + (swap ? b : a), 1u);
  }
}

// ---- id relabellings of the format tools ----------------------------------
__global__ void k_present_flags(const uint32_t* __restrict__ deg, uint32_t n,
                                uint32_t* __restrict__ f) {
  for (uint64_t v = gtid(); v < n; v += gstride()) f[v] = deg[v] ? 1u : 0u;
}

__global__ void k_fill_u64(uint64_t* p, uint64_t v, uint64_t n) {
  for (uint64_t i = gtid(); i < n; i += gstride()) p[i] = v;
}

// first[v] = smallest record index whose source is v
__global__ void k_first_src(const uint32_t* __restrict__ s, uint64_t m,
                            unsigned long long* first) {
  for (uint64_t i = gtid(); i < m; i += gstride()) atomicMin(first + s[i], (unsigned long long)i);
}

// adjust2tc order: ids by first appearance as a source, then the others by id
__global__ void k_first_keys(const uint64_t* __restrict__ first, uint32_t n, uint64_t m,
                             uint64_t* __restrict__ key, uint32_t* __restrict__ ids) {
  for (uint64_t v = gtid(); v < n; v += gstride()) {
    key[v] = first[v] != ~0ull ? first[v] : m + v;
    ids[v] = (uint32_t)v;
  }
}

// directionByReorder order: (degree, id) ascending
__global__ void k_degree_keys(const uint32_t* __restrict__ deg, uint32_t n,
                              uint64_t* __restrict__ key, uint32_t* __restrict__ ids) {
  for (uint64_t v = gtid(); v < n; v += gstride()) {
    key[v] = ((uint64_t)deg[v] << 32) | v;
    ids[v] = (uint32_t)v;
  }
}

// Bisson/A-direction.cpp:287-293 order: (priority, runtime degree at peel)
// ascending; ties keep ascending ids (stable sort of ids in order)
__global__ void k_adir_relabel_keys(const int32_t* __restrict__ prio,
                                    const int32_t* __restrict__ rec, uint32_t n,
                                    uint64_t* __restrict__ key, uint32_t* __restrict__ ids) {
  for (uint64_t v = gtid(); v < n; v += gstride()) {
    key[v] = ((uint64_t)(uint32_t)prio[v] << 32) | (uint32_t)rec[v];
    ids[v] = (uint32_t)v;
  }
}

// perm[order[j]] = j, or n - 1 - j when reversed
__global__ void k_rank_perm(const uint32_t* __restrict__ order, uint32_t n, bool reversed,
                            uint32_t* __restrict__ perm) {
  for (uint64_t j = gtid(); j < n; j += gstride())
    perm[order[j]] = reversed ? (uint32_t)(n - 1 - j) : (uint32_t)j;
}

__global__ void k_apply_perm(uint32_t* s, uint32_t* d, uint64_t m,
                             const uint32_t* __restrict__ perm) {
  for (uint64_t i = gtid(); i < m; i += gstride()) {
    s[i] = perm[s[i]];
    d[i] = perm[d[i]];
  }
}

__global__ void k_aorder_apply(uint32_t* s, uint32_t* d, uint64_t m, const uint32_t* __restrict__ deg,
                               const uint32_t* __restrict__ perm) {
  for (uint64_t i = gtid(); i < m; i += gstride()) {
    uint32_t a = s[i], b = d[i];
    bool swap = deg[a] > deg[b] || (deg[a] == deg[b] && a < b);
    uint32_t os = swap ? b : a, od = swap ? a : b;
    s[i] = perm[os];
    d[i] = perm[od];
  }
}

// rowptr + col (+ esrc) of the CSR of m sorted, unique keys over n rows.
int csr_launch(tc_ctx* c, const uint64_t* keys, uint64_t m, uint32_t n, uint32_t* rowptr,
               uint32_t* col, uint32_t* esrc) {
  if (m)
    hipLaunchKernelGGL(k_csr_cols, dim3(grid_for(m)), dim3(TB), 0, c->stream, keys, m, col, esrc);
  hipLaunchKernelGGL(dev::k_rowptr_search<uint64_t>, dim3(grid_for((uint64_t)n + 1)), dim3(TB), 0,
                     c->stream, keys, m, n, rowptr);
  TCX_HIP(hipGetLastError());
  return TC_OK;
}

int read_u32(tc_ctx* c, const uint32_t* dptr, uint32_t* out) {
  return fetch(c, out, dptr, sizeof(uint32_t));
}

// One peel level: *ns vertices of the next frontier N from the frontier F of
// fs vertices.
template <class Step>
int peel_level(tc_ctx* c, const uint32_t* F, uint32_t fs, const uint32_t* rp, const uint32_t* col,
               Step step, uint32_t* N, uint2* big, uint32_t* ns) {
  uint32_t* cnt = c->scratch.as<uint32_t>();
  TCX_HIP(hipMemsetAsync(cnt, 0, 8, c->stream));
  // one vertex a wave until every wave of the GPU has one
  uint32_t per = 1;
  while (per < 64 && fs / (2 * per) >= (uint32_t)c->num_cus * 32u) per *= 2;
  hipLaunchKernelGGL(k_peel_expand<Step>,
                     dim3(std::min<unsigned>((unsigned)c->num_cus * 8u,
                                             grid_for(((uint64_t)fs + per - 1) / per * 64))),
                     dim3(TB), 0, c->stream, F, fs, per, rp, col, step, N, cnt, big, cnt + 1);
  TCX_HIP(hipGetLastError());
  uint32_t h[2];  // next frontier, pieces of long rows
  TCX_TRY(fetch(c, h, cnt, 8));
  if (h[1]) {
    hipLaunchKernelGGL(k_peel_big<Step>,
                       dim3(std::min<unsigned>((unsigned)c->num_cus * 8u, grid_for(64ull * h[1]))),
                       dim3(TB), 0, c->stream, big, h[1], col, step, N, cnt);
    TCX_HIP(hipGetLastError());
    TCX_TRY(read_u32(c, cnt, h));
  }
  *ns = h[0];
  return TC_OK;
}

// Levels from the frontier F (fs vertices) on in one workgroup: *taken vertices
// in *levels levels (0: the first is too large; at most kSmallLevels), after which F
// and fs are the frontier to go on with.
template <class Step>
int peel_small(tc_ctx* c, uint32_t*& F, uint32_t*& N, uint32_t& fs, const uint32_t* rp,
               const uint32_t* col, Step step, uint32_t* taken, uint32_t* levels) {
  uint32_t* st = c->scratch.as<uint32_t>() + 4;
  hipLaunchKernelGGL(k_peel_small<Step>, dim3(1), dim3(kSmallThreads), 0, c->stream, F, N, fs, rp,
                     col, step, st);
  TCX_HIP(hipGetLastError());
  uint32_t h[4];
  TCX_TRY(fetch(c, h, st, 16));
  *taken = h[0];
  *levels = h[1];
  fs = h[2];
  if (h[3]) std::swap(F, N);
  return TC_OK;
}

}  // namespace

// Keys a << shift | b of ids up to n (the sentinel's source) that unique_u64 turns
// into a << 32 | b: without the unused bits between, sorting takes two passes
// fewer at n = 2^18 (37 us each for 4.2 * 10^6 keys) and one at 2^21 (0.36 ms, 6.7 *
// 10^7 keys).
static int key_shift(uint64_t nkeys, uint32_t n) {
  return nkeys >= kMinCompact ? std::max(1, (int)bit_width_u32(n)) : 32;
}

// Sort keys (in `keys`, scratch of the same size in `tmp`), drop duplicates
// and the sentinel, build the graph's oriented CSR.
static int csr_from_keys(tc_ctx* c, tc_graph* g, DevBuf& keys, DevBuf& tmp, uint64_t nkeys,
                         uint32_t n_out, bool already_sorted_unique, int shift = 32) {
  uint64_t* sorted = keys.as<uint64_t>();
  uint64_t nuniq = nkeys;
  uint64_t* uniq = sorted;
  if (!already_sorted_unique) {
    int end_bit = shift + bit_width_u32(n_out);
    TCX_TRY(sort_u64(c, keys.as<uint64_t>(), tmp.as<uint64_t>(), nkeys, end_bit, &sorted));
    uint64_t* other = sorted == keys.as<uint64_t>() ? tmp.as<uint64_t>() : keys.as<uint64_t>();
    uint64_t last = 0;
    TCX_TRY(unique_u64(c, sorted, other, nkeys, &nuniq, shift, &last));
    uniq = other;
    if (nuniq > 0 && last >> shift == n_out) --nuniq;  // sentinel
  }
  if (nuniq > kMaxCsrEntries)
    return fail(TC_ERR_RANGE, "%llu oriented edges exceed the 32-bit CSR offsets",
                (unsigned long long)nuniq);
  if (g->exported) TCX_HIP(hipDeviceSynchronize());
  g->n = n_out;
  g->m_or = nuniq;
  TCX_TRY(g->rowptr.reserve(sizeof(uint32_t) * ((size_t)n_out + 1)));
  TCX_TRY(g->col.reserve(sizeof(uint32_t) * std::max<uint64_t>(nuniq, 1)));
  TCX_TRY(g->esrc.reserve(sizeof(uint32_t) * std::max<uint64_t>(nuniq, 1)));
  TCX_TRY(csr_launch(c, uniq, nuniq, n_out, g->rowptr.as<uint32_t>(), g->col.as<uint32_t>(),
                     g->esrc.as<uint32_t>()));
  g->sched_version++;
  return compute_csr_stats(c, g);
}

int compute_csr_stats(tc_ctx* c, tc_graph* g) {
  TCX_TRY(c->accum.reserve(64));
  unsigned long long* acc = c->accum.as<unsigned long long>();
  TCX_HIP(hipMemsetAsync(acc, 0, 3 * sizeof(unsigned long long), c->stream));
  const uint64_t blocks = (std::max<uint64_t>(g->n, g->m_or) + kStatThreads - 1) / kStatThreads;
  hipLaunchKernelGGL(k_csr_stats,
                     dim3((unsigned)std::min<uint64_t>(std::max<uint64_t>(blocks, 1),
                                                       (uint64_t)c->num_cus)),
                     dim3(kStatThreads), 0, c->stream, g->rowptr.as<uint32_t>(), g->col.as<uint32_t>(), g->n,
                     g->m_or, acc);
  TCX_HIP(hipGetLastError());
  unsigned long long h[3];
  TCX_TRY(fetch(c, h, acc, sizeof(h)));
  g->sum_out_sq = h[0];
  g->sum_in_out = h[1];
  g->max_out = (uint32_t)h[2];
  return TC_OK;
}

// Simple symmetric adjacency as sorted unique keys (both directions).
static int sym_keys(tc_ctx* c, tc_graph* g, DevBuf& keys, DevBuf& tmp, uint64_t** out,
                    uint64_t* m2) {
  uint64_t nk = 2 * g->m_raw;
  const int shift = key_shift(nk, g->n_raw);
  TCX_TRY(keys.reserve(8 * std::max<uint64_t>(nk, 1)));
  TCX_TRY(tmp.reserve(8 * std::max<uint64_t>(nk, 1)));
  hipLaunchKernelGGL(k_sym_keys, dim3(grid_for(g->m_raw)), dim3(TB), 0, c->stream,
                     g->src.as<uint32_t>(), g->dst.as<uint32_t>(), g->m_raw, g->n_raw, shift,
                     keys.as<uint64_t>());
  TCX_HIP(hipGetLastError());
  uint64_t* sorted;
  TCX_TRY(sort_u64(c, keys.as<uint64_t>(), tmp.as<uint64_t>(), nk,
                   shift + bit_width_u32(g->n_raw), &sorted));
  uint64_t* other = sorted == keys.as<uint64_t>() ? tmp.as<uint64_t>() : keys.as<uint64_t>();
  uint64_t nu = 0;
  uint64_t last = 0;
  TCX_TRY(unique_u64(c, sorted, other, nk, &nu, shift, &last));
  if (nu > 0 && last >> shift == g->n_raw) --nu;
  *out = other;
  *m2 = nu;
  return TC_OK;
}

static int sym_csr(tc_ctx* c, const uint64_t* keys, uint64_t m2, uint32_t n, DevBuf& rp,
                   DevBuf& col) {
  TCX_TRY(rp.reserve(sizeof(uint32_t) * ((size_t)n + 1)));
  TCX_TRY(col.reserve(sizeof(uint32_t) * std::max<uint64_t>(m2, 1)));
  TCX_TRY(csr_launch(c, keys, m2, n, rp.as<uint32_t>(), col.as<uint32_t>(), nullptr));
  return TC_OK;
}

// One round-level of Bisson's peel with the serial frontier order (see the
// degree-record kernels): frontier F (fs, in serial order) -> next frontier
// N in serial order; *ns its size.
struct AdirOrdered {
  DevBuf ev, evtmp, nkey, nktmp, nid, nitmp, flags;
};

static int adir_level_ordered(tc_ctx* c, AdirOrdered& o, const uint32_t* F, uint32_t fs,
                              const uint32_t* rp, const uint32_t* col, int32_t* rtd,
                              int32_t* prio, float t, int32_t label, int32_t* rec, uint32_t* N,
                              uint32_t* ns) {
  unsigned long long* ecount = c->accum.as<unsigned long long>();
  uint32_t* cnt = c->scratch.as<uint32_t>();
  TCX_HIP(hipMemsetAsync(ecount, 0, 8, c->stream));
  hipLaunchKernelGGL(k_adir_events, dim3(std::min<unsigned>(4096, grid_for(fs * 64ull))),
                     dim3(TB), 0, c->stream, F, fs, rp, col, rtd, prio, o.ev.as<uint64_t>(),
                     ecount);
  TCX_HIP(hipGetLastError());
  unsigned long long E = 0;
  TCX_HIP(hipMemcpyAsync(&E, ecount, 8, hipMemcpyDeviceToHost, c->stream));
  TCX_HIP(hipStreamSynchronize(c->stream));
  *ns = 0;
  if (E == 0) return TC_OK;
  uint64_t* sorted;
  TCX_TRY(sort_u64(c, o.ev.as<uint64_t>(), o.evtmp.as<uint64_t>(), E, 64, &sorted));
  TCX_HIP(hipMemsetAsync(cnt, 0, 4, c->stream));
  hipLaunchKernelGGL(k_adir_cross, dim3(grid_for(E)), dim3(TB), 0, c->stream, sorted,
                     (uint64_t)E, F, rp, col, rtd, prio, (int32_t)floorf(t), label, rec,
                     o.nkey.as<uint64_t>(), o.nid.as<uint32_t>(), cnt);
  TCX_HIP(hipGetLastError());
  uint32_t pushed = 0;
  TCX_TRY(read_u32(c, cnt, &pushed));
  if (pushed) {
    uint64_t* sk;
    uint32_t* order;
    TCX_TRY(sort_pairs_u64_u32(c, o.nkey.as<uint64_t>(), o.nktmp.as<uint64_t>(),
                               o.nid.as<uint32_t>(), o.nitmp.as<uint32_t>(), pushed, 64, &sk,
                               &order));
    TCX_HIP(hipMemcpyAsync(N, order, 4ull * pushed, hipMemcpyDeviceToDevice, c->stream));
  }
  *ns = pushed;
  return TC_OK;
}

// A-direction peel.  With rec non-NULL it also fills Bisson's degree record
// (zero where nothing is written, as the reference's memset leaves it), which
// needs the serial frontier order; without it the frontiers are unordered.
// thre_param > 0 selects the OpenMP program's schedule
// (edge_directing/A-direction.cpp:36-161): threshold0 = 2 totalEdge / n, a
// round's cascade runs only while its frontier holds more than n / 5000 and
// more than 200 vertices, for at most six levels, and the threshold grows by
// (int)threshold0 * thre_param / 5 per round.
static int adir_peel(tc_ctx* c, uint32_t n, uint64_t m2, const uint32_t* rp, const uint32_t* col,
                     int32_t* prio, int32_t* rec = nullptr, double thre_param = 0) {
  const bool omp = thre_param > 0;
  DevBuf rtd, fa, fb, big;
  TCX_TRY(big.reserve(16 * (m2 / kLongRow + 1)));
  TCX_TRY(rtd.reserve(sizeof(int32_t) * ((size_t)n + 1)));
  TCX_TRY(fa.reserve(sizeof(uint32_t) * ((size_t)n + 1)));
  TCX_TRY(fb.reserve(sizeof(uint32_t) * ((size_t)n + 1)));
  TCX_TRY(c->scratch.reserve(64));
  TCX_TRY(c->accum.reserve(64));
  uint32_t* cnt = c->scratch.as<uint32_t>();
  AdirOrdered ord;
  if (rec) {
    TCX_TRY(ord.ev.reserve(8 * std::max<uint64_t>(m2, 1)));
    TCX_TRY(ord.evtmp.reserve(8 * std::max<uint64_t>(m2, 1)));
    TCX_TRY(ord.nkey.reserve(8 * ((size_t)n + 1)));
    TCX_TRY(ord.nktmp.reserve(8 * ((size_t)n + 1)));
    TCX_TRY(ord.nid.reserve(4 * ((size_t)n + 1)));
    TCX_TRY(ord.nitmp.reserve(4 * ((size_t)n + 1)));
    TCX_TRY(ord.flags.reserve((size_t)n + 1));
    TCX_HIP(hipMemsetAsync(rec, 0, 4ull * n, c->stream));
  }
  hipLaunchKernelGGL(k_adir_init, dim3(grid_for(n)), dim3(TB), 0, c->stream, rp, n,
                     rtd.as<int32_t>(), prio);
  TCX_HIP(hipGetLastError());
  // A-direction-seri.cpp:37 and :77, with edgeNum = 2m (totalEdge, :228,:252);
  // A-direction.cpp:38,78
  unsigned int edgeNum = (unsigned int)m2;
  int nodeNum = (int)n;
  float threshold = omp ? 2 * ((float)edgeNum) / nodeNum : ((float)edgeNum) / nodeNum + 1;
  int threshold_old = threshold;
  auto step = [&]() {
    if (omp) threshold += (double)threshold_old * thre_param / 5;  // A-direction.cpp:139
    else threshold += threshold_old;                               // A-direction-seri.cpp:127
  };
  int32_t label = 0;
  uint64_t peeled = 0;
  uint32_t* F = fa.as<uint32_t>();
  uint32_t* N = fb.as<uint32_t>();
  for (;;) {
    uint32_t fs = 0;
    if (rec) {  // ascending ids, as the serial scan appends them
      hipLaunchKernelGGL(k_adir_scan_flags, dim3(grid_for(n)), dim3(TB), 0, c->stream, n,
                         rtd.as<int32_t>(), prio, threshold, ord.flags.as<uint8_t>());
      TCX_HIP(hipGetLastError());
      uint64_t f64 = 0;
      TCX_TRY(select_indices(c, ord.flags.as<uint8_t>(), n, F, &f64));
      fs = (uint32_t)f64;
      if (fs)
        hipLaunchKernelGGL(k_adir_mark_scan, dim3(grid_for(fs)), dim3(TB), 0, c->stream, F, fs,
                           rtd.as<int32_t>(), prio, label, rec);
      TCX_HIP(hipGetLastError());
    } else {
      TCX_HIP(hipMemsetAsync(cnt, 0, sizeof(uint32_t), c->stream));
      hipLaunchKernelGGL(k_adir_scan, dim3(std::min(grid_for(n), 1024u)), dim3(TB), 0, c->stream, n,
                         rtd.as<int32_t>(), prio, threshold, label, F, cnt);
      TCX_HIP(hipGetLastError());
      TCX_TRY(read_u32(c, cnt, &fs));
    }
    peeled += fs;
    label++;
    int inner = 0;
    // one workgroup while it can; rows are no shorter than half the last threshold
    const double arcs = (threshold - threshold_old) / 2;
    bool small = !omp && !rec;
    while (fs > 0 && (!omp || (fs > (uint32_t)(nodeNum / 5000) && fs > 200 && inner <= 5))) {
      if (small && fs <= kSmallFrontier && fs * arcs <= kSmallArcs) {
        uint32_t taken = 0, levels = 0;
        TCX_TRY(peel_small(c, F, N, fs, rp, col,
                           AdirStep{rtd.as<int32_t>(), prio, threshold, label}, &taken, &levels));
        peeled += taken;
        label += (int32_t)levels;
        small = levels == kSmallLevels;  // else what is left, if any, is too large
        continue;
      }
      small = !omp && !rec;
      inner++;
      uint32_t ns = 0;
      if (rec) {
        TCX_TRY(adir_level_ordered(c, ord, F, fs, rp, col, rtd.as<int32_t>(), prio, threshold,
                                   label, rec, N, &ns));
      } else {
        TCX_TRY(peel_level(c, F, fs, rp, col,
                           AdirStep{rtd.as<int32_t>(), prio, threshold, label}, N,
                           big.as<uint2>(), &ns));
      }
      peeled += ns;
      std::swap(F, N);
      fs = ns;
      label++;
    }
    if (peeled >= n) break;
    step();
    // Rounds whose scan finds nothing only advance the label and threshold.
    TCX_HIP(hipMemsetAsync(cnt, 0x7f, sizeof(int32_t), c->stream));
    hipLaunchKernelGGL(k_min_unpeeled, dim3(std::min(grid_for(n), 512u)), dim3(TB), 0, c->stream, n,
                       rtd.as<int32_t>(), prio, (int32_t*)cnt);
    TCX_HIP(hipGetLastError());
    int32_t minr = 0;
    TCX_TRY(read_u32(c, cnt, (uint32_t*)&minr));
    while (!((float)minr <= threshold)) {
      label++;
      step();
    }
  }
  return TC_OK;
}

// Core numbers into `core`; with `step` non-NULL, also the removal step of
// every vertex.  A vertex removed at step t has at most core[v] neighbours
// removed at step t or later (its remaining degree when its frontier formed),
// so orienting every edge from the lower (step, id) bounds d+(v) by core[v].
static int kcore_peel(tc_ctx* c, uint32_t n, uint64_t m2, const uint32_t* rp, const uint32_t* col,
                      int32_t* core, int32_t* step = nullptr) {
  DevBuf deg, fa, fb, big;
  TCX_TRY(big.reserve(16 * (m2 / kLongRow + 1)));
  TCX_TRY(deg.reserve(sizeof(int32_t) * ((size_t)n + 1)));
  TCX_TRY(fa.reserve(sizeof(uint32_t) * ((size_t)n + 1)));
  TCX_TRY(fb.reserve(sizeof(uint32_t) * ((size_t)n + 1)));
  TCX_TRY(c->scratch.reserve(64));
  uint32_t* cnt = c->scratch.as<uint32_t>();
  hipLaunchKernelGGL(k_core_init, dim3(grid_for(n)), dim3(TB), 0, c->stream, rp, n,
                     deg.as<int32_t>(), core);
  TCX_HIP(hipGetLastError());
  uint64_t removed = 0;
  int32_t k = 0, t = 0;
  uint32_t* F = fa.as<uint32_t>();
  uint32_t* N = fb.as<uint32_t>();
  while (removed < n) {
    TCX_HIP(hipMemsetAsync(cnt, 0, sizeof(uint32_t), c->stream));
    hipLaunchKernelGGL(k_core_scan, dim3(std::min(grid_for(n), 1024u)), dim3(TB), 0, c->stream, n,
                       deg.as<int32_t>(), core, k, F, cnt, step, t);
    TCX_HIP(hipGetLastError());
    uint32_t fs = 0;
    TCX_TRY(read_u32(c, cnt, &fs));
    removed += fs;
    if (fs) ++t;
    bool small = true;  // (rows are no shorter than k)
    while (fs > 0) {
      if (small && fs <= kSmallFrontier && (uint64_t)fs * k <= kSmallArcs) {
        uint32_t taken = 0, levels = 0;
        TCX_TRY(peel_small(c, F, N, fs, rp, col, CoreStep{deg.as<int32_t>(), core, k, step, t},
                           &taken, &levels));
        removed += taken;
        t += (int32_t)levels;
        if (levels && fs == 0) --t;  // the last level took nothing
        small = levels == kSmallLevels;
        continue;
      }
      small = true;
      uint32_t ns = 0;
      TCX_TRY(peel_level(c, F, fs, rp, col, CoreStep{deg.as<int32_t>(), core, k, step, t}, N,
                         big.as<uint2>(), &ns));
      removed += ns;
      if (ns) ++t;
      std::swap(F, N);
      fs = ns;
    }
    if (removed >= n) break;
    TCX_HIP(hipMemsetAsync(cnt, 0x7f, sizeof(int32_t), c->stream));
    hipLaunchKernelGGL(k_min_unpeeled, dim3(std::min(grid_for(n), 512u)), dim3(TB), 0, c->stream, n,
                       deg.as<int32_t>(), core, (int32_t*)cnt);
    TCX_HIP(hipGetLastError());
    int32_t mind = 0;
    TCX_TRY(read_u32(c, cnt, (uint32_t*)&mind));
    k = std::max(k + 1, mind);
  }
  return TC_OK;
}

int vertex_degrees(tc_ctx* c, tc_graph* g) {
  if (g->vdeg_version == g->sched_version) return TC_OK;
  TCX_TRY(g->vdeg.reserve(4 * ((size_t)g->n + 1)));
  hipLaunchKernelGGL(k_fill_u32, dim3(grid_for(g->n)), dim3(TB), 0, c->stream,
                     g->vdeg.as<uint32_t>(), 0u, (uint64_t)g->n);
  TCX_TRY(count_ids(c, g->col.as<uint32_t>(), nullptr, g->m_or, g->n, g->vdeg.as<uint32_t>()));
  g->vdeg_version = g->sched_version;
  return TC_OK;
}

int graph_clone_records(tc_ctx* c, const tc_graph* g, tc_graph** out) {
  *out = nullptr;
  const bool from_csr = g->csr_only;
  const uint64_t m = from_csr ? (g->orient_mode >= 0 ? g->m_or : 0) : g->m_raw;
  const void* ps = from_csr ? g->esrc.p : g->src.p;
  const void* pd = from_csr ? g->col.p : g->dst.p;
  tc_graph* h = new tc_graph();
  h->ctx = c;
  h->m_raw = m;
  int st = h->src.reserve(4 * std::max<uint64_t>(m, 1));
  if (st == TC_OK) st = h->dst.reserve(4 * std::max<uint64_t>(m, 1));
  if (st == TC_OK && m &&
      (hipMemcpyAsync(h->src.p, ps, 4 * m, hipMemcpyDeviceToDevice, c->stream) != hipSuccess ||
       hipMemcpyAsync(h->dst.p, pd, 4 * m, hipMemcpyDeviceToDevice, c->stream) != hipSuccess))
    st = fail(TC_ERR_HIP, "record copy failed");
  uint32_t mx = 0;
  if (st == TC_OK && m) st = max_ids(c, h->src.as<uint32_t>(), h->dst.as<uint32_t>(), m, &mx);
  if (st != TC_OK) {
    delete h;
    return st;
  }
  h->n = m ? mx + 1 : 0;
  h->n_raw = h->n;
  *out = h;
  return TC_OK;
}

}  // namespace tcx

using namespace tcx;

static int check_graph(tc_graph* g) {
  if (!g || !g->ctx) return fail(TC_ERR_ARG, "NULL graph");
  TCX_HIP(hipSetDevice(g->ctx->device));
  return TC_OK;
}

// Passes over the raw records need them: a graph loaded from a CSR has none.
static int check_records(tc_graph* g) {
  TCX_TRY(check_graph(g));
  if (g->csr_only)
    return fail(TC_ERR_STATE, "the graph was built from an oriented CSR and holds no raw records");
  return TC_OK;
}

extern "C" {

int tc_graph_create(tc_ctx* c, const uint32_t* src, const uint32_t* dst, uint64_t m,
                    uint32_t n_hint, tc_graph** out) {
  PoolScope scope(c);
  if (!c || !out) return fail(TC_ERR_ARG, "NULL argument");
  if (m && (!src || !dst)) return fail(TC_ERR_ARG, "NULL edge arrays");
  *out = nullptr;
  TCX_HIP(hipSetDevice(c->device));
  tc_graph* g = new tc_graph();
  g->ctx = c;
  g->m_raw = m;
  int st = g->src.reserve(4 * std::max<uint64_t>(m, 1));
  if (st == TC_OK) st = g->dst.reserve(4 * std::max<uint64_t>(m, 1));
  if (st != TC_OK) { delete g; return st; }
  if (m) {
    st = upload(c, g->src.p, src, 4 * m);
    if (st == TC_OK) st = upload(c, g->dst.p, dst, 4 * m);
    uint32_t mx = 0;
    if (st == TC_OK) st = max_ids(c, g->src.as<uint32_t>(), g->dst.as<uint32_t>(), m, &mx);
    if (st != TC_OK) { delete g; return st; }
    if (mx >= 0x7FFFFFFFu) {
      delete g;
      return fail(TC_ERR_RANGE, "vertex id %u exceeds 2^31-2", mx);
    }
    if (n_hint && mx >= n_hint) {
      delete g;
      return fail(TC_ERR_RANGE, "vertex id %u >= n_hint %u", mx, n_hint);
    }
    g->n = n_hint ? n_hint : mx + 1;
  } else {
    g->n = n_hint;
  }
  g->n_raw = g->n;
  *out = g;
  return TC_OK;
}

int tc_graph_destroy(tc_graph* g) {
  if (!g) return TC_OK;
  if (g->ctx) {
    (void)hipSetDevice(g->ctx->device);
    (void)hipStreamSynchronize(g->ctx->stream);
    if (g->exported) (void)hipDeviceSynchronize();
  }
  delete g;
  return TC_OK;
}

int tc_graph_simplify(tc_ctx* c, tc_graph* g) {
  PoolScope scope(c);
  TCX_TRY(check_records(g));
  if (c != g->ctx) return fail(TC_ERR_ARG, "graph belongs to another context");
  if (g->m_raw == 0) return TC_OK;
  DevBuf keys, tmp;
  TCX_TRY(keys.reserve(8 * g->m_raw));
  TCX_TRY(tmp.reserve(8 * g->m_raw));
  hipLaunchKernelGGL(k_simple_keys, dim3(grid_for(g->m_raw)), dim3(TB), 0, c->stream,
                     g->src.as<uint32_t>(), g->dst.as<uint32_t>(), g->m_raw, g->n_raw,
                     keys.as<uint64_t>());
  TCX_HIP(hipGetLastError());
  uint64_t* sorted;
  TCX_TRY(sort_u64(c, keys.as<uint64_t>(), tmp.as<uint64_t>(), g->m_raw,
                   32 + bit_width_u32(g->n_raw), &sorted));
  uint64_t* other = sorted == keys.as<uint64_t>() ? tmp.as<uint64_t>() : keys.as<uint64_t>();
  uint64_t nu = 0;
  TCX_TRY(unique_u64(c, sorted, other, g->m_raw, &nu));
  if (nu > 0) {
    uint64_t last = 0;
    TCX_TRY(fetch(c, &last, other + nu - 1, 8));
    if ((uint32_t)(last >> 32) == g->n_raw) --nu;
  }
  hipLaunchKernelGGL(k_unzip, dim3(grid_for(nu)), dim3(TB), 0, c->stream, other, nu,
                     g->src.as<uint32_t>(), g->dst.as<uint32_t>());
  TCX_HIP(hipGetLastError());
  TCX_HIP(hipStreamSynchronize(c->stream));
  g->m_raw = nu;
  return TC_OK;
}

int tc_graph_relabel_aorder(tc_ctx* c, tc_graph* g, uint32_t* perm_out) {
  tc_bw_model ref;
  bw_model_reference(&ref);
  return tc_graph_relabel_aorder_model(c, g, &ref, perm_out);
}

int tc_graph_relabel_aorder_model(tc_ctx* c, tc_graph* g, const tc_bw_model* model,
                                  uint32_t* perm_out) {
  PoolScope scope(c);
  if (!model) return fail(TC_ERR_ARG, "NULL bandwidth model");
  // the bucket heaps need a strict weak order: finite, positive bandwidths
  for (int l = 2; l < 10; ++l)
    if (!(std::isfinite(model->table[l]) && model->table[l] > 0 &&
          std::isfinite(model->lambda[l]) && model->lambda[l] >= 0))
      return fail(TC_ERR_ARG, "bandwidth model entry %d is not finite and positive", l);
  if (!(std::isfinite(model->a) && model->a > 0 && std::isfinite(model->b) &&
        std::isfinite(model->lambda_tail) && model->lambda_tail >= 0))
    return fail(TC_ERR_ARG, "bandwidth model power law is not finite and positive");
  TCX_TRY(check_records(g));
  if (c != g->ctx) return fail(TC_ERR_ARG, "graph belongs to another context");
  uint32_t n = g->n_raw;
  if (n == 0) return fail(TC_ERR_UNSUPPORTED, "A-order on an empty graph");
  DevBuf deg, rtd, perm;
  TCX_TRY(deg.reserve(4 * (size_t)n));
  TCX_TRY(rtd.reserve(4 * (size_t)n));
  TCX_TRY(perm.reserve(4 * (size_t)n));
  hipLaunchKernelGGL(k_fill_u32, dim3(grid_for(n)), dim3(TB), 0, c->stream, deg.as<uint32_t>(),
                     0u, (uint64_t)n);
  hipLaunchKernelGGL(k_fill_u32, dim3(grid_for(n)), dim3(TB), 0, c->stream, rtd.as<uint32_t>(),
                     0u, (uint64_t)n);
  TCX_TRY(count_ids(c, g->src.as<uint32_t>(), g->dst.as<uint32_t>(), g->m_raw, n,
                    deg.as<uint32_t>()));
  hipLaunchKernelGGL(k_aorder_outdeg, dim3(grid_for(g->m_raw)), dim3(TB), 0, c->stream,
                     g->src.as<uint32_t>(), g->dst.as<uint32_t>(), g->m_raw, deg.as<uint32_t>(),
                     rtd.as<uint32_t>());
  TCX_HIP(hipGetLastError());
  std::vector<uint32_t> h_rtd(n), h_perm(n);
  TCX_HIP(hipMemcpyAsync(h_rtd.data(), rtd.p, 4 * (size_t)n, hipMemcpyDeviceToHost, c->stream));
  TCX_HIP(hipStreamSynchronize(c->stream));
  TCX_TRY(aorder_perm_from_outdeg(h_rtd.data(), n, h_perm.data(), *model));
  TCX_HIP(hipMemcpyAsync(perm.p, h_perm.data(), 4 * (size_t)n, hipMemcpyHostToDevice, c->stream));
  hipLaunchKernelGGL(k_aorder_apply, dim3(grid_for(g->m_raw)), dim3(TB), 0, c->stream,
                     g->src.as<uint32_t>(), g->dst.as<uint32_t>(), g->m_raw, deg.as<uint32_t>(),
                     perm.as<uint32_t>());
  TCX_HIP(hipGetLastError());
  // The relabelled records are what A-order writes to its "reordered" file
  // (A-order.cpp:206-228); a program reading them back takes the vertex count
  // as the largest id + 1 (A-direction-seri.cpp:187-193), not the old n.
  uint32_t new_n = 0;
  if (g->m_raw) {
    uint32_t mx = 0;
    TCX_TRY(max_ids(c, g->src.as<uint32_t>(), g->dst.as<uint32_t>(), g->m_raw, &mx));
    new_n = mx + 1;
  }
  TCX_HIP(hipStreamSynchronize(c->stream));
  if (perm_out) std::copy(h_perm.begin(), h_perm.end(), perm_out);
  g->n = g->n_raw = new_n;
  g->orient_mode = -1;  // any CSR built before is stale
  return TC_OK;
}

int tc_graph_relabel(tc_ctx* c, tc_graph* g, int mode, uint32_t* perm_out) {
  PoolScope scope(c);
  TCX_TRY(check_records(g));
  if (c != g->ctx) return fail(TC_ERR_ARG, "graph belongs to another context");
  if (mode < TC_RELABEL_COMPACT || mode > TC_RELABEL_ADIR)
    return fail(TC_ERR_ARG, "unknown relabel mode %d", mode);
  const uint64_t m = g->m_raw;
  uint32_t* s = g->src.as<uint32_t>();
  uint32_t* d = g->dst.as<uint32_t>();
  uint32_t n = 1;  // max id + 1 over the records, as the tools compute it
  if (m) {
    uint32_t mx = 0;
    TCX_TRY(max_ids(c, s, d, m, &mx));
    n = mx + 1;
  }
  DevBuf deg, perm, key, ktmp, ids, itmp;
  TCX_TRY(perm.reserve(4ull * n));
  uint32_t n_new = n;
  if (mode == TC_RELABEL_COMPACT || mode == TC_RELABEL_DEGREE) {
    TCX_TRY(deg.reserve(4ull * n));
    hipLaunchKernelGGL(k_fill_u32, dim3(grid_for(n)), dim3(TB), 0, c->stream,
                       deg.as<uint32_t>(), 0u, (uint64_t)n);
    TCX_TRY(count_ids(c, s, d, m, n, deg.as<uint32_t>()));
  }
  if (mode == TC_RELABEL_COMPACT) {
    // new id = number of present ids below (tools/serialize.cpp:32-44)
    DevBuf flags;
    TCX_TRY(flags.reserve(4ull * n));
    hipLaunchKernelGGL(k_present_flags, dim3(grid_for(n)), dim3(TB), 0, c->stream,
                       deg.as<uint32_t>(), n, flags.as<uint32_t>());
    TCX_TRY(exclusive_scan_u32(c, flags.as<uint32_t>(), perm.as<uint32_t>(), n));
    uint32_t last_perm = 0, last_flag = 0;
    TCX_TRY(read_u32(c, perm.as<uint32_t>() + n - 1, &last_perm));
    TCX_TRY(read_u32(c, flags.as<uint32_t>() + n - 1, &last_flag));
    n_new = m ? last_perm + last_flag : 1;
  } else {
    TCX_TRY(key.reserve(8ull * n));
    TCX_TRY(ktmp.reserve(8ull * n));
    TCX_TRY(ids.reserve(4ull * n));
    TCX_TRY(itmp.reserve(4ull * n));
    if (mode == TC_RELABEL_ADIR) {
      // peel the simple symmetric graph over the tools' n = max id + 1
      DevBuf skeys_buf, stmp, srp, scol, prio, rec;
      uint64_t* skeys = nullptr;
      uint64_t m2 = 0;
      TCX_TRY(sym_keys(c, g, skeys_buf, stmp, &skeys, &m2));
      TCX_TRY(sym_csr(c, skeys, m2, n, srp, scol));
      TCX_TRY(prio.reserve(4ull * n));
      TCX_TRY(rec.reserve(4ull * n));
      TCX_TRY(adir_peel(c, n, m2, srp.as<uint32_t>(), scol.as<uint32_t>(), prio.as<int32_t>(),
                        rec.as<int32_t>()));
      hipLaunchKernelGGL(k_adir_relabel_keys, dim3(grid_for(n)), dim3(TB), 0, c->stream,
                         prio.as<int32_t>(), rec.as<int32_t>(), n, key.as<uint64_t>(),
                         ids.as<uint32_t>());
    } else if (mode == TC_RELABEL_FIRST_SRC) {
      DevBuf first;
      TCX_TRY(first.reserve(8ull * n));
      hipLaunchKernelGGL(k_fill_u64, dim3(grid_for(n)), dim3(TB), 0, c->stream,
                         first.as<uint64_t>(), ~0ull, (uint64_t)n);
      if (m)
        hipLaunchKernelGGL(k_first_src, dim3(grid_for(m)), dim3(TB), 0, c->stream, s, m,
                           first.as<unsigned long long>());
      hipLaunchKernelGGL(k_first_keys, dim3(grid_for(n)), dim3(TB), 0, c->stream,
                         first.as<uint64_t>(), n, m, key.as<uint64_t>(), ids.as<uint32_t>());
    } else {
      hipLaunchKernelGGL(k_degree_keys, dim3(grid_for(n)), dim3(TB), 0, c->stream,
                         deg.as<uint32_t>(), n, key.as<uint64_t>(), ids.as<uint32_t>());
    }
    TCX_HIP(hipGetLastError());
    uint64_t* sk;
    uint32_t* order;
    TCX_TRY(sort_pairs_u64_u32(c, key.as<uint64_t>(), ktmp.as<uint64_t>(), ids.as<uint32_t>(),
                               itmp.as<uint32_t>(), n, 64, &sk, &order));
    hipLaunchKernelGGL(k_rank_perm, dim3(grid_for(n)), dim3(TB), 0, c->stream, order, n,
                       mode == TC_RELABEL_DEGREE || mode == TC_RELABEL_ADIR, perm.as<uint32_t>());
  }
  if (m)
    hipLaunchKernelGGL(k_apply_perm, dim3(grid_for(m)), dim3(TB), 0, c->stream, s, d, m,
                       perm.as<uint32_t>());
  TCX_HIP(hipGetLastError());
  if (perm_out)
    TCX_HIP(hipMemcpyAsync(perm_out, perm.p, 4ull * n, hipMemcpyDeviceToHost, c->stream));
  TCX_HIP(hipStreamSynchronize(c->stream));
  g->n = g->n_raw = n_new;
  g->orient_mode = -1;  // any CSR built before is stale
  return TC_OK;
}

static int orient_peeled(tc_ctx* c, tc_graph* g, int mode, double thre_param, int tie);
static int orient_impl(tc_ctx* c, tc_graph* g, int mode, uint32_t flags, int tie);

int tc_graph_orient(tc_ctx* c, tc_graph* g, int mode, uint32_t flags) {
  PoolScope scope(c);
  TCX_TRY(check_records(g));
  if (c != g->ctx) return fail(TC_ERR_ARG, "graph belongs to another context");
  if (mode < TC_ORIENT_ID || mode > TC_ORIENT_DEGENERACY)
    return fail(TC_ERR_ARG, "unknown orientation mode %d", mode);
  if ((flags & TC_FLAG_PRUNE_DEG1) && mode != TC_ORIENT_DEGREE)
    return fail(TC_ERR_ARG, "degree<=1 pruning applies to TC_ORIENT_DEGREE only");
  return orient_impl(c, g, mode, flags, TC_TIE_ID);
}

int tc_graph_orient_ties(tc_ctx* c, tc_graph* g, int mode, int tie) {
  PoolScope scope(c);
  TCX_TRY(check_records(g));
  if (c != g->ctx) return fail(TC_ERR_ARG, "graph belongs to another context");
  if (mode != TC_ORIENT_ADIR && mode != TC_ORIENT_DEGREE)
    return fail(TC_ERR_ARG, "tie rules apply to TC_ORIENT_ADIR and TC_ORIENT_DEGREE");
  if (tie < TC_TIE_ID || tie > TC_TIE_FORCED_DESC) return fail(TC_ERR_ARG, "unknown tie rule %d", tie);
  return orient_impl(c, g, mode, 0, tie);
}

int tc_graph_adir_cost(tc_ctx* c, tc_graph* g, double* cost) {
  PoolScope scope(c);
  if (!c || !g || !cost) return fail(TC_ERR_ARG, "NULL argument");
  if (c != g->ctx) return fail(TC_ERR_ARG, "graph belongs to another context");
  if (g->orient_mode < 0) return fail(TC_ERR_STATE, "graph must be oriented");
  TCX_HIP(hipSetDevice(c->device));
  *cost = 0;
  if (g->n == 0) return TC_OK;
  constexpr unsigned kGrid = 1024;
  DevBuf part;
  TCX_TRY(part.reserve(8 * kGrid));
  const double avg = (double)g->m_or / (double)g->n;
  hipLaunchKernelGGL(k_adir_cost, dim3(kGrid), dim3(256), 0, c->stream, g->rowptr.as<uint32_t>(),
                     g->n, avg, part.as<double>());
  TCX_HIP(hipGetLastError());
  std::vector<double> h(kGrid);
  TCX_HIP(hipMemcpyAsync(h.data(), part.p, 8 * kGrid, hipMemcpyDeviceToHost, c->stream));
  TCX_HIP(hipStreamSynchronize(c->stream));
  double sum = 0;
  for (double x : h) sum += x;
  *cost = sum;
  return TC_OK;
}

static int orient_impl(tc_ctx* c, tc_graph* g, int mode, uint32_t flags, int tie) {
  // Every pass over the raw records uses their id range; only a pruned CSR
  // has fewer rows.
  const uint32_t n = g->n_raw;
  const uint64_t m = g->m_raw;
  if (mode == TC_ORIENT_ID || mode == TC_ORIENT_DEGREE || mode == TC_ORIENT_DEGREE_TRICORE) {
    DevBuf deg, pruned, keys, tmp;
    TCX_TRY(deg.reserve(4 * ((size_t)n + 1)));
    TCX_TRY(keys.reserve(8 * std::max<uint64_t>(m, 1)));
    TCX_TRY(tmp.reserve(8 * std::max<uint64_t>(m, 1)));
    hipLaunchKernelGGL(k_fill_u32, dim3(grid_for(n + 1)), dim3(TB), 0, c->stream,
                       deg.as<uint32_t>(), 0u, (uint64_t)n + 1);
    if (mode != TC_ORIENT_ID)
      TCX_TRY(count_ids(c, g->src.as<uint32_t>(), g->dst.as<uint32_t>(), m, n, deg.as<uint32_t>()));
    TCX_HIP(hipGetLastError());
    uint32_t n_out = n;
    const uint32_t* pruned_before = nullptr;
    DevBuf tkey;
    if (tie != TC_TIE_ID) {
      TCX_TRY(tkey.reserve(4 * ((size_t)n + 1)));
      hipLaunchKernelGGL(k_fill_u32, dim3(grid_for(n + 1)), dim3(TB), 0, c->stream,
                         tkey.as<uint32_t>(), 0u, (uint64_t)n + 1);
      hipLaunchKernelGGL(k_forced_raw, dim3(grid_for(m)), dim3(TB), 0, c->stream,
                         g->src.as<uint32_t>(), g->dst.as<uint32_t>(), m, deg.as<uint32_t>(),
                         tkey.as<uint32_t>());
      if (tie == TC_TIE_FORCED_DESC)
        hipLaunchKernelGGL(k_tie_flip, dim3(grid_for(n)), dim3(TB), 0, c->stream,
                           tkey.as<uint32_t>(), n);
      TCX_HIP(hipGetLastError());
    }
    if (flags & TC_FLAG_PRUNE_DEG1) {
      DevBuf flag;
      TCX_TRY(flag.reserve(4 * ((size_t)n + 1)));
      TCX_TRY(pruned.reserve(4 * ((size_t)n + 1)));
      hipLaunchKernelGGL(k_low_degree_flag, dim3(grid_for(n)), dim3(TB), 0, c->stream,
                         deg.as<uint32_t>(), n, flag.as<uint32_t>());
      TCX_HIP(hipGetLastError());
      TCX_TRY(exclusive_scan_u32(c, flag.as<uint32_t>(), pruned.as<uint32_t>(), n));
      uint32_t lastp = 0, lastf = 0;
      if (n) {
        TCX_TRY(read_u32(c, pruned.as<uint32_t>() + n - 1, &lastp));
        TCX_TRY(read_u32(c, flag.as<uint32_t>() + n - 1, &lastf));
      }
      n_out = n - (lastp + lastf);
      pruned_before = pruned.as<uint32_t>();
      TCX_HIP(hipStreamSynchronize(c->stream));
    }
    hipLaunchKernelGGL(k_orient_keys, dim3(grid_for(m)), dim3(TB), 0, c->stream,
                       g->src.as<uint32_t>(), g->dst.as<uint32_t>(), m, deg.as<uint32_t>(), mode,
                       pruned_before, n_out, tie != TC_TIE_ID ? tkey.as<uint32_t>() : nullptr,
                       key_shift(m, n_out), keys.as<uint64_t>());
    TCX_HIP(hipGetLastError());
    TCX_TRY(csr_from_keys(c, g, keys, tmp, m, n_out, false, key_shift(m, n_out)));
    g->orient_mode = mode;
    if (mode != TC_ORIENT_ID && n_out == n) {  // the raw degrees stay with the graph
      swap(g->vdeg, deg);
      g->vdeg_version = g->sched_version;
    }
    return TC_OK;
  }
  return orient_peeled(c, g, mode, 0, tie);
}

// A-direction / k-core: peel the simple symmetric graph, then keep the
// symmetric entries that point up the peel order.
static int orient_peeled(tc_ctx* c, tc_graph* g, int mode, double thre_param, int tie) {
  const uint32_t n = g->n_raw;
  DevBuf keys, tmp, srp, scol, keep;
  uint64_t* skeys = nullptr;
  uint64_t m2 = 0;
  TCX_TRY(sym_keys(c, g, keys, tmp, &skeys, &m2));
  TCX_TRY(sym_csr(c, skeys, m2, n, srp, scol));
  TCX_TRY(g->vkey.reserve(4 * ((size_t)n + 1)));
  if (n > 0) {
    if (mode == TC_ORIENT_ADIR || mode == TC_ORIENT_ADIR_OMP) {
      TCX_TRY(adir_peel(c, n, m2, srp.as<uint32_t>(), scol.as<uint32_t>(), g->vkey.as<int32_t>(),
                        nullptr, mode == TC_ORIENT_ADIR_OMP ? thre_param : 0));
    } else if (mode == TC_ORIENT_KCORE) {
      TCX_TRY(kcore_peel(c, n, m2, srp.as<uint32_t>(), scol.as<uint32_t>(), g->vkey.as<int32_t>()));
    } else {
      DevBuf core;
      TCX_TRY(core.reserve(4 * ((size_t)n + 1)));
      TCX_TRY(kcore_peel(c, n, m2, srp.as<uint32_t>(), scol.as<uint32_t>(), core.as<int32_t>(),
                         g->vkey.as<int32_t>()));
    }
  }
  DevBuf tkey;
  if (tie != TC_TIE_ID && n > 0) {
    TCX_TRY(tkey.reserve(4 * ((size_t)n + 1)));
    hipLaunchKernelGGL(k_forced_sym, dim3(grid_for(n)), dim3(TB), 0, c->stream,
                       srp.as<uint32_t>(), scol.as<uint32_t>(), n, g->vkey.as<int32_t>(),
                       tie == TC_TIE_FORCED_DESC ? 1 : 0, tkey.as<uint32_t>());
    TCX_HIP(hipGetLastError());
  }
  TCX_TRY(keep.reserve(std::max<uint64_t>(m2, 1)));
  hipLaunchKernelGGL(k_sym_keep, dim3(grid_for(m2)), dim3(TB), 0, c->stream, skeys, m2,
                     g->vkey.as<int32_t>(), mode, tkey.p ? tkey.as<uint32_t>() : nullptr,
                     keep.as<uint8_t>());
  TCX_HIP(hipGetLastError());
  uint64_t* dst_keys = skeys == keys.as<uint64_t>() ? tmp.as<uint64_t>() : keys.as<uint64_t>();
  uint64_t mo = 0;
  TCX_TRY(select_flagged_u64(c, skeys, keep.as<uint8_t>(), dst_keys, m2, &mo));
  DevBuf* holder = dst_keys == keys.as<uint64_t>() ? &keys : &tmp;
  DevBuf* spare = holder == &keys ? &tmp : &keys;
  TCX_TRY(csr_from_keys(c, g, *holder, *spare, mo, n, true));
  g->orient_mode = mode;
  TCX_TRY(g->vdeg.reserve(4 * ((size_t)n + 1)));
  hipLaunchKernelGGL(k_row_degrees, dim3(grid_for(n)), dim3(TB), 0, c->stream, srp.as<uint32_t>(),
                     n, g->vdeg.as<uint32_t>());
  TCX_HIP(hipGetLastError());
  g->vdeg_version = g->sched_version;
  return TC_OK;
}

int tc_graph_orient_adir_omp(tc_ctx* c, tc_graph* g, double thre_param) {
  PoolScope scope(c);
  TCX_TRY(check_records(g));
  if (c != g->ctx) return fail(TC_ERR_ARG, "graph belongs to another context");
  if (!(thre_param > 0) || !std::isfinite(thre_param))
    return fail(TC_ERR_ARG, "thre_param must be finite and positive (the threshold never grows "
                            "otherwise)");
  return orient_peeled(c, g, TC_ORIENT_ADIR_OMP, thre_param, TC_TIE_ID);
}

// Stage file of an oriented CSR: "TCAMDCSR", uint32 version 1, uint32 n,
// uint64 m, int32 orientation, uint32 has_key, rowptr[n+1], col[m] (uint32),
// then key[n] (int32) when has_key; little endian.
namespace {
struct CsrFileHeader {
  char magic[8];
  uint32_t version, n;
  uint64_t m;
  int32_t orient_mode;
  uint32_t has_key;
};
static_assert(sizeof(CsrFileHeader) == 32, "stage file header is 32 bytes");
constexpr char kCsrMagic[8] = {'T', 'C', 'A', 'M', 'D', 'C', 'S', 'R'};

bool has_vertex_key(int mode) {
  return mode == TC_ORIENT_ADIR || mode == TC_ORIENT_KCORE || mode == TC_ORIENT_DEGENERACY ||
         mode == TC_ORIENT_ADIR_OMP;
}
}  // namespace

int tc_graph_save_csr(const tc_graph* g, const char* path) {
  if (!g || !g->ctx || !path) return fail(TC_ERR_ARG, "NULL argument");
  if (g->orient_mode < 0) return fail(TC_ERR_STATE, "graph not oriented");
  const uint32_t n = g->n;
  const uint64_t m = g->m_or;
  std::vector<uint32_t> rp((size_t)n + 1), col(std::max<uint64_t>(m, 1));
  std::vector<int32_t> key;
  const bool wk = has_vertex_key(g->orient_mode);
  TCX_TRY(tc_graph_get_csr(g, rp.data(), col.data()));
  if (wk && n) {
    key.resize(n);
    TCX_TRY(tc_graph_get_vertex_key(g, key.data()));
  }
  CsrFileHeader h;
  memcpy(h.magic, kCsrMagic, 8);
  h.version = 1;
  h.n = n;
  h.m = m;
  h.orient_mode = g->orient_mode;
  h.has_key = wk ? 1u : 0u;
  FILE* f = fopen(path, "wb");
  if (!f) return fail(TC_ERR_IO, "cannot open %s for writing", path);
  bool ok = fwrite(&h, sizeof(h), 1, f) == 1 &&
            fwrite(rp.data(), 4, (size_t)n + 1, f) == (size_t)n + 1 &&
            (m == 0 || fwrite(col.data(), 4, m, f) == m) &&
            (!wk || n == 0 || fwrite(key.data(), 4, n, f) == n);
  ok = (fclose(f) == 0) && ok;
  if (!ok) return fail(TC_ERR_IO, "write to %s failed", path);
  return TC_OK;
}

int tc_graph_load_csr(tc_ctx* c, const char* path, tc_graph** out) {
  PoolScope scope(c);
  if (!c || !path || !out) return fail(TC_ERR_ARG, "NULL argument");
  *out = nullptr;
  FILE* f = fopen(path, "rb");
  if (!f) return fail(TC_ERR_IO, "cannot open %s", path);
  CsrFileHeader h;
  if (fread(&h, sizeof(h), 1, f) != 1 || memcmp(h.magic, kCsrMagic, 8) != 0 || h.version != 1 ||
      h.orient_mode < TC_ORIENT_ID || h.orient_mode > TC_ORIENT_ADIR_OMP ||
      h.has_key != (has_vertex_key(h.orient_mode) ? 1u : 0u) || h.n > 0x7FFFFFFEu ||
      h.m > kMaxCsrEntries) {
    fclose(f);
    return fail(TC_ERR_FORMAT, "%s is not an oriented-CSR stage file", path);
  }
  const uint32_t n = h.n;
  const uint64_t m = h.m;
  std::vector<uint32_t> rp((size_t)n + 1), col(std::max<uint64_t>(m, 1));
  std::vector<int32_t> key(h.has_key ? std::max<uint32_t>(n, 1) : 0);
  bool ok = fread(rp.data(), 4, (size_t)n + 1, f) == (size_t)n + 1 &&
            (m == 0 || fread(col.data(), 4, m, f) == m) &&
            (!h.has_key || n == 0 || fread(key.data(), 4, n, f) == n);
  char extra;
  ok = ok && fread(&extra, 1, 1, f) == 0;  // nothing after the arrays
  fclose(f);
  if (!ok) return fail(TC_ERR_FORMAT, "%s is truncated or has trailing bytes", path);
  // the kernels index rp[col[e] + 1]: every structural property is checked
  if (rp[0] != 0 || rp[n] != m) return fail(TC_ERR_FORMAT, "%s: row offsets do not span m", path);
  std::vector<uint32_t> esrc(std::max<uint64_t>(m, 1));
  for (uint32_t v = 0; v < n; ++v) {
    if (rp[v + 1] < rp[v] || rp[v + 1] > m)
      return fail(TC_ERR_FORMAT, "%s: row offsets decrease at or after %u", path, v);
    for (uint32_t e = rp[v]; e < rp[v + 1]; ++e) {
      if (col[e] >= n || col[e] == v || (e > rp[v] && col[e] <= col[e - 1]))
        return fail(TC_ERR_FORMAT, "%s: row %u is not ascending, loop-free and in range", path, v);
      esrc[e] = v;
    }
  }
  TCX_HIP(hipSetDevice(c->device));
  tc_graph* g = new tc_graph();
  g->ctx = c;
  g->n = g->n_raw = n;
  g->csr_only = true;
  g->m_or = m;
  int st = g->rowptr.reserve(4 * ((size_t)n + 1));
  if (st == TC_OK) st = g->col.reserve(4 * std::max<uint64_t>(m, 1));
  if (st == TC_OK) st = g->esrc.reserve(4 * std::max<uint64_t>(m, 1));
  if (st == TC_OK && h.has_key) st = g->vkey.reserve(4 * ((size_t)n + 1));
  if (st == TC_OK &&
      (hipMemcpyAsync(g->rowptr.p, rp.data(), 4 * ((size_t)n + 1), hipMemcpyHostToDevice,
                      c->stream) != hipSuccess ||
       (m && hipMemcpyAsync(g->col.p, col.data(), 4 * m, hipMemcpyHostToDevice, c->stream) !=
                 hipSuccess) ||
       (m && hipMemcpyAsync(g->esrc.p, esrc.data(), 4 * m, hipMemcpyHostToDevice, c->stream) !=
                 hipSuccess) ||
       (h.has_key && n &&
        hipMemcpyAsync(g->vkey.p, key.data(), 4 * (size_t)n, hipMemcpyHostToDevice, c->stream) !=
            hipSuccess)))
    st = fail(TC_ERR_HIP, "stage file upload failed");
  if (st == TC_OK && hipStreamSynchronize(c->stream) != hipSuccess)
    st = fail(TC_ERR_HIP, "stage file upload failed");
  if (st == TC_OK) {
    g->orient_mode = h.orient_mode;
    g->sched_version++;
    st = compute_csr_stats(c, g);
  }
  if (st != TC_OK) {
    delete g;
    return st;
  }
  *out = g;
  return TC_OK;
}

int tc_graph_info_get(const tc_graph* g, tc_graph_info* info) {
  if (!g || !info) return fail(TC_ERR_ARG, "NULL argument");
  info->n = g->n;
  info->max_out_degree = g->max_out;
  info->m_raw = g->m_raw;
  info->m_oriented = g->orient_mode >= 0 ? g->m_or : 0;
  info->orient_mode = g->orient_mode;
  info->n_raw = g->n_raw;
  info->sum_out_sq = g->orient_mode >= 0 ? g->sum_out_sq : 0;
  info->sum_in_out = g->orient_mode >= 0 ? g->sum_in_out : 0;
  double n1 = (double)g->n + 1, mo = (double)info->m_oriented;
  info->bytes_alg = 4 * n1 + 8 * mo + 4.0 * (double)info->sum_out_sq + 4.0 * (double)info->sum_in_out;
  info->bytes_min = 4 * n1 + 4 * mo;
  return TC_OK;
}

int tc_graph_get_csr(const tc_graph* g, uint32_t* rowptr, uint32_t* col) {
  if (!g || !g->ctx) return fail(TC_ERR_ARG, "NULL graph");
  if (g->orient_mode < 0) return fail(TC_ERR_STATE, "graph not oriented");
  TCX_HIP(hipSetDevice(g->ctx->device));
  hipStream_t s = g->ctx->stream;
  if (rowptr)
    TCX_HIP(hipMemcpyAsync(rowptr, g->rowptr.p, 4 * ((size_t)g->n + 1), hipMemcpyDeviceToHost, s));
  if (col && g->m_or)
    TCX_HIP(hipMemcpyAsync(col, g->col.p, 4 * g->m_or, hipMemcpyDeviceToHost, s));
  TCX_HIP(hipStreamSynchronize(s));
  return TC_OK;
}

int tc_graph_get_edges(const tc_graph* g, uint32_t* src, uint32_t* dst) {
  if (!g || !g->ctx) return fail(TC_ERR_ARG, "NULL graph");
  TCX_HIP(hipSetDevice(g->ctx->device));
  hipStream_t s = g->ctx->stream;
  if (g->m_raw) {
    if (src) TCX_HIP(hipMemcpyAsync(src, g->src.p, 4 * g->m_raw, hipMemcpyDeviceToHost, s));
    if (dst) TCX_HIP(hipMemcpyAsync(dst, g->dst.p, 4 * g->m_raw, hipMemcpyDeviceToHost, s));
  }
  TCX_HIP(hipStreamSynchronize(s));
  return TC_OK;
}

int tc_graph_get_vertex_key(const tc_graph* g, int32_t* key) {
  if (!g || !g->ctx || !key) return fail(TC_ERR_ARG, "NULL argument");
  if (g->orient_mode != TC_ORIENT_ADIR && g->orient_mode != TC_ORIENT_KCORE &&
      g->orient_mode != TC_ORIENT_DEGENERACY && g->orient_mode != TC_ORIENT_ADIR_OMP)
    return fail(TC_ERR_STATE,
                "vertex keys exist after ADIR, ADIR_OMP, KCORE or DEGENERACY orientation only");
  TCX_HIP(hipSetDevice(g->ctx->device));
  if (g->n)
    TCX_HIP(hipMemcpyAsync(key, g->vkey.p, 4 * (size_t)g->n, hipMemcpyDeviceToHost, g->ctx->stream));
  TCX_HIP(hipStreamSynchronize(g->ctx->stream));
  return TC_OK;
}

int tc_graph_device_csr(const tc_graph* g, const uint32_t** rowptr, const uint32_t** col) {
  if (!g || !rowptr || !col) return fail(TC_ERR_ARG, "NULL argument");
  if (g->orient_mode < 0) return fail(TC_ERR_STATE, "graph not oriented");
  *rowptr = g->rowptr.as<uint32_t>();
  *col = g->col.as<uint32_t>();
  g->exported = true;
  return TC_OK;
}

}  // extern "C"

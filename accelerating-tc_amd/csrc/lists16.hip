// Builds and counts over the 16-bit list layer (lists16.h).
#include "lists16.h"

#include <algorithm>
#include <vector>

#include "internal.h"

namespace tcx {
namespace {

using namespace dev;

constexpr uint32_t kHistBins = 4096;  // degree histogram, the last bin open
// A graph of more than 65,535 vertices takes the layer when kMinShare of its
// entries get a 16-bit id; or, where the average pushed list has kLongList
// entries, when kMinEntries of them do and kMinStream of the entries that the
// push lists stream (sum over edges of the target's row).  Skewed graphs stream
// their hubs' entries most (R-MAT-24: 22 against 44 ms).  With short rows, all
// alike, the tail's work lists and tasks cost more than the layer saves
// (random geometric, 90,000 vertices, average list 17: 116 against 103 us;
// Barabasi-Albert, 10^6 vertices, average list 8, by Hu's method: 680 against
// 323 us over 32-bit rows).  Smaller graphs always take it: 14 against 60-120
// us at 3,001 vertices, 41 against 90 us on ER of 65,536 vertices and 2^20
// edges.
constexpr double kMinShare = 0.85, kMinEntries = 0.4, kMinStream = 0.75;
constexpr uint64_t kLongList = 32;
constexpr int kU32 = 2;             // steps in flight over 32-bit rows
constexpr uint32_t kWg32 = 8;       // workgroups a CU over 32-bit rows
constexpr uint64_t kTaskCost = 48;  // a task's own row and map, in group steps

unsigned grid_for(uint64_t n, int tb = TB) {
  uint64_t b = (n + tb - 1) / tb;
  return (unsigned)std::max<uint64_t>(1, std::min<uint64_t>(b, 1u << 20));
}

__global__ void k_fill16(uint32_t* p, uint32_t v, uint64_t n) {
  for (uint64_t i = gtid(); i < n; i += gstride()) p[i] = v;
}

// hist[min(deg, bins - 1)] += 1, and the degree sum of the open bin
__global__ __launch_bounds__(TB) void k_deg_hist(const uint32_t* __restrict__ deg, uint32_t n,
                                                   uint32_t* __restrict__ hist,
                                                   unsigned long long* open_sum) {
  __shared__ uint32_t h[kHistBins];
  for (uint32_t i = threadIdx.x; i < kHistBins; i += TB) h[i] = 0;
  __syncthreads();
  unsigned long long s = 0;
  for (uint64_t v = gtid(); v < n; v += gstride()) {
    const uint32_t d = deg[v];
    if (d >= kHistBins - 1) s += d;
    atomicAdd(h + min(d, kHistBins - 1), 1u);
  }
  __syncthreads();
  for (uint32_t i = threadIdx.x; i < kHistBins; i += TB)
    if (h[i]) atomicAdd(hist + i, h[i]);
  flush_count(s, open_sum);
}

__global__ void k_hub_flags(const uint32_t* __restrict__ deg, uint32_t n, uint32_t t,
                            uint32_t* __restrict__ f) {
  for (uint64_t v = gtid(); v < n; v += gstride()) f[v] = deg[v] >= t ? 1u : 0u;
}

__global__ void k_hub_ids(const uint32_t* __restrict__ deg, const uint32_t* __restrict__ pos,
                          uint32_t n, uint32_t t, uint16_t* __restrict__ id) {
  for (uint64_t v = gtid(); v < n; v += gstride())
    id[v] = deg[v] >= t ? (uint16_t)pos[v] : (uint16_t)kPad16;
}

// f[e] = 1 where the entry has a 16-bit id; f[m] = 0
__global__ void k_entry_flags(const uint32_t* __restrict__ col, uint64_t m,
                              const uint16_t* __restrict__ id, uint32_t* __restrict__ f) {
  for (uint64_t e = gtid(); e <= m; e += gstride())
    f[e] = e < m && id[col[e]] != kPad16 ? 1u : 0u;
}

// Rows are laid out so that none touches a cache line more than its length
// needs: rows above four units start on a 128-byte line, shorter ones are
// grouped by their size rounded up to 1, 2 or 4 units (lists average a few
// lines: with rows packed one after the other R-MAT-22, A-ordered, moved 28.0
// instead of 25.5 GB a count, in 3.80 instead of 3.57 ms).  A row's place is the number of
// rows, or of 8-unit lines, before it in its class; the four counters ride
// in two 64-bit scans.
struct Place16 {
  uint64_t a, b;  // (lines of the 8-unit class, rows of 4), (rows of 2, rows of 1)
};

__device__ inline Place16 place16(uint32_t units) {
  if (units > 4) return {(uint64_t)((units + 7) / 8) << 32, 0ull};
  if (units > 2) return {1ull, 0ull};
  return units == 2 ? Place16{0ull, 1ull << 32} : Place16{0ull, units ? 1ull : 0ull};
}

// First unit of a row from its place and the classes' totals t.
__device__ inline uint32_t start16(uint32_t units, Place16 p, Place16 t) {
  const uint32_t base4 = (uint32_t)(t.a >> 32) * 8u, base2 = base4 + (uint32_t)t.a * 4u,
                 base1 = base2 + (uint32_t)(t.b >> 32) * 2u;
  if (units > 4) return (uint32_t)(p.a >> 32) * 8u;
  if (units > 2) return base4 + (uint32_t)p.a * 4u;
  return units == 2 ? base2 + (uint32_t)(p.b >> 32) * 2u : base1 + (uint32_t)p.b;
}

// Entries of each row with (cnt) and without (tcnt) a 16-bit id, from the
// prefix `pre` of k_entry_flags (null: all of them have one).
__global__ void k_counts16(const uint32_t* __restrict__ rp, const uint32_t* __restrict__ pre,
                           uint32_t n, uint32_t* __restrict__ cnt, uint32_t* __restrict__ tcnt) {
  for (uint64_t u = gtid(); u < n; u += gstride()) {
    const uint32_t b = rp[u], e = rp[u + 1], c = pre ? pre[e] - pre[b] : e - b;
    cnt[u] = c;
    if (tcnt) tcnt[u] = e - b - c;
  }
}

// *sum += the 16-bit entries that the push lists stream
__global__ __launch_bounds__(TB) void k_streamed(const uint32_t* __restrict__ col, uint64_t m,
                                                 const uint32_t* __restrict__ cnt,
                                                 unsigned long long* sum) {
  __shared__ unsigned long long red[TB / 64];
  unsigned long long s = 0;
  for (uint64_t e = gtid(); e < m; e += gstride()) s += cnt[col[e]];
  flush_block(s, sum, red);
}

// The rows' class counters (n + 1 entries), per entries to a unit.
__global__ void k_places16(const uint32_t* __restrict__ cnt, uint32_t n, uint32_t per,
                           uint64_t* __restrict__ pa, uint64_t* __restrict__ pb) {
  for (uint64_t u = gtid(); u <= n; u += gstride()) {
    const Place16 p = place16(u < n ? (cnt[u] + per - 1) / per : 0u);
    pa[u] = p.a;
    pb[u] = p.b;
  }
}

__global__ void k_row_pairs(const uint32_t* __restrict__ cnt, const uint64_t* __restrict__ pa,
                            const uint64_t* __restrict__ pb, uint32_t n, uint32_t per,
                            uint2* __restrict__ row) {
  const Place16 t{pa[n], pb[n]};
  for (uint64_t u = gtid(); u < n; u += gstride()) {
    const uint32_t units = (cnt[u] + per - 1) / per;
    row[u] = make_uint2(start16(units, Place16{pa[u], pb[u]}, t), units);
  }
}

__global__ void k_scatter16(const uint32_t* __restrict__ rp, const uint32_t* __restrict__ col,
                            const uint32_t* __restrict__ esrc, uint64_t m,
                            const uint16_t* __restrict__ id, const uint32_t* __restrict__ pre,
                            const uint2* __restrict__ row, uint16_t* __restrict__ col16,
                            const uint2* __restrict__ trow, uint32_t* __restrict__ tcol) {
  for (uint64_t e = gtid(); e < m; e += gstride()) {
    const uint32_t u = esrc[e], v = col[e], b = rp[u];
    const uint32_t h = id ? id[v] : v;
    const uint32_t p = pre ? pre[e] : (uint32_t)e, pb = pre ? pre[b] : b;
    if (h != kPad16) col16[8ull * row[u].x + (p - pb)] = (uint16_t)h;
    else tcol[4ull * trow[u].x + ((uint32_t)e - b - (p - pb))] = v;
  }
}

constexpr uint32_t kInEdge = 0x80000000u;  // key flag: the owner is the edge's target

// Work-list key (owner << 32 | streamed) of every edge u -> v: the end with
// the longer row (cnt entries) owns it, u on a tie; no key ((n << 32), sorted
// last) when either row is empty, or the owner u's only entry is v itself.
// id: the 16-bit ids (null: every vertex has one); tail: rows of the entries
// without one.
__global__ void k_keys16(const uint32_t* __restrict__ esrc, const uint32_t* __restrict__ col,
                         uint64_t m, uint32_t n, const uint32_t* __restrict__ cnt,
                         const uint16_t* __restrict__ id, bool tail, uint64_t* __restrict__ key,
                         uint8_t* __restrict__ flag) {
  for (uint64_t e = gtid(); e < m; e += gstride()) {
    const uint32_t u = esrc[e], v = col[e], cu = cnt[u], cv = cnt[v];
    uint64_t k = (uint64_t)n << 32;
    if (cu && cv) {
      if (cv > cu) k = ((uint64_t)v << 32) | u | kInEdge;
      else if (cu > 1 || (id && id[v] == kPad16) != tail) k = ((uint64_t)u << 32) | v;
    }
    key[e] = k;
    if (flag) flag[e] = k != (uint64_t)n << 32;
  }
}

// se[i] = row of the streamed list of sorted key i; cred[i] (optional) = whom a
// per-vertex count credits it to (lists16.h); cost[owner] += its group
// steps, summed over each wave's runs of one owner before the atomic.
__global__ __launch_bounds__(TB) void k_entries16(const uint64_t* __restrict__ key, uint64_t E,
                                                  const uint2* __restrict__ row,
                                                  uint2* __restrict__ se,
                                                  uint32_t* __restrict__ cred,
                                                  unsigned long long* __restrict__ cost) {
  const uint32_t lane = threadIdx.x & 63;
  for (uint64_t b = gtid() & ~63ull; b < E; b += gstride()) {
    const uint64_t i = b + lane;
    uint32_t o = 0xFFFFFFFFu, st = 0;
    if (i < E) {
      const uint64_t k = key[i];
      const uint32_t y = (uint32_t)k & ~kInEdge;
      const uint2 r = row[y];
      se[i] = r;
      if (cred) cred[i] = (uint32_t)k & kInEdge ? y : kEmpty;
      o = (uint32_t)(k >> 32);
      st = (r.y + kGroup16 - 1) / kGroup16;
    }
    const uint32_t incl = wave_incl_scan_dpp(st);
    const uint32_t prev = (uint32_t)__shfl_up((int)o, 1, 64), next = (uint32_t)__shfl_down((int)o, 1, 64);
    const uint64_t heads = lanes(lane == 0 || o != prev);
    const uint32_t h = 63u - (uint32_t)__builtin_clzll(heads & (~0ull >> (63 - lane)));
    const uint32_t before = (uint32_t)__shfl((int)(incl - st), (int)h, 64);
    if (i < E && (lane == 63 || o != next))
      atomicAdd(cost + o, (unsigned long long)(incl - before));
  }
}

__global__ void k_nonempty(const uint32_t* __restrict__ wrp, uint32_t n, uint8_t* __restrict__ f) {
  for (uint64_t x = gtid(); x < n; x += gstride()) f[x] = wrp[x + 1] > wrp[x] ? 1 : 0;
}

// act[i] of k_count16 for the owners ids[0, nt), one closing entry after them
__global__ void k_tasks16(const uint32_t* __restrict__ ids, uint32_t nt,
                          const uint32_t* __restrict__ wrp, const uint2* __restrict__ row,
                          const unsigned long long* __restrict__ cost, uint4* __restrict__ act,
                          uint64_t* __restrict__ work) {
  for (uint64_t i = gtid(); i <= nt; i += gstride()) {
    if (i == nt) {
      const uint32_t end = wrp[ids[nt - 1] + 1];
      act[i] = make_uint4(end, end, 0u, 0u);
      work[i] = 0;
      continue;
    }
    const uint32_t x = ids[i];
    const uint2 r = row[x];
    act[i] = make_uint4(wrp[x], wrp[x + 1], r.x, r.y);
    work[i] = cost[x] + kTaskCost;
  }
}

// slice[s] = the (task, entry) at s / ns of the total work; a task's work is
// taken as spread evenly over its entries.
__global__ void k_slices16(const uint64_t* __restrict__ pre, const uint4* __restrict__ act,
                           uint32_t nt, uint64_t E, uint32_t ns, uint2* __restrict__ slice) {
  const uint64_t total = pre[nt];
  for (uint64_t s = gtid(); s <= ns; s += gstride()) {
    if (s == ns) {
      slice[s] = make_uint2(nt, (uint32_t)E);
      continue;
    }
    const uint64_t t = (uint64_t)((double)total * (double)s / (double)ns);
    uint32_t lo = 0, hi = nt - 1;  // last task with pre[task] <= t
    while (lo < hi) {
      const uint32_t mid = (lo + hi + 1) >> 1;
      if (pre[mid] <= t) lo = mid;
      else hi = mid - 1;
    }
    const uint4 a = act[lo];
    const double f = (double)(t - pre[lo]) / (double)(pre[lo + 1] - pre[lo]);
    const uint32_t off = min(a.y - a.x - 1, (uint32_t)((double)(a.y - a.x) * f));
    slice[s] = make_uint2(lo, a.x + off);
  }
}

__global__ void k_local_ids(const uint32_t* __restrict__ gid, const uint32_t* __restrict__ voff,
                            uint32_t n, uint16_t* __restrict__ id) {
  for (uint64_t v = gtid(); v < n; v += gstride()) id[v] = (uint16_t)(v - voff[gid[v]]);
}

__global__ void k_graph_of(uint32_t* __restrict__ who, uint64_t nt,
                           const uint32_t* __restrict__ gid) {
  for (uint64_t i = gtid(); i < nt; i += gstride()) who[i] = gid[who[i]];
}

// The push lists of Hu's method: owner u streams the rows of its out-edges'
// targets, in CSR order.
__global__ void k_push16(const uint32_t* __restrict__ col, uint64_t m,
                         const uint2* __restrict__ row, uint2* __restrict__ se) {
  for (uint64_t e = gtid(); e < m; e += gstride()) se[e] = row[col[e]];
}

__global__ void k_push_flags(const uint32_t* __restrict__ rp, const uint2* __restrict__ row,
                             uint32_t n, uint8_t* __restrict__ f) {
  for (uint64_t u = gtid(); u < n; u += gstride()) f[u] = rp[u + 1] - rp[u] >= 2 && row[u].y ? 1 : 0;
}

__global__ void k_push_tasks(const uint32_t* __restrict__ ids, uint32_t nt,
                             const uint32_t* __restrict__ rp, const uint2* __restrict__ row,
                             uint32_t m, uint4* __restrict__ act) {
  for (uint64_t i = gtid(); i <= nt; i += gstride()) {
    if (i == nt) {
      act[i] = make_uint4(m, m, 0u, 0u);
      continue;
    }
    const uint32_t u = ids[i];
    const uint2 r = row[u];
    act[i] = make_uint4(rp[u], rp[u + 1], r.x, r.y);
  }
}

// slice[s]: vertex block s / parts (start; null: one block of all n vertices),
// its edges cut into `parts`; first task with edges beyond the cut.
__global__ void k_edge_slices(const int32_t* __restrict__ start, uint32_t nblocks, uint32_t parts,
                              uint32_t n, const uint32_t* __restrict__ rp,
                              const uint4* __restrict__ act, uint32_t nt, uint32_t m,
                              uint2* __restrict__ slice) {
  for (uint64_t s = gtid(); s <= (uint64_t)nblocks * parts; s += gstride()) {
    uint32_t at = m;
    if (s < (uint64_t)nblocks * parts) {
      const uint32_t b = start ? rp[start[s / parts]] : 0u;
      const uint32_t e = start ? rp[start[s / parts + 1]] : rp[n];
      at = b + (uint32_t)((uint64_t)(e - b) * (s % parts) / parts);
    }
    uint32_t lo = 0, hi = nt;  // first task that ends beyond the cut
    while (lo < hi) {
      const uint32_t mid = (lo + hi) >> 1;
      if (act[mid].y > at) hi = mid;
      else lo = mid + 1;
    }
    slice[s] = make_uint2(lo, max(at, act[lo].x));
  }
}

// Every entry as a 32-bit one (rows of graphs that the 16-bit ids do not suit)
__global__ void k_scatter32(const uint32_t* __restrict__ rp, const uint32_t* __restrict__ col,
                            const uint32_t* __restrict__ esrc, uint64_t m,
                            const uint2* __restrict__ row, uint32_t* __restrict__ out) {
  for (uint64_t e = gtid(); e < m; e += gstride()) {
    const uint32_t u = esrc[e];
    out[4ull * row[u].x + ((uint32_t)e - rp[u])] = col[e];
  }
}

template <class T>
int read_back(tc_ctx* c, const void* src, T* out) {
  return fetch(c, out, src, sizeof(T));
}

// 16-bit ids by degree (in skewed graphs the in-degree follows it: R-MAT-21 has
// 0.928 of its entries among the 65,535 vertices of largest degree, 0.929 among
// those of largest in-degree): the vertices of degree t and above for the
// smallest t that leaves at most kMax16 of them.  *some: whether they can hold
// enough of the entries (in-degrees are at most the degrees).
int hub_ids(tc_ctx* c, tc_graph* g, DevBuf& id, bool* some) {
  const uint32_t n = g->n;
  *some = false;
  // just above the limit (65,536 vertices) in-degrees decide: the few that are
  // zero need no id, so nothing is left to the tail
  if (n <= kMax16 + 1024) g->vdeg_version = ~0ull;
  TCX_TRY(vertex_degrees(c, g));
  DevBuf hist;
  TCX_TRY(hist.reserve(4 * kHistBins + 8));
  TCX_HIP(hipMemsetAsync(hist.p, 0, 4 * kHistBins + 8, c->stream));
  hipLaunchKernelGGL(k_deg_hist, dim3(std::min<unsigned>(grid_for(n), c->num_cus * 2u)), dim3(TB),
                     0, c->stream, g->vdeg.as<uint32_t>(), n, hist.as<uint32_t>(),
                     reinterpret_cast<unsigned long long*>(hist.as<uint32_t>() + kHistBins));
  TCX_HIP(hipGetLastError());
  struct { uint32_t bin[kHistBins]; unsigned long long open; } h;
  TCX_TRY(read_back(c, hist.p, &h));
  uint64_t have = 0, sum = 0;
  uint32_t t = kHistBins;
  while (t > 1 && have + h.bin[t - 1] <= kMax16) {
    --t;
    have += h.bin[t];
    sum += t == kHistBins - 1 ? h.open : (uint64_t)t * h.bin[t];
  }
  // (t == kHistBins: too many in the open bin)
  const double least = g->sum_in_out >= kLongList * g->m_or ? kMinEntries : kMinShare;
  if (t == kHistBins || (double)sum < least * (double)g->m_or) return TC_OK;
  *some = true;
  DevBuf flag, pos;
  TCX_TRY(flag.reserve(4 * ((size_t)n + 1)));
  TCX_TRY(pos.reserve(4 * ((size_t)n + 1)));
  TCX_TRY(id.reserve(2 * ((size_t)n + 1)));
  hipLaunchKernelGGL(k_hub_flags, dim3(grid_for(n)), dim3(TB), 0, c->stream, g->vdeg.as<uint32_t>(),
                     n, t, flag.as<uint32_t>());
  TCX_TRY(exclusive_scan_u32(c, flag.as<uint32_t>(), pos.as<uint32_t>(), n));
  hipLaunchKernelGGL(k_hub_ids, dim3(grid_for(n)), dim3(TB), 0, c->stream, g->vdeg.as<uint32_t>(),
                     pos.as<uint32_t>(), n, t, id.as<uint16_t>());
  TCX_HIP(hipGetLastError());
  return TC_OK;
}

// Row places for cnt entries a row, `per` to a unit; the entries are padding.
int place_rows(tc_ctx* c, uint32_t n, const uint32_t* cnt, uint32_t per, Rows16& R) {
  DevBuf pa, pb, sa, sb;
  for (DevBuf* b : {&pa, &pb, &sa, &sb}) TCX_TRY(b->reserve(8 * ((size_t)n + 1)));
  hipLaunchKernelGGL(k_places16, dim3(grid_for((uint64_t)n + 1)), dim3(TB), 0, c->stream, cnt, n,
                     per, pa.as<uint64_t>(), pb.as<uint64_t>());
  TCX_TRY(exclusive_scan_u64(c, pa.as<uint64_t>(), sa.as<uint64_t>(), (uint64_t)n + 1));
  TCX_TRY(exclusive_scan_u64(c, pb.as<uint64_t>(), sb.as<uint64_t>(), (uint64_t)n + 1));
  uint64_t ta = 0, tb = 0;
  TCX_TRY(fetch2(c, &ta, sa.as<uint64_t>() + n, &tb, sb.as<uint64_t>() + n));
  R.units = 8 * (ta >> 32) + 4 * (ta & 0xFFFFFFFFu) + 2 * (tb >> 32) + (tb & 0xFFFFFFFFu);
  if (R.units > 0xFFFFFFFFull) return fail(TC_ERR_RANGE, "list rows exceed 2^32 16-byte units");
  TCX_TRY(R.row.reserve(8 * ((size_t)n + 1)));
  TCX_TRY(R.col.reserve(16 * std::max<uint64_t>(R.units, 1)));
  hipLaunchKernelGGL(k_row_pairs, dim3(grid_for(n)), dim3(TB), 0, c->stream, cnt,
                     sa.as<uint64_t>(), sb.as<uint64_t>(), n, per, R.row.as<uint2>());
  hipLaunchKernelGGL(k_fill16, dim3(std::min<unsigned>(grid_for(4 * R.units), 16384)), dim3(TB), 0,
                     c->stream, R.col.as<uint32_t>(), 0xFFFFFFFFu, 4 * R.units);
  TCX_HIP(hipGetLastError());
  return TC_OK;
}

// Work lists over the rows R (cnt entries each), grouped by owner, and
// slices of equal work.
int work_lists(tc_ctx* c, tc_graph* g, const uint32_t* cnt, const uint16_t* id, bool tail,
               bool credit, Rows16& R) {
  const uint32_t n = g->n;
  const uint64_t m = g->m_or;
  DevBuf keys, tmp, wrp, cost, flags, work, prew;
  DevBuf& ids = R.who;
  TCX_TRY(keys.reserve(8 * m));
  TCX_TRY(tmp.reserve(8 * m));
  TCX_TRY(wrp.reserve(4 * ((size_t)n + 1)));
  TCX_TRY(flags.reserve(std::max<uint64_t>(n, tail ? m : 0) + 1));
  hipLaunchKernelGGL(k_keys16, dim3(grid_for(m)), dim3(TB), 0, c->stream, g->esrc.as<uint32_t>(),
                     g->col.as<uint32_t>(), m, n, cnt, id, tail, keys.as<uint64_t>(),
                     tail ? flags.as<uint8_t>() : nullptr);
  TCX_HIP(hipGetLastError());
  // few edges have tail entries at both ends: their keys alone are sorted (R-MAT-18:
  // 0.20 -> 0.06 ms)
  uint64_t nk = m;
  uint64_t *from = keys.as<uint64_t>(), *to = tmp.as<uint64_t>();
  if (tail) {
    TCX_TRY(compact_u64(c, from, flags.as<uint8_t>(), m, to, &nk));
    std::swap(from, to);
  }
  // only the owner's bits are sorted: the order within a list is free
  uint64_t* sorted;
  TCX_TRY(sort_u64(c, from, to, nk, 32 + bit_width_u32(n), &sorted, 32));
  hipLaunchKernelGGL(k_rowptr_search<uint64_t>, dim3(grid_for((uint64_t)n + 1)), dim3(TB), 0,
                     c->stream, sorted, nk, n, wrp.as<uint32_t>());
  TCX_HIP(hipGetLastError());
  uint32_t kept = (uint32_t)nk;
  if (!tail) TCX_TRY(read_back(c, wrp.as<uint32_t>() + n, &kept));
  R.entries = kept;
  R.tasks = 0;
  R.nslice = 0;
  if (!kept) return TC_OK;
  TCX_TRY(R.se.reserve(8ull * kept));
  if (credit) TCX_TRY(R.cred.reserve(4ull * kept));
  TCX_TRY(cost.reserve(8 * ((size_t)n + 1)));
  TCX_TRY(ids.reserve(4 * ((size_t)n + 1)));
  TCX_HIP(hipMemsetAsync(cost.p, 0, 8 * (size_t)n, c->stream));
  hipLaunchKernelGGL(k_entries16, dim3(grid_for(kept)), dim3(TB), 0, c->stream, sorted,
                     (uint64_t)kept, R.row.as<uint2>(), R.se.as<uint2>(),
                     credit ? R.cred.as<uint32_t>() : nullptr, cost.as<unsigned long long>());
  hipLaunchKernelGGL(k_nonempty, dim3(grid_for(n)), dim3(TB), 0, c->stream, wrp.as<uint32_t>(), n,
                     flags.as<uint8_t>());
  TCX_HIP(hipGetLastError());
  TCX_TRY(select_indices(c, flags.as<uint8_t>(), n, ids.as<uint32_t>(), &R.tasks));
  const uint64_t nt = R.tasks;
  TCX_TRY(R.act.reserve(16 * (nt + 1)));
  TCX_TRY(work.reserve(8 * (nt + 1)));
  TCX_TRY(prew.reserve(8 * (nt + 1)));
  hipLaunchKernelGGL(k_tasks16, dim3(grid_for(nt + 1)), dim3(TB), 0, c->stream, ids.as<uint32_t>(),
                     (uint32_t)nt, wrp.as<uint32_t>(), R.row.as<uint2>(),
                     cost.as<unsigned long long>(), R.act.as<uint4>(), work.as<uint64_t>());
  TCX_TRY(exclusive_scan_u64(c, work.as<uint64_t>(), prew.as<uint64_t>(), nt + 1));
  uint64_t total = 0;
  TCX_TRY(read_back(c, prew.as<uint64_t>() + nt, &total));
  // One slice per wave of the default grid, at least 256 group steps long; up
  // to 32 a wave where they still have 2,048.  A slice begins with a claim and
  // a chain of reads: with 1,024-step slices a batch of 128 small ER graphs
  // took 0.67 instead of 0.48 ms, and with eight slices a wave instead of 32
  // the last ones left R-MAT-23 waiting (10.15 instead of 9.85 ms).
  const uint64_t nw = (uint64_t)c->num_cus * 16u;
  uint64_t ns = std::min<uint64_t>(std::max<uint64_t>(total / 256, 1), nw);
  if (total / 2048 > 2 * nw) ns = std::min<uint64_t>(total / 2048, 32 * nw);
  R.nslice = (uint32_t)ns;
  TCX_TRY(R.slice.reserve(8 * (ns + 1)));
  hipLaunchKernelGGL(k_slices16, dim3(grid_for(ns + 1)), dim3(TB), 0, c->stream,
                     prew.as<uint64_t>(), R.act.as<uint4>(), (uint32_t)nt, R.entries, (uint32_t)ns,
                     R.slice.as<uint2>());
  TCX_HIP(hipGetLastError());
  return TC_OK;
}

// The hub's work lists of a layer built without them.
int hub_lists(tc_ctx* c, tc_graph* g, Lists16& L) {
  ++g->sc.builds;
  TCX_TRY(work_lists(c, g, L.cnt.as<uint32_t>(), L.id.as<uint16_t>(), false, L.credit, L.hub));
  L.id.release();
  L.cnt.release();
  L.listed = true;
  return TC_OK;
}

// Rows, work lists and slices for the ids `id` (null: every vertex id is its
// own 16-bit id; id_all: every vertex has one, and there is no tail).
// lists: with the hub's work lists; without them, id and the row lengths stay
// with L for hub_lists().  L.usable is left false when too few entries have an id.
int build(tc_ctx* c, tc_graph* g, DevBuf& idbuf, bool id_all, bool credit, bool lists, Lists16& L) {
  const uint16_t* id = idbuf.as<uint16_t>();
  const uint32_t n = g->n;
  const uint64_t m = g->m_or;
  const uint32_t* rp = g->rowptr.as<uint32_t>();
  const uint32_t* col = g->col.as<uint32_t>();
  const uint32_t* esrc = g->esrc.as<uint32_t>();
  DevBuf pre_b, cnt, tcnt;
  const uint32_t* pre = nullptr;
  uint32_t with_id = (uint32_t)m;
  if (!id_all) {
    DevBuf flag;
    TCX_TRY(flag.reserve(4 * (m + 1)));
    TCX_TRY(pre_b.reserve(4 * (m + 1)));
    hipLaunchKernelGGL(k_entry_flags, dim3(grid_for(m + 1)), dim3(TB), 0, c->stream, col, m, id,
                       flag.as<uint32_t>());
    TCX_TRY(exclusive_scan_u32(c, flag.as<uint32_t>(), pre_b.as<uint32_t>(), m + 1));
    pre = pre_b.as<uint32_t>();
    TCX_TRY(read_back(c, pre + m, &with_id));
    const double least = g->sum_in_out >= kLongList * m ? kMinEntries : kMinShare;
    if ((double)with_id < least * (double)m) return TC_OK;
  }
  const bool tail = with_id < m;
  TCX_TRY(cnt.reserve(4 * ((size_t)n + 1)));
  if (tail) TCX_TRY(tcnt.reserve(4 * ((size_t)n + 1)));
  hipLaunchKernelGGL(k_counts16, dim3(grid_for(n)), dim3(TB), 0, c->stream, rp, pre, n,
                     cnt.as<uint32_t>(), tail ? tcnt.as<uint32_t>() : nullptr);
  if ((double)with_id < kMinShare * (double)m) {
    TCX_TRY(c->accum.reserve(64));
    TCX_HIP(hipMemsetAsync(c->accum.p, 0, 8, c->stream));
    hipLaunchKernelGGL(k_streamed, dim3(std::min<unsigned>(grid_for(m), c->num_cus * 8u)), dim3(TB),
                       0, c->stream, col, m, cnt.as<uint32_t>(), c->accum.as<unsigned long long>());
    TCX_HIP(hipGetLastError());
    unsigned long long hub = 0;
    TCX_TRY(read_back(c, c->accum.p, &hub));
    if ((double)hub < kMinStream * (double)g->sum_in_out) return TC_OK;
  }
  TCX_TRY(place_rows(c, n, cnt.as<uint32_t>(), 8, L.hub));
  if (tail) TCX_TRY(place_rows(c, n, tcnt.as<uint32_t>(), 4, L.tail));
  hipLaunchKernelGGL(k_scatter16, dim3(grid_for(m)), dim3(TB), 0, c->stream, rp, col, esrc, m, id,
                     pre, L.hub.row.as<uint2>(), L.hub.col.as<uint16_t>(),
                     L.tail.row.as<uint2>(), L.tail.col.as<uint32_t>());
  TCX_HIP(hipGetLastError());
  L.credit = credit;
  L.listed = lists;
  if (lists) TCX_TRY(work_lists(c, g, cnt.as<uint32_t>(), id, false, credit, L.hub));
  L.tail.tasks = 0;
  if (tail) TCX_TRY(work_lists(c, g, tcnt.as<uint32_t>(), id, true, credit, L.tail));
  if (!lists) {
    swap(L.id, idbuf);
    swap(L.cnt, cnt);
  }
  L.usable = true;
  return TC_OK;
}

}  // namespace

// Bytes that one count over R streams: *sum += 16 per unit of every task's own row
// and of every list, 8 per work-list entry, 16 per task.
static __global__ __launch_bounds__(TB) void k_rows_bytes(const uint2* __restrict__ se,
                                                          uint64_t entries,
                                                          const uint4* __restrict__ act,
                                                          uint64_t tasks, unsigned long long* sum) {
  __shared__ unsigned long long red[TB / 64];
  unsigned long long s = 0;
  for (uint64_t i = gtid(); i < entries; i += gstride()) s += 8ull + 16ull * se[i].y;
  for (uint64_t i = gtid(); i < tasks; i += gstride()) s += 16ull + 16ull * act[i].w;
  flush_block(s, sum, red);
}

int rows_bytes(tc_ctx* c, const Lists16& L, double* bytes) {
  TCX_TRY(c->accum.reserve(64));
  TCX_HIP(hipMemsetAsync(c->accum.p, 0, 8, c->stream));
  for (const Rows16* R : {&L.hub, &L.tail})
    if (R->tasks)
      hipLaunchKernelGGL(k_rows_bytes, dim3(std::min<unsigned>(grid_for(R->entries), c->num_cus * 8u)),
                         dim3(TB), 0, c->stream, R->se.as<uint2>(), R->entries, R->act.as<uint4>(),
                         R->tasks, c->accum.as<unsigned long long>());
  TCX_HIP(hipGetLastError());
  unsigned long long h = 0;
  TCX_TRY(read_back(c, c->accum.p, &h));
  *bytes = (double)h;
  return TC_OK;
}

static bool no_room(int status) { return status == TC_ERR_NOMEM || status == TC_ERR_RANGE; }

// The rows, and (lists) the hub's work lists, which the push methods do without.
static int build_layer16(tc_ctx* c, tc_graph* g, bool credit, bool lists) {
  Lists16& L = g->sc.l16;
  if (L.version == g->sched_version && (!L.usable || L.credit || !credit)) {
    if (L.usable && lists && !L.listed) TCX_TRY(hub_lists(c, g, L));
    return TC_OK;
  }
  ++g->sc.builds;
  L.version = ~0ull;
  L.usable = false;
  if (g->n && g->m_or) {
    DevBuf id;
    bool some = true;
    if (g->n > kMax16) TCX_TRY(hub_ids(c, g, id, &some));
    if (some) TCX_TRY(build(c, g, id, g->n <= kMax16, credit, lists, L));
  }
  L.version = g->sched_version;
  return TC_OK;
}

// A layer that there is no room for does not suit the graph: every count has a
// kernel that needs less.
static int layer16(tc_ctx* c, tc_graph* g, bool credit, bool lists) {
  const int st = build_layer16(c, g, credit, lists);
  if (!no_room(st)) return st;
  g->sc.l16.release();
  g->sc.push16.release();  // (over its rows)
  g->sc.l16.version = g->sched_version;
  return TC_OK;
}

int lists16(tc_ctx* c, tc_graph* g, bool credit) { return layer16(c, g, credit, true); }

int without_rows(tc_graph* g, int status) {
  if (!no_room(status)) return status;
  g->sc.push16.release();
  g->sc.l32.release();
  g->sc.l32.version = ~0ull;
  g->sc.no_rows_version = g->sched_version;
  return TC_OK;
}

int lists16_batch(tc_ctx* c, tc_graph* g, const uint32_t* gid, const uint32_t* voff) {
  Lists16& L = g->sc.l16;
  if (L.version == g->sched_version) return TC_OK;
  L.usable = false;
  if (g->n && g->m_or) {
    DevBuf id;
    int st = id.reserve(2 * (size_t)g->n);
    if (st == TC_OK) {
      hipLaunchKernelGGL(k_local_ids, dim3(grid_for(g->n)), dim3(TB), 0, c->stream, gid, voff, g->n,
                         id.as<uint16_t>());
      TCX_HIP(hipGetLastError());
      st = build(c, g, id, true, false, true, L);
    }
    if (no_room(st)) L.release();
    else TCX_TRY(st);
    if (L.usable && L.hub.tasks)
      hipLaunchKernelGGL(k_graph_of, dim3(grid_for(L.hub.tasks)), dim3(TB), 0, c->stream,
                         L.hub.who.as<uint32_t>(), L.hub.tasks, gid);
    TCX_HIP(hipGetLastError());
  }
  L.version = g->sched_version;
  return TC_OK;
}

int count16_graphs(tc_ctx* c, tc_graph* g, uint32_t grid, uint32_t* cursor,
                   unsigned long long* counts) {
  const Rows16& R = g->sc.l16.hub;
  if (R.tasks)
    hipLaunchKernelGGL((k_count16<true, kOutGraph, 4>),
                       dim3(std::min<uint32_t>(grid, (uint32_t)c->num_cus * 4u)), dim3(TB), 0,
                       c->stream, R.col.as<uint4>(), R.se.as<uint2>(), R.act.as<uint4>(),
                       R.who.as<uint32_t>(), (const uint32_t*)nullptr, R.slice.as<uint2>(),
                       R.nslice, cursor, counts);
  TCX_HIP(hipGetLastError());
  return TC_OK;
}

int count16(tc_ctx* c, const Lists16& L, uint32_t grid, unsigned long long* acc,
            uint32_t* launches) {
  const uint32_t G = grid ? grid : (uint32_t)c->num_cus * 4u;
  const uint32_t G32 = grid ? grid : (uint32_t)c->num_cus * kWg32;
  // the cursors ride between the accumulators, one line each
  static_assert(kCurStride16 * 4 == kAccStride16 * 8, "one line per accumulator");
  auto launch = [&](auto kernel, uint32_t G, const Rows16& R, uint32_t* cur) {
    if (!R.tasks) return;
    hipLaunchKernelGGL(kernel, dim3(G), dim3(TB), 0, c->stream, R.col.as<uint4>(),
                       R.se.as<uint2>(), R.act.as<uint4>(), R.who.as<uint32_t>(),
                       R.cred.as<uint32_t>(), R.slice.as<uint2>(), R.nslice, cur, acc);
    ++*launches;
  };
  launch(k_count16<true, kOutTotal, 4>, G, L.hub, reinterpret_cast<uint32_t*>(acc + 8));
  launch(k_count16<false, kOutTotal, kU32>, G32, L.tail, reinterpret_cast<uint32_t*>(acc + 9));
  TCX_HIP(hipGetLastError());
  return TC_OK;
}

int count16_vertices(tc_ctx* c, tc_graph* g, uint32_t* cursor, unsigned long long* tri) {
  const Lists16& L = g->sc.l16;
  auto launch = [&](auto kernel, uint32_t per_cu, const Rows16& R, uint32_t* cur) {
    if (R.tasks)
      hipLaunchKernelGGL(kernel, dim3((uint32_t)c->num_cus * per_cu), dim3(TB), 0, c->stream,
                         R.col.as<uint4>(), R.se.as<uint2>(), R.act.as<uint4>(),
                         R.who.as<uint32_t>(), R.cred.as<uint32_t>(), R.slice.as<uint2>(),
                         R.nslice, cur, tri);
  };
  launch(k_count16<true, kOutVertex, 4>, 4u, L.hub, cursor);
  launch(k_count16<false, kOutVertex, kU32>, kWg32, L.tail, cursor + 1);
  TCX_HIP(hipGetLastError());
  return TC_OK;
}

// The rows of l32: every entry a 32-bit one (graphs that the 16-bit ids do not
// suit).  cnt: row lengths.
static int rows32(tc_ctx* c, tc_graph* g, DevBuf& cnt) {
  Lists16& L = g->sc.l32;
  const uint32_t n = g->n;
  const uint64_t m = g->m_or;
  const uint32_t* rp = g->rowptr.as<uint32_t>();
  TCX_TRY(cnt.reserve(4 * ((size_t)n + 1)));
  hipLaunchKernelGGL(k_counts16, dim3(grid_for(n)), dim3(TB), 0, c->stream, rp,
                     (const uint32_t*)nullptr, n, cnt.as<uint32_t>(), (uint32_t*)nullptr);
  if (L.version == g->sched_version) return TC_OK;
  L.version = ~0ull;
  L.usable = false;  // until the work lists are there
  TCX_TRY(place_rows(c, n, cnt.as<uint32_t>(), 4, L.tail));
  hipLaunchKernelGGL(k_scatter32, dim3(grid_for(m)), dim3(TB), 0, c->stream, rp,
                     g->col.as<uint32_t>(), g->esrc.as<uint32_t>(), m, L.tail.row.as<uint2>(),
                     L.tail.col.as<uint32_t>());
  TCX_HIP(hipGetLastError());
  L.version = g->sched_version;
  return TC_OK;
}

// TriCore's rule (tricore/src/tricount_gpu.cu:215-290), and Fox's
// (Fox/tc.cu:18-125): every edge's shorter list is looked up in its longer one.
// Grouped by the owner of the longer list, the edges share one bit map of it,
// where a wave spent six searches in sampled pivots and about three in the list
// (one line each) on every entry (TriCore), or log2 of the list's length of
// them (Fox); slices of equal work take the place of Fox's bins by work.
// TriCore: R-MAT-19 4.9 -> 0.32 ms, random geometric of 300,000 vertices 2.08 ->
// 0.67 ms; Fox: 7.6 -> 0.32 and 2.9 -> 0.66 ms, ER of 65,536 vertices and 2^20
// edges 0.18 -> 0.041 ms.
int lists16or32(tc_ctx* c, tc_graph* g, const Lists16** use) {
  TCX_TRY(lists16(c, g));
  *use = &g->sc.l16;
  if (g->sc.l16.usable) return TC_OK;
  Lists16& L = g->sc.l32;
  *use = &L;
  if (L.version == g->sched_version && L.usable) return TC_OK;
  ++g->sc.builds;
  DevBuf cnt;
  TCX_TRY(rows32(c, g, cnt));
  TCX_TRY(work_lists(c, g, cnt.as<uint32_t>(), nullptr, false, false, L.tail));
  L.usable = true;
  return TC_OK;
}

// Hu's method (Hu/tc.cu:69-201): the vertex blocks of its work model, N+(u)
// held in LDS, every wedge u -> v -> w looked up in it.  Here N+(u) is the bit
// map of k_count16 and a block's edges are the slices, so a block costs a wave
// 3.5 vector instructions an entry where a workgroup spent an owner search and
// a binary search on each wedge: R-MAT-19 11.8 -> 0.98 ms, ER of 10^6 vertices
// and 8 * 10^6 edges (32-bit rows) 0.40 -> 0.31 ms, random geometric of 300,000
// vertices and average degree 48 1.59 -> 0.53 ms.
int push16(tc_ctx* c, tc_graph* g) {
  Push16& H = g->sc.push16;
  TCX_TRY(layer16(c, g, false, false));
  if (H.version == g->sched_version) return TC_OK;
  ++g->sc.builds;
  const bool b16 = g->sc.l16.usable;
  const uint32_t n = g->n;
  const uint64_t m = g->m_or;
  const uint32_t* rp = g->rowptr.as<uint32_t>();
  DevBuf cnt, flags, ids;
  if (!b16) TCX_TRY(rows32(c, g, cnt));
  const uint2* row = (b16 ? g->sc.l16.hub : g->sc.l32.tail).row.as<uint2>();
  TCX_TRY(flags.reserve((size_t)n + 1));
  TCX_TRY(ids.reserve(4 * ((size_t)n + 1)));
  TCX_TRY(H.se.reserve(8 * m));
  hipLaunchKernelGGL(k_push16, dim3(grid_for(m)), dim3(TB), 0, c->stream, g->col.as<uint32_t>(),
                     m, row, H.se.as<uint2>());
  hipLaunchKernelGGL(k_push_flags, dim3(grid_for(n)), dim3(TB), 0, c->stream, rp, row, n,
                     flags.as<uint8_t>());
  TCX_TRY(select_indices(c, flags.as<uint8_t>(), n, ids.as<uint32_t>(), &H.tasks));
  TCX_TRY(H.act.reserve(16 * (H.tasks + 1)));
  hipLaunchKernelGGL(k_push_tasks, dim3(grid_for(H.tasks + 1)), dim3(TB), 0, c->stream,
                     ids.as<uint32_t>(), (uint32_t)H.tasks, rp, row, (uint32_t)m,
                     H.act.as<uint4>());
  TCX_HIP(hipGetLastError());
  H.version = g->sched_version;
  H.hu_blocks = 0;
  H.nslice = 0;
  return TC_OK;
}

static int edge_slices(tc_ctx* c, tc_graph* g, const int32_t* start, uint32_t nblocks,
                       uint32_t parts, DevBuf& slice, uint32_t* nslice) {
  ++g->sc.builds;
  const Push16& H = g->sc.push16;
  const uint32_t ns = nblocks * parts;
  *nslice = 0;
  TCX_TRY(slice.reserve(8 * ((size_t)ns + 1)));
  hipLaunchKernelGGL(k_edge_slices, dim3(grid_for((uint64_t)ns + 1)), dim3(TB), 0, c->stream, start,
                     nblocks, parts, g->n, g->rowptr.as<uint32_t>(), H.act.as<uint4>(),
                     (uint32_t)H.tasks, (uint32_t)g->m_or, slice.as<uint2>());
  TCX_HIP(hipGetLastError());
  *nslice = ns;
  return TC_OK;
}

int hu16(tc_ctx* c, tc_graph* g, const int32_t* start, uint32_t nblocks) {
  TCX_TRY(push16(c, g));
  Push16& H = g->sc.push16;
  if (H.hu_blocks == nblocks) return TC_OK;
  H.hu_blocks = 0;
  // few blocks: four waves each, as a workgroup would have; two where a block
  // has some 200 edges (R-MAT-19: 258 of them, 0.98 against 1.27 ms with one
  // and 0.86 with four, which costs ER, 65,536 vertices, 35 of them, 101
  // against 51 us)
  const uint32_t parts = nblocks < (uint32_t)c->num_cus * 32u ? 4u
                         : g->m_or >= 200ull * nblocks        ? 2u
                                                              : 1u;
  TCX_TRY(edge_slices(c, g, start, nblocks, parts, H.hu_slice, &H.hu_nslice));
  H.hu_blocks = nblocks;
  return TC_OK;
}

// Bisson's method (Bisson/tc.cu:18-104): a bit map of N+(u) in which the lists
// of u's out-neighbours are looked up.  The map is k_count16's, in LDS and
// exact, where a workgroup had n bits in memory behind a hashed filter; the
// slices have equally many edges, 16 a wave.  R-MAT-19 19.4 -> 0.75 ms, ER of
// 10^6 vertices 1.25 -> 0.30 ms (8 * 10^6 edges, 32-bit rows).
int bisson16(tc_ctx* c, tc_graph* g) {
  TCX_TRY(push16(c, g));
  Push16& H = g->sc.push16;
  if (H.nslice) return TC_OK;
  return edge_slices(c, g, nullptr, 1u, (uint32_t)c->num_cus * 256u, H.slice, &H.nslice);
}

int count_push16(tc_ctx* c, tc_graph* g, const DevBuf& slice, uint32_t nslice, uint32_t grid,
                 unsigned long long* acc, uint32_t* launches) {
  const Lists16& L = g->sc.l16;
  const Push16& H = g->sc.push16;
  auto launch = [&](auto kernel, uint32_t per_cu, const uint4* col, const uint2* se,
                    const uint4* act, uint64_t tasks, const DevBuf& slice, uint32_t nslice,
                    uint32_t* cur) {
    if (!tasks) return;
    hipLaunchKernelGGL(kernel, dim3(grid ? grid : (uint32_t)c->num_cus * per_cu), dim3(TB), 0,
                       c->stream, col, se, act, (const uint32_t*)nullptr, (const uint32_t*)nullptr,
                       slice.as<uint2>(), nslice, cur, acc);
    ++*launches;
  };
  uint32_t* cur = reinterpret_cast<uint32_t*>(acc + 8);
  const uint2* se = H.se.as<uint2>();
  const uint4* act = H.act.as<uint4>();
  if (L.usable) {
    launch(k_count16<true, kOutTotal, 4>, 4u, L.hub.col.as<uint4>(), se, act, H.tasks, slice,
           nslice, cur);
    const Rows16& T = L.tail;
    launch(k_count16<false, kOutTotal, kU32>, kWg32, T.col.as<uint4>(), T.se.as<uint2>(),
           T.act.as<uint4>(), T.tasks, T.slice, T.nslice, cur + 2);
  } else {
    launch(k_count16<false, kOutTotal, kU32>, kWg32, g->sc.l32.tail.col.as<uint4>(), se, act,
           H.tasks, slice, nslice, cur);
  }
  TCX_HIP(hipGetLastError());
  return TC_OK;
}

unsigned long long sum16(const unsigned long long* acc) {
  unsigned long long s = 0;
  for (uint32_t i = 0; i < kAcc16; ++i) s += acc[i * kAccStride16];
  return s;
}

}  // namespace tcx

// Device code of the 16-bit list layer.
//
// Most streamed entries of a skewed graph name one of few targets.  The
// layer gives the targets of largest in-degree (all of them when the graph,
// or each graph of a batch, has at most 65,535 vertices) 16-bit ids and keeps
// every out-list's entries among them as uint16 rows, padded with kPad16 to
// whole 16-byte units.  Task x sets the bits of its own row in an exact
// 65,536-bit map in LDS and streams the rows of its work list against it: an
// entry costs two bytes of memory, one LDS byte read and 3.5 vector
// instructions, against four bytes, 12 LDS bytes and 9 instructions in the
// rank-indexed table of engine.h, and no id pattern can make it collide.
// Out-list entries beyond the 16-bit ids (the tail) keep 32-bit rows in the
// same layout, with work lists and tasks of their own; their map is hashed,
// and an entry whose bit is set is queued and searched in the owner's row.
// A triangle's closing vertex is in one of the two parts, so the two counts
// add up to the whole.
#pragma once

#include "engine.h"

namespace tcx {
namespace dev {

constexpr uint32_t kPad16 = 0xFFFFu;    // padding entry: its bit is never set
constexpr uint32_t kMax16 = 65535u;     // 16-bit ids are below this
constexpr uint32_t kMap16Words = 2048;  // bit map: id c is bit c >> 13 of byte c & 8191
constexpr uint32_t kGroup16 = 4;        // lanes that read one list together (64 bytes a step)
constexpr uint32_t kRing16 = 128;       // list bounds held in LDS per wave

constexpr uint32_t kMap32Words = 512;   // hashed map of a 32-bit row

// LDS of one wave.  The hashed map takes a quarter of the exact one's: twice
// the waves fit, and its false hits (a row of 100 entries: 0.6 % of the
// streamed ones) only cost a search.
template <bool B16>
struct Wave16 {
  static constexpr uint32_t kWords = B16 ? kMap16Words : kMap32Words;
  uint32_t map[kWords];
  uint2 ring[kRing16];
};

// What a per-vertex count adds to the LDS of a wave: whom each list of the ring
// and each queued entry is credited to (kEmpty: the task's owner).
struct Credit16 {
  uint32_t ring[kRing16];
  uint32_t q[128];
};

// Sum over each group of four lanes (DPP quad permutations).
__device__ inline uint32_t group_sum(uint32_t x) {
  static_assert(kGroup16 == 4, "a group is a DPP quad");
  x += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, 0xB1, 0xf, 0xf, false);  // lanes 1 0 3 2
  x += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, 0x4E, 0xf, 0xf, false);  // lanes 2 3 0 1
  return x;
}

__device__ inline void map16_set(uint32_t* map, uint32_t c) {
  if (c != kPad16) atomicOr(map + ((c & 8191u) >> 2), 1u << ((c >> 13) + 8u * (c & 3u)));
}

__device__ inline void map16_set8(uint32_t* map, const uint4& q) {
  const uint32_t d[4] = {q.x, q.y, q.z, q.w};
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    map16_set(map, d[i] & 0xFFFFu);
    map16_set(map, d[i] >> 16);
  }
}

__device__ inline void map16_clear8(uint32_t* map, const uint4& q) {
  const uint32_t d[4] = {q.x, q.y, q.z, q.w};
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    map[(d[i] & 0x1FFCu) >> 2] = 0u;
    map[(d[i] >> 18) & 0x7FFu] = 0u;
  }
}

// Members among the eight entries of q.
__device__ inline uint32_t map16_count8(const uint8_t* map, const uint4& q) {
  const uint32_t d[4] = {q.x, q.y, q.z, q.w};
  uint32_t b0[4], b1[4], c = 0;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    b0[i] = map[d[i] & 8191u];
    b1[i] = map[__builtin_amdgcn_ubfe(d[i], 16u, 13u)];
  }
#pragma unroll
  for (int i = 0; i < 4; ++i)
    c += __builtin_amdgcn_ubfe(b0[i], __builtin_amdgcn_ubfe(d[i], 13u, 3u), 1u) +
         __builtin_amdgcn_ubfe(b1[i], d[i] >> 29, 1u);
  return c;
}

// The hashed map of a 32-bit row: id x sets bit (t >> 18) & 7 of byte t >> 21,
// t = x * K (24-bit factors, one full-rate multiply).
__device__ inline uint32_t hash24(uint32_t x) { return __umul24(x, 0x9E3779u); }

__device__ inline void map32_set4(uint32_t* map, const uint4& q) {
  const uint32_t d[4] = {q.x, q.y, q.z, q.w};
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const uint32_t t = hash24(d[i]);
    if (d[i] != kEmpty) atomicOr(map + (t >> 23), 1u << (((t >> 18) & 7u) + 8u * ((t >> 21) & 3u)));
  }
}

__device__ inline void map32_clear4(uint32_t* map, const uint4& q) {
  const uint32_t d[4] = {q.x, q.y, q.z, q.w};
#pragma unroll
  for (int i = 0; i < 4; ++i)
    if (d[i] != kEmpty) map[hash24(d[i]) >> 23] = 0u;
}

// Per-wave state of a 32-bit task: its row (entries of col seen as uint32)
// and the queued entries.
struct Probe32 {
  const uint32_t* a;
  uint32_t lo, hi, qn;
  uint32_t* Q;
};

// The n queued entries from position `from` on that are in the task's row
// (this lane's one, for the owner).  CRED: those of a list that is credited
// elsewhere are added there.
template <bool CRED>
__device__ inline uint32_t queue32(const Probe32& P, uint32_t from, uint32_t n, uint32_t lane,
                                   const Credit16* C, unsigned long long* out) {
  wave_sync();
  const uint32_t x = lane < n ? P.Q[from + lane] : kEmpty;
  const uint32_t to = CRED && lane < n ? C->q[from + lane] : kEmpty;
  wave_sync();
  if (x == kEmpty || !contains(P.a, P.lo, P.hi, x)) return 0u;
  if (to == kEmpty) return 1u;
  atomicAdd(out + to, 1ull);
  return 0u;
}

// The four entries of q: those whose bit is set are queued; 64 queued ones
// are searched at once.
template <bool CRED>
__device__ inline uint32_t map32_count4(const uint8_t* map, const uint4& q, Probe32& P,
                                        uint32_t lane, uint32_t to, Credit16* C,
                                        unsigned long long* out) {
  const uint32_t d[4] = {q.x, q.y, q.z, q.w};
  uint32_t b[4], t[4], c = 0;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    t[i] = hash24(d[i]);
    b[i] = map[t[i] >> 21];
  }
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const bool hit = __builtin_amdgcn_ubfe(b[i], __builtin_amdgcn_ubfe(t[i], 18u, 3u), 1u) != 0u &&
                     d[i] != kEmpty;
    const uint64_t m = lanes(hit);
    if (m) {
      if (hit) {
        const uint32_t k = lanes_below(m, P.qn);
        P.Q[k] = d[i];
        if (CRED) C->q[k] = to;
      }
      P.qn = uniform(P.qn + (uint32_t)__popcll(m));
      if (P.qn >= 64) {
        P.qn -= 64;
        c += queue32<CRED>(P, P.qn, 64, lane, C, out);
      }
    }
  }
  return c;
}

// Streams the lists (start, 16-byte units) se[0, total) against the wave's
// map; returns this lane's members.  Each group of four lanes reads one list,
// 64 bytes a step, and takes the next list not yet taken when its own
// is used up, so lists of unequal length keep all groups busy; U steps of
// every group are in flight together.  The bounds pass through a ring in
// LDS, 64 per refill, the next 64 already loaded (nb: this lane's of the
// first 64).  B16: 16-bit entries (else 32-bit ones, with P).
// CRED: the members of a list with cred[list] != kEmpty are added to
// out[cred[list]] instead of being returned, by its group when it goes on to
// another list.
template <bool B16, bool CRED, int U>
__device__ inline unsigned long long stream16(const uint4* __restrict__ col,
                                              const uint2* __restrict__ se, uint32_t total,
                                              uint2 nb, uint32_t lane, Wave16<B16>& W,
                                              Probe32& P,
                                              const uint32_t* __restrict__ cred, Credit16* C,
                                              unsigned long long* out) {
  const uint8_t* map = reinterpret_cast<const uint8_t*>(W.map);
  const uint32_t j = lane & (kGroup16 - 1);
  constexpr uint64_t kLastLanes = 0x8888888888888888ull;
  static_assert(kGroup16 == 4, "kLastLanes has the last lane of each group");
  unsigned long long sum = 0;
  uint32_t acc = 0;
  uint32_t cur = 0;            // next unit of this group's list
  int32_t rem = 0;             // its units left
  uint32_t cnt = 0, held = 0;  // wave-uniform: lists taken, list bounds in the ring so far
  uint32_t tag = kEmpty, ctag = kEmpty, cacc = 0;  // CRED: list being read / counted, its members
  uint32_t ncr = kEmpty;
  if (CRED && lane < total) ncr = cred[lane];
  for (;;) {
    uint4 w[U];
    uint64_t busy[U];
    uint32_t tg[U];
#pragma unroll
    for (int s = 0; s < U; ++s) {
      // one bit per group that needs a list, at its last lane, so that every
      // lane of a group has the same number of bits below it
      const uint64_t m = lanes(rem <= 0) & kLastLanes;
      if (m && cnt < total) {
        if (held - cnt < 64 / kGroup16 && held < total) {
          W.ring[(held + lane) & (kRing16 - 1)] = nb;
          if (CRED) C->ring[(held + lane) & (kRing16 - 1)] = ncr;
          held = uniform(total - held < 64 ? total : held + 64);
          nb = held + lane < total ? se[held + lane] : make_uint2(0u, 0u);
          if (CRED) ncr = held + lane < total ? cred[held + lane] : kEmpty;
          wave_sync();
          sum += acc;  // at most 64 lists since the last refill: no overflow
          acc = 0;
        }
        const uint32_t k = lanes_below(m, cnt);
        if (rem <= 0 && k < total) {
          const uint2 b = W.ring[k & (kRing16 - 1)];
          cur = b.x;
          rem = (int32_t)b.y;
          if (CRED) tag = C->ring[k & (kRing16 - 1)];
        }
        cnt = uniform(cnt + (uint32_t)__popcll(m));
      }
      busy[s] = lanes(rem > 0);
      tg[s] = tag;
      w[s] = (int32_t)j < rem ? col[(uint64_t)cur + j] : make_uint4(~0u, ~0u, ~0u, ~0u);
      cur += kGroup16;
      rem -= (int32_t)kGroup16;
    }
#pragma unroll
    for (int s = 0; s < U; ++s) {
      if (!busy[s]) continue;
      if (!B16) {
        acc += map32_count4<CRED>(map, w[s], P, lane, tg[s], C, out);
      } else if (!CRED) {
        acc += map16_count8(map, w[s]);
      } else {
        if (lanes(tg[s] != ctag)) {
          const uint32_t t = group_sum(cacc);
          if (tg[s] != ctag) {
            if (ctag == kEmpty) acc += cacc;
            else if (j == 0 && t) atomicAdd(out + ctag, (unsigned long long)t);
            cacc = 0;
            ctag = tg[s];
          }
        }
        cacc += map16_count8(map, w[s]);
      }
    }
    if (cnt >= total && lanes(rem > 0) == 0) break;
  }
  if (B16 && CRED) {
    const uint32_t t = group_sum(cacc);
    if (ctag == kEmpty) acc += cacc;
    else if (j == 0 && t) atomicAdd(out + ctag, (unsigned long long)t);
  }
  return sum + acc;
}

template <bool B16>
__device__ inline void map_set(uint32_t* map, const uint4& q) {
  if (B16) map16_set8(map, q);
  else map32_set4(map, q);
}

template <bool B16>
__device__ inline void map_clear(uint32_t* map, const uint4& q) {
  if (B16) map16_clear8(map, q);
  else map32_clear4(map, q);
}

// One task: the owner's row own (first unit, units; q0: its unit `lane`) and
// the lists se[0, total) (nb: list `lane`).
template <bool B16, bool CRED, int U>
__device__ inline unsigned long long task16(const uint4* __restrict__ col, uint2 own, uint4 q0,
                                            const uint2* __restrict__ se, uint32_t total, uint2 nb,
                                            uint32_t lane, Wave16<B16>& W, uint32_t* Q,
                                            const uint32_t* __restrict__ cred, Credit16* C,
                                            unsigned long long* out) {
  map_set<B16>(W.map, q0);
  for (uint32_t k = lane + 64; k < own.y; k += 64) map_set<B16>(W.map, col[(uint64_t)own.x + k]);
  wave_sync();
  Probe32 P{reinterpret_cast<const uint32_t*>(col + own.x), 0u, 4 * own.y, 0u, Q};
  unsigned long long c = stream16<B16, CRED, U>(col, se, total, nb, lane, W, P, cred, C, out);
  if (!B16 && P.qn) c += queue32<CRED>(P, 0, P.qn, lane, C, out);
  wave_sync();
  // (a 16-bit padding entry clears the last word, whose bits all go in this
  // pass)
  map_clear<B16>(W.map, q0);
  for (uint32_t k = lane + 64; k < own.y; k += 64) map_clear<B16>(W.map, col[(uint64_t)own.x + k]);
  wave_sync();
  return c;
}

// Where the counts of k_count16 go: one total; one per vertex (who[task], the
// owner, is the first vertex of the triangles on the lists of its out-edges;
// cred[entry] names it for the lists of its in-edges); or one per graph
// (who[task]).
enum Out16 { kOutTotal = 0, kOutVertex = 1, kOutGraph = 2 };

// Counts over the rows.  act[i] = (first and end entry of the task's work list
// in se, first unit and units of the owner's row); slice s runs from (task,
// entry) slice[s] to slice[s + 1], slices of equal work, a wave each.  The
// workgroups form up to kAcc16 groups, group q with every kAcc16-th slice from
// q on and a cursor of its own (kCurStride16 words apart): its waves take one
// slice each, then claim the rest.  (One cursor for all serialised the claims
// at about 14 ns: R-MAT-18 took 0.40 ms, and takes 0.145.)  A task cut by a slice
// border is counted in parts.  While a task is streamed, the next
// one's own row and first 64 list bounds and the description of the one after
// it are on their way: with a few lists per task (the tail, most of an R-MAT
// graph's owners) those three dependent reads took longer than the lists.
// `total` holds kAcc16 accumulators kAccStride16 words apart (kOutTotal), or
// one word per vertex or graph.
// Bound by the fabric between memory and L2 on large graphs: R-MAT-23 (A-order,
// A-direction) reads 61 GB in 8.57 ms, 7.2 TB/s, with vector-ALU issue near
// 0.68 and LDS near 0.65 of their rates; the whole count takes 9.8 ms where
// the 32-bit rank tables took 19.7, R-MAT-24 22.5 where they took 43.6.  36 KB
// of LDS a workgroup, four workgroups a CU.  Four lanes a list and U = 4 steps
// in flight: R-MAT-23 9.65 ms against 9.75 with 8 lanes and 10.37 with 2, a
// batch of 384 small graphs 1.67 against 1.90 ms with 8; R-MAT-22 with U = 2
// 4.91 against 4.75 ms.
constexpr uint32_t kAcc16 = 64, kAccStride16 = 16, kCurStride16 = 32;

template <bool B16, int OUT, int U>
__global__ __launch_bounds__(TB) void k_count16(const uint4* __restrict__ col,
                                                const uint2* __restrict__ se,
                                                const uint4* __restrict__ act,
                                                const uint32_t* __restrict__ who,
                                                const uint32_t* __restrict__ cred,
                                                const uint2* __restrict__ slice, uint32_t nslice,
                                                uint32_t* __restrict__ cursor,
                                                unsigned long long* __restrict__ total) {
  __shared__ Wave16<B16> S[TB / 64];
  __shared__ uint32_t Q[TB / 64][B16 ? 1 : 128];
  constexpr bool kCred = OUT == kOutVertex;
  __shared__ Credit16 C[kCred ? TB / 64 : 1];
  __shared__ unsigned long long red[TB / 64];
  const uint32_t lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  const uint4 pad = make_uint4(~0u, ~0u, ~0u, ~0u);
  Wave16<B16>& W = S[wv];
  for (uint32_t i = lane; i < W.kWords; i += 64) W.map[i] = 0;
  wave_sync();
  unsigned long long cnt = 0;
  uint32_t graph = 0xFFFFFFFFu;
  const uint32_t ng = min(kAcc16, gridDim.x), q = blockIdx.x % ng;
  const uint32_t nw = (gridDim.x - q + ng - 1) / ng * (TB / 64);  // the group's waves
  for (uint32_t s = uniform(q + ng * (blockIdx.x / ng * (TB / 64) + wv)); s < nslice;) {
    const uint2 b = slice[s], e = slice[s + 1];
    // tasks [i, last], entries [at, stop) of the work lists
    uint32_t i = b.x, at = b.y;
    const uint32_t stop = e.y, last = stop > at ? e.x - (e.y == act[e.x].x ? 1u : 0u) : 0u;
    if (stop > at) {
      uint4 a = act[i], an = act[min(i + 1, last)];
      uint32_t w = 0, wn = 0;
      if (OUT != kOutTotal) {
        w = who[i];
        wn = who[min(i + 1, last)];
      }
      uint4 own = lane < a.w ? col[(uint64_t)a.z + lane] : pad;
      uint32_t end = min(a.y, stop);
      uint2 nb = at + lane < end ? se[at + lane] : make_uint2(0u, 0u);
      for (;;) {
        const bool more = i < last;
        const uint32_t nend = min(an.y, stop);
        uint4 ownn = pad;
        uint2 nbn = make_uint2(0u, 0u);
        uint4 an2 = an;
        uint32_t wn2 = wn;
        if (more) {
          if (lane < an.w) ownn = col[(uint64_t)an.z + lane];
          if (an.x + lane < nend) nbn = se[an.x + lane];
          an2 = act[min(i + 2, last)];
          if (OUT != kOutTotal) wn2 = who[min(i + 2, last)];
        }
        if (OUT == kOutGraph && w != graph) {
          if (graph != 0xFFFFFFFFu) {
            const unsigned long long t = wave_sum(cnt);
            if (lane == 0 && t) atomicAdd(total + graph, t);
            cnt = 0;
          }
          graph = w;
        }
        const unsigned long long c =
            task16<B16, kCred, U>(col, make_uint2(a.z, a.w), own, se + at, end - at, nb, lane, W,
                                  Q[wv], kCred ? cred + at : nullptr, C + (kCred ? wv : 0), total);
        if (OUT == kOutVertex) {
          const unsigned long long t = wave_sum(c);
          if (lane == 0 && t) atomicAdd(total + w, t);
        } else {
          cnt += c;
        }
        if (!more) break;
        ++i;
        a = an;
        w = wn;
        wn = wn2;
        at = an.x;
        end = nend;
        own = ownn;
        nb = nbn;
        an = an2;
      }
    }
    if ((uint64_t)nw * ng + q >= nslice) break;  // one slice a wave at most
    uint32_t nx = 0;
    if (lane == 0) nx = atomicAdd(cursor + q * kCurStride16, 1u);
    s = q + ng * (nw + uniform((uint32_t)__shfl((int)nx, 0, 64)));
  }
  if (OUT == kOutTotal) flush_block(cnt, total + (blockIdx.x % kAcc16) * kAccStride16, red);
  if (OUT == kOutGraph && graph != 0xFFFFFFFFu) {
    const unsigned long long t = wave_sum(cnt);
    if (lane == 0 && t) atomicAdd(total + graph, t);
  }
}

}  // namespace dev
}  // namespace tcx

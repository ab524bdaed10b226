// Direct path of the k-clique counter, k = 3, 4, 5, roots with d+ <= 512.
//
// Pivoting pays where branches are many levels deep.  With k <= 5 at most two
// levels are left above the closed forms, and nearly every candidate is a
// branch, so the pivot search and the walk's stack were overhead, and the
// closed form's lanes ran over neighbour sets of unequal size, one scattered
// LDS row at a time.  Here every wave of a root holds the root's whole strictly
// upper bit matrix in registers: lane z has rows z, z + 64, ...  A candidate
// pair's common neighbours A = N+(x) & N+(y) are wave-uniform and live in
// scalar registers (v_readlane, s_and); one v_and and one v_bcnt per 32 bits add
// up the edges inside A, with A itself as the execution mask.  No LDS and no
// divergence in the inner loop; words below y are left out at compile time.
// For k = 5 the out-neighbours are numbered by ascending degree: most pairs then
// have their y, and their few words, at the end (4-word rows: 2.7 words a pair
// against 4.0 in the order of ids; R-MAT-16 3.9 -> 3.2 ms in all).
// One-word rows (d+ <= 64) would leave most lanes idle and run at the scalar
// unit's rate; there a lane takes an edge of the sub-graph, from a list
// written while the matrix is built (k = 5, random geometric, 250,000 vertices,
// degree 48: 0.52 against 1.23 ms; k = 4: 0.39 against 0.47).
//
// Measured with the pivot kernels before, R-MAT-16 of 1.7 * 10^6 edges, k = 5:
// 8 words 4.4 -> 1.07 ms, 4 words 12.2 -> 1.30, 2 words 5.5 -> 0.53, 1 word 3.5 ->
// 0.26; k = 4: 7.3 -> 0.85 ms in all.  Vector-ALU issue was 80 % busy in the 4-word
// kernel with the order of ids (26 * 10^6 pairs, 10^9 instructions, a third of
// them building the matrix).
#pragma once

#include "internal.h"

namespace tcx {
namespace {

__device__ inline uint32_t uniform32(uint32_t v) { return __builtin_amdgcn_readfirstlane(v); }

__device__ inline uint64_t uniform64(uint64_t v) {
  return (uint64_t)uniform32((uint32_t)v) | ((uint64_t)uniform32((uint32_t)(v >> 32)) << 32);
}

// v of lane `from` (wave-uniform), in scalar registers
__device__ inline uint64_t lane64(uint64_t v, uint32_t from) {
  return (uint64_t)(uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)v, (int)from) |
         ((uint64_t)(uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)(v >> 32), (int)from) << 32);
}

// binom(p, r), p <= 512, r <= 4
__device__ inline unsigned long long binom4(unsigned long long p, uint32_t r) {
  unsigned long long c = p;
  if (r > 1) c = c * (p - 1) / 2;
  if (r > 2) c = p < 2 ? 0 : c * (p - 2) / 3;
  if (r > 3) c = p < 3 ? 0 : c * (p - 3) / 4;
  return c;
}

// Triangles of the upper bit matrix R inside the vertex set C (wave-uniform)
// whose smallest vertex is in C and in sel (repeated in every word): this
// lane's share.  R[t][w], w >= t: word w of row 64 t + lane; N words are in use.
template <int N, int W>
__device__ inline uint32_t upper_triangles(const uint64_t (&R)[W][W], const uint64_t (&C)[W],
                                           uint64_t sel) {
  uint32_t c = 0;
#pragma unroll
  for (int ty = 0; ty < N; ++ty) {
    for (uint64_t ys = C[ty] & sel; ys; ys &= ys - 1) {
      const uint32_t y = (uint32_t)__builtin_ctzll(ys);
      uint64_t A[W];
#pragma unroll
      for (int w = ty; w < N; ++w) A[w] = lane64(R[ty][w], y) & C[w];
#pragma unroll
      for (int t = ty; t < N; ++t) {
        if (__builtin_amdgcn_inverse_ballot_w64(A[t])) {
#pragma unroll
          for (int w = t; w < N; ++w) c += (uint32_t)__popcll(R[t][w] & A[w]);
        }
      }
    }
  }
  return c;
}

// Edges of R inside C: this lane's share.
template <int W>
__device__ inline uint32_t upper_edges(const uint64_t (&R)[W][W], const uint64_t (&C)[W]) {
  uint32_t c = 0;
#pragma unroll
  for (int t = 0; t < W; ++t) {
    if (__builtin_amdgcn_inverse_ballot_w64(C[t])) {
#pragma unroll
      for (int w = t; w < W; ++w) c += (uint32_t)__popcll(R[t][w] & C[w]);
    }
  }
  return c;
}

// k = 4: the triangles inside C0 whose smallest vertex is in sel.  k = 5: those
// inside C0 & N+(x), over all x of C0 in sel; and, p > 0, p times the former.
// M: the matrix in LDS, c0: C0 in LDS.
template <int N, int W>
__device__ inline unsigned long long direct_count(const uint64_t (&R)[W][W],
                                                  const uint64_t (&C0)[W], const uint64_t* M,
                                                  const uint64_t* c0, uint64_t sel, uint32_t k,
                                                  uint32_t p) {
  unsigned long long cnt = 0;
  bool first = k == 4 || p;
  uint32_t tx = 0;
  uint64_t xs = k == 5 ? uniform64(c0[0]) & sel : 0ull;
  for (;;) {
    uint64_t C[W], ys = ~0ull;
    uint32_t times = 1;
    if (first) {
#pragma unroll
      for (int w = 0; w < N; ++w) C[w] = C0[w];
      ys = sel;
      if (k == 5) times = p;
    } else {
      while (!xs && ++tx < (uint32_t)N) xs = uniform64(c0[tx]) & sel;
      if (!xs) break;
      const uint32_t x = 64 * tx + (uint32_t)__builtin_ctzll(xs);
      xs &= xs - 1;
#pragma unroll
      for (int w = 0; w < N; ++w) C[w] = uniform64(M[x * W + w]) & C0[w];
    }
    cnt += (unsigned long long)times * upper_triangles<N, W>(R, C, ys);
    if (first && k == 4) break;
    first = false;
  }
  return cnt;
}

constexpr uint32_t kClaimGroups = 64, kClaimStride = 32;  // claim counters, a line each

// (root, copy) tasks go in chunks, heaviest first: one a workgroup, then the
// workgroups of each of kClaimGroups groups claim the rest of its share (one
// counter for all serialises claims at about 14 ns: 60,000 narrow roots 0.92
// ms).  NW waves share a root: they build its matrix together (each takes every
// NW-th out-list of the root's out-neighbours), then walker q of the root's
// Q = copies * NW (a power of two <= 64) takes the first vertices q, q + Q, ...
// BOTH, for a CSR that the engine did not orient itself: it may hold both arcs of an
// edge, and the edge list of one-word rows takes an edge once, where its bit was
// clear, as the wider rows' bits do; the list has room for all 64 * 63 / 2.  (Waiting
// for the old word costs 5 %: random geometric, 250,000 vertices, k = 4, 391 -> 412 us.)
// Vertices adjacent to all others of N+(u) are taken out first when few pairs
// are missing: p of them add binom(p, j) times the smaller cliques of the rest,
// so near-complete roots cost little, as they did with pivots.
template <int W, int NW, bool BOTH = false>
__global__ __launch_bounds__(64 * NW)
__attribute__((amdgpu_waves_per_eu(W == 8 ? 4 : W == 4 ? 6 : 8))) void k_kcl_direct(
    const uint32_t* __restrict__ rp, const uint32_t* __restrict__ col,
    const uint32_t* __restrict__ deg, const uint32_t* __restrict__ roots, uint64_t nroots,
    uint32_t copies, uint32_t chunk, uint32_t k, unsigned long long* total,
    uint32_t* claim, float* __restrict__ cost, float cost_scale) {
  constexpr uint32_t D = 64 * W, T = 64 * NW;
  constexpr bool kPairs = W == 1;
  constexpr uint32_t kG = 8;  // lanes that read one out-list together
  constexpr uint32_t kU = 4;  // entries a lane takes of it at once
  constexpr uint64_t kLast = 0x8080808080808080ull;  // the groups' last lanes
  static_assert(kG == 8, "kLast has the last lane of each group");
  __shared__ uint32_t s_list[D];
  __shared__ uint2 s_be[D];
  __shared__ __align__(16) uint64_t s_M[D * W];  // bit (a, b), a < b
  __shared__ uint64_t s_C0[NW][W];
  // wider rows: the place of each out-neighbour in ascending order of degree
  __shared__ __align__(16) uint32_t s_key[kPairs ? 4 : D];
  __shared__ uint16_t s_pos[kPairs ? 1 : D];
  __shared__ uint32_t s_ti;
  // one-word rows: the edges a | b << 8 of the sub-graph, each the work of a lane
  __shared__ uint16_t s_pair[kPairs ? 64 * 63 / 2 : 1];
  const uint32_t tid = threadIdx.x, lane = tid & 63, wv = uniform32(tid >> 6);
  const uint32_t Q = copies * NW;
  const bool by_degree = !kPairs && k == 5;
  const uint64_t ntask = nroots * copies;
  unsigned long long cnt = 0;
  const uint32_t ng = min(kClaimGroups, gridDim.x), cq = blockIdx.x % ng;
  const uint32_t in_group = (gridDim.x - cq + ng - 1) / ng;
  // chunk ci has tasks ci, ci + nchunk, ...: all chunks some heavy and some light
  const uint64_t nchunk = (ntask + chunk - 1) / chunk;
  for (uint64_t ci = blockIdx.x; ci < nchunk;) {
    const uint32_t nt = (uint32_t)((ntask - ci + nchunk - 1) / nchunk);  // <= chunk <= 64
    // the chunk's roots and row bounds, one per lane
    uint32_t cu = 0, cb = 0, ce = 0;
    if (lane < nt) {
      cu = roots[(ci + lane * nchunk) / copies];
      cb = rp[cu];
      ce = rp[cu + 1];
    }
    // NW = 1: the next root's list, loaded behind this one's work
    uint32_t px = 0xFFFFFFFFu;
    uint2 pbe = make_uint2(0u, 0u);
    for (uint32_t ti = 0; ti < nt; ++ti) {
      const uint64_t t_task = (cost && tid == 0) ? wall_clock64() : 0;
      const uint32_t base = (uint32_t)__builtin_amdgcn_readlane((int)cb, (int)ti);
      const uint32_t d = (uint32_t)__builtin_amdgcn_readlane((int)ce, (int)ti) - base;  // <= D
      const uint32_t q = (uint32_t)((ci + ti * nchunk) % copies) * NW + wv;
      for (uint32_t i = tid; i < D; i += T) {
        uint32_t x = 0xFFFFFFFFu;
        uint2 be = make_uint2(0u, 0u);
        if (kPairs && ti) {
          x = px;
          be = pbe;
        } else if (i < d) {
          x = col[base + i];
          be = make_uint2(rp[x], rp[x + 1]);
        }
        s_list[i] = x;
        s_be[i] = be;
        if (by_degree) s_key[i] = i < d ? min(deg[x], (1u << 22) - 1) << 10 | i : 0xFFFFFFFFu;
      }
      for (uint32_t i = tid; i < D * W / 2; i += T)
        reinterpret_cast<uint4*>(s_M)[i] = make_uint4(0u, 0u, 0u, 0u);
      __syncthreads();
      if (by_degree) {
        for (uint32_t i = tid; i < d; i += T) {
          const uint32_t key = s_key[i];
          uint32_t r = 0;
          for (uint32_t j = 0; j < d; j += 4) {
            const uint4 o = *reinterpret_cast<const uint4*>(s_key + j);
            r += (o.x < key) + (o.y < key) + (o.z < key) + (o.w < key);
          }
          s_pos[i] = (uint16_t)r;
        }
        __syncthreads();
      }
      if (kPairs) {
        px = 0xFFFFFFFFu;
        pbe = make_uint2(0u, 0u);
        if (ti + 1 < nt) {
          const uint32_t b = (uint32_t)__builtin_amdgcn_readlane((int)cb, (int)(ti + 1));
          const uint32_t e = (uint32_t)__builtin_amdgcn_readlane((int)ce, (int)(ti + 1));
          if (b + lane < e) px = col[b + lane];
        }
      }
      uint32_t np = 0;  // (wave-uniform)
      // Every entry of the out-lists is searched in N+(u).  Each group of kG
      // lanes takes kU * kG entries a step, and the wave's next list when its own
      // is used up; the next step's entries are loaded before this one's are
      // searched.  8 lanes and 4 entries each: R-MAT-16, k = 4, 886 us against 954
      // with 4 lanes (one-word rows) and 992 with 4 lanes and 8 entries.
      {
        const uint32_t j = lane & (kG - 1);
        const uint32_t nl = d > wv ? (d - wv + NW - 1) / NW : 0;  // this wave's lists
        uint32_t top = D / 2;  // (only one-word rows may have fewer than D / 2 entries)
        while (W == 1 && top > 1 && top >= d) top >>= 1;
        uint32_t cur = 0, end = 0, li = 0, taken = 0;
        auto next = [&](uint32_t (&x)[kU]) -> bool {
          uint64_t m = __ballot(cur >= end) & kLast;
          while (m && taken < nl) {
            const uint32_t i = taken + __builtin_amdgcn_mbcnt_hi(
                                           (uint32_t)(m >> 32),
                                           __builtin_amdgcn_mbcnt_lo((uint32_t)m, 0u));
            if (cur >= end && i < nl) {
              li = wv + NW * i;
              const uint2 be = s_be[li];
              cur = be.x + j;
              end = be.y + j;
            }
            taken = uniform32(taken + (uint32_t)__popcll(m));
            if (__ballot(cur < end)) break;  // (else only empty lists)
            m = kLast;
          }
          const uint32_t left = end > cur ? end - cur : 0;  // of the group
#pragma unroll
          for (uint32_t s = 0; s < kU; ++s) x[s] = j + s * kG < left ? col[cur + s * kG] : 0xFFFFFFFFu;
          if (left) cur += min(left, kU * kG);
          return __ballot(left != 0) != 0;
        };
        auto step = [&](uint32_t (&lo)[kU], const uint32_t (&x)[kU], uint32_t half) {
#pragma unroll
          for (uint32_t s = 0; s < kU; ++s) lo[s] += s_list[lo[s] + half] <= x[s] ? half : 0u;
        };
        uint32_t x[kU];
        bool more = next(x);
        while (more) {
          const uint32_t xi = li;
          uint32_t y[kU], lo[kU];
          more = next(y);
#pragma unroll
          for (uint32_t s = 0; s < kU; ++s) lo[s] = 0;
          if (W == 1) {
            for (uint32_t half = top; half; half >>= 1) step(lo, x, half);
          } else {
#pragma unroll
            for (uint32_t half = D / 2; half; half >>= 1) step(lo, x, half);
          }
#pragma unroll
          for (uint32_t s = 0; s < kU; ++s) {
            const bool hit = x[s] != 0xFFFFFFFFu && s_list[lo[s]] == x[s];
            uint32_t pa = xi, pb = lo[s];
            if (by_degree && hit) {
              pa = s_pos[pa];
              pb = s_pos[pb];
            }
            const uint32_t a = min(pa, pb), b = max(pa, pb), bit = 1u << (b & 31);
            bool enter = hit;
            if (hit) {
              uint32_t* word = reinterpret_cast<uint32_t*>(s_M) + 2 * W * a + (b >> 5);
              if (BOTH) enter = !(atomicOr(word, bit) & bit);
              else atomicOr(word, bit);
            }
            if (kPairs) {
              const uint64_t m = __ballot(enter);
              if (enter)
                s_pair[np + __builtin_amdgcn_mbcnt_hi(
                                (uint32_t)(m >> 32),
                                __builtin_amdgcn_mbcnt_lo((uint32_t)m, 0u))] = (uint16_t)(a | b << 8);
              np = uniform32(np + (uint32_t)__popcll(m));
            }
            x[s] = y[s];
          }
        }
      }
      __syncthreads();

      if constexpr (kPairs) {
        if (px != 0xFFFFFFFFu) pbe = make_uint2(rp[px], rp[px + 1]);
        // lane i: the common neighbours A of an edge's ends above both (k = 4), or
        // the edges inside A
        const uint2* M2 = reinterpret_cast<const uint2*>(s_M);
        uint32_t c = 0;
        if (k == 3) c = lane == 0 ? np : 0u;
        else
          for (uint32_t i = lane; i < np; i += 64) {
            const uint32_t pr = s_pair[i];
            const uint2 ra = M2[pr & 255u], rb = M2[pr >> 8];
            const uint32_t lo = ra.x & rb.x, hi = ra.y & rb.y;
            if (k == 4) {
              c += __popc(lo) + __popc(hi);
              continue;
            }
            for (uint32_t zs = lo; zs; zs &= zs - 1) {
              const uint2 r = M2[__builtin_ctz(zs)];
              c += __popc(lo & r.x) + __popc(hi & r.y);
            }
            for (uint32_t zs = hi; zs; zs &= zs - 1) c += __popc(hi & M2[32 + __builtin_ctz(zs)].y);
          }
        cnt += c;
      } else {
        uint64_t R[W][W], C0[W];
        uint32_t e = 0, p = 0, size = 0;
  #pragma unroll
        for (int t = 0; t < W; ++t) {
  #pragma unroll
          for (int w = t; w < W; ++w) {
            R[t][w] = s_M[(64 * t + lane) * W + w];
            e += (uint32_t)__popcll(R[t][w]);
          }
          C0[t] = d >= 64u * t + 64 ? ~0ull : (d > 64u * t ? (1ull << (d - 64u * t)) - 1 : 0ull);
        }
        e = uniform32(wave_sum_u32(e));
        if (d * (d - 1) / 2 - e <= d) {
          // vertices adjacent to all above them (F) and to all below (not in low)
          uint64_t F[W], low[W];
  #pragma unroll
          for (int w = 0; w < W; ++w) low[w] = 0;
  #pragma unroll
          for (int t = 0; t < W; ++t) {
            uint64_t miss = 0;
            const bool in = 64u * t + lane < d;
  #pragma unroll
            for (int w = t; w < W; ++w) {
              uint64_t v = C0[w] & ~R[t][w];
              if (w == t) v &= ~((2ull << lane) - 1);
              if (!in) v = 0;
              miss |= v;
              low[w] |= v;
            }
            F[t] = __ballot(miss == 0);
          }
  #pragma unroll
          for (int w = 0; w < W; ++w) {
            const uint64_t all = C0[w] & F[w] & ~uniform64(wave_or_u64(low[w]));
            p += (uint32_t)__popcll(all);
            C0[w] &= ~all;
          }
        }
  #pragma unroll
        for (int w = 0; w < W; ++w) size += (uint32_t)__popcll(C0[w]);
        const bool lead = q == 0 && lane == 0;
        if (k == 3) {
          if (lead) cnt += e;
        } else {
          uint64_t sel = 0;
          for (uint32_t b = q; b < 64; b += Q) sel |= 1ull << b;
          if (p) {  // k - 1 of C0 and the p others, fewer than k - 2 of them from C0
            const uint32_t r = k - 1;
            if (q == 0) cnt += binom4(p, r - 2) * upper_edges<W>(R, C0);
            if (lead) cnt += binom4(p, r - 1) * size + binom4(p, r);
          }
          if (lane == 0) {
  #pragma unroll
            for (int w = 0; w < W; ++w) s_C0[wv][w] = C0[w];
          }
          wave_sync_kcl();
          const uint64_t* c0 = s_C0[wv];
          // the words in use, past half of W (a shorter row takes a narrower kernel)
          if (W == 8 && d <= 320) cnt += direct_count<W == 8 ? 5 : W, W>(R, C0, s_M, c0, sel, k, p);
          else if (W == 8 && d <= 384) cnt += direct_count<W == 8 ? 6 : W, W>(R, C0, s_M, c0, sel, k, p);
          else if (W == 8 && d <= 448) cnt += direct_count<W == 8 ? 7 : W, W>(R, C0, s_M, c0, sel, k, p);
          else if (W == 4 && d <= 192) cnt += direct_count<W == 4 ? 3 : W, W>(R, C0, s_M, c0, sel, k, p);
          else cnt += direct_count<W, W>(R, C0, s_M, c0, sel, k, p);
        }
      }
      __syncthreads();
      if (cost && tid == 0)
        atomicAdd(cost + (uint32_t)__builtin_amdgcn_readlane((int)cu, (int)ti),
                  (float)(wall_clock64() - t_task) * cost_scale);
    }
    if ((uint64_t)in_group * ng + cq >= nchunk) break;  // one chunk each at most
    if (tid == 0) s_ti = atomicAdd(claim + cq * kClaimStride, 1u);
    __syncthreads();
    ci = cq + ng * (in_group + (uint64_t)uniform32(s_ti));
  }
  cnt = wave_sum(cnt);
  if (lane == 0 && cnt) atomicAdd(total, cnt);
}

}  // namespace
}  // namespace tcx

// Passes over long arrays that build graphs: the histogram of vertex ids and
// the compaction of sorted keys.
#include <algorithm>

#include "engine.h"
#include "internal.h"

namespace tcx {
namespace {

constexpr uint32_t TB = 256;

__device__ inline uint64_t gtid() { return (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; }
__device__ inline uint64_t gstride() { return (uint64_t)gridDim.x * blockDim.x; }

unsigned grid_for(uint64_t n, unsigned tb = TB) {
  const uint64_t b = (n + tb - 1) / tb;
  return (unsigned)(b < 1 ? 1 : b > (1u << 20) ? 1u << 20 : b);
}

// ---- histogram of ids --------------------------------------------------------
// One atomic in memory per id ran at about 9 * 10^9 ids a second where the ids
// are skewed (their words share few lines).  Instead the ids are split into bins of
// kBinIds consecutive hashed ids, each counted in LDS:
//   k_bin_ids   sorts tiles of kTileIds ids by bin and writes them as 16-bit
//               numbers within the bin, with each tile's bin borders;
//   k_bin_hist  S workgroups a bin count every S-th tile's part of it in LDS;
//   k_bin_sum   adds the S counts of every id.
// The hash, a multiplication by an odd number modulo a power of two, permutes the
// ids, so that bins of skewed ids fill evenly.  Bound by the LDS atomics of the
// first two.  R-MAT-21, 6.7 * 10^7 ids: 6.6 -> 0.27 ms; with the compaction
// below, degree orientation of R-MAT-21 9.9 -> 2.7 ms, of R-MAT-18 1.53 -> 0.65.
// Fewer than kMinBinned ids gain nothing (ER of 65,536 vertices, 2^20 ids: 0.35
// against 0.37 ms for the orientation, R-MAT-16 0.43 against 0.36).
constexpr uint32_t kTileIds = 8192, kTileThreads = 512, kTilePer = kTileIds / kTileThreads;
constexpr uint32_t kBinBits = 14, kBinIds = 1u << kBinBits, kMaxBins = 256;
constexpr uint32_t kHash = 0x9E3779B1u, kHashInv = 0x0E8B2F51u;
static_assert((uint32_t)(kHash * kHashInv) == 1u, "inverse modulo 2^32");

__global__ __launch_bounds__(kTileThreads) void k_bin_ids(const uint32_t* __restrict__ a,
                                                          uint64_t m, uint32_t n, uint32_t bits,
                                                          uint32_t nb, uint16_t* __restrict__ out,
                                                          uint16_t* __restrict__ border) {
  __shared__ uint32_t cnt[kMaxBins], off[kMaxBins + 1];
  __shared__ __align__(16) uint16_t stage[kTileIds];
  const uint32_t tid = threadIdx.x, lane = tid & 63;
  const uint32_t mask = bits == 32 ? ~0u : (1u << bits) - 1;
  for (uint32_t i = tid; i < kMaxBins; i += kTileThreads) cnt[i] = 0;
  __syncthreads();
  const uint64_t base = (uint64_t)blockIdx.x * kTileIds;
  uint32_t x[kTilePer], rank[kTilePer];
#pragma unroll
  for (uint32_t i = 0; i < kTilePer; ++i) {
    const uint64_t at = base + (uint64_t)i * kTileThreads + tid;
    const uint32_t id = at < m ? a[at] : 0xFFFFFFFFu;
    x[i] = id < n ? (id * kHash) & mask : 0xFFFFFFFFu;
  }
#pragma unroll
  for (uint32_t i = 0; i < kTilePer; ++i)
    rank[i] = x[i] != 0xFFFFFFFFu ? atomicAdd(cnt + (x[i] >> kBinBits), 1u) : 0u;
  __syncthreads();
  if (tid < 64) {  // four bins a lane
    uint32_t c[kMaxBins / 64], sum = 0;
#pragma unroll
    for (uint32_t i = 0; i < kMaxBins / 64; ++i) sum += c[i] = cnt[lane * (kMaxBins / 64) + i];
    uint32_t run = dev::wave_incl_scan_dpp(sum) - sum;
#pragma unroll
    for (uint32_t i = 0; i < kMaxBins / 64; ++i) {
      off[lane * (kMaxBins / 64) + i] = run;
      run += c[i];
    }
    if (lane == 63) off[kMaxBins] = run;
  }
  __syncthreads();
#pragma unroll
  for (uint32_t i = 0; i < kTilePer; ++i)
    if (x[i] != 0xFFFFFFFFu)
      stage[off[x[i] >> kBinBits] + rank[i]] = (uint16_t)(x[i] & (kBinIds - 1));
  __syncthreads();
  uint4* dst = reinterpret_cast<uint4*>(out + (uint64_t)blockIdx.x * kTileIds);
  for (uint32_t i = tid; i < kTileIds / 8; i += kTileThreads)
    dst[i] = reinterpret_cast<const uint4*>(stage)[i];
  uint16_t* b = border + (uint64_t)blockIdx.x * (nb + 1);
  for (uint32_t i = tid; i <= nb; i += kTileThreads) b[i] = (uint16_t)off[i];  // <= 8192
}

// Workgroup (bin, s): part[s][ids of the bin].  A wave takes the borders of
// `per` (a multiple of 4, at most 64) tiles at a time and keeps four tiles' ids
// in flight.
__global__ __launch_bounds__(1024) void k_bin_hist(const uint16_t* __restrict__ ids,
                                                   const uint16_t* __restrict__ border,
                                                   uint32_t ntile, uint32_t nb, uint32_t S,
                                                   uint32_t per, uint32_t* __restrict__ part) {
  __shared__ uint32_t hist[kBinIds];
  const uint32_t tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
  const uint32_t bin = blockIdx.x % nb, s = blockIdx.x / nb;
  for (uint32_t i = tid; i < kBinIds; i += 1024) hist[i] = 0;
  __syncthreads();
  // tiles s + S * j, j = wv * per + lane, and on by 16 waves
  for (uint64_t j0 = (uint64_t)wv * per; s + S * j0 < ntile; j0 += 16 * per) {
    const uint64_t t = s + S * (j0 + lane);
    uint32_t lo = 0, hi = 0;
    if (lane < per && t < ntile) {
      lo = border[t * (nb + 1) + bin];
      hi = border[t * (nb + 1) + bin + 1];
    }
    for (uint32_t q = 0; q < per; q += 4) {
      uint32_t l[4], h[4], v[4];
      const uint16_t* p[4];
#pragma unroll
      for (uint32_t i = 0; i < 4; ++i) {
        l[i] = (uint32_t)__builtin_amdgcn_readlane((int)lo, (int)(q + i));
        h[i] = (uint32_t)__builtin_amdgcn_readlane((int)hi, (int)(q + i));
        p[i] = ids + (s + S * (j0 + q + i)) * kTileIds;
        v[i] = l[i] + lane < h[i] ? p[i][l[i] + lane] : kBinIds;
      }
#pragma unroll
      for (uint32_t i = 0; i < 4; ++i)
        if (v[i] != kBinIds) atomicAdd(hist + v[i], 1u);
#pragma unroll
      for (uint32_t i = 0; i < 4; ++i)
        for (uint32_t k = l[i] + 64 + lane; k < h[i]; k += 64) atomicAdd(hist + p[i][k], 1u);
    }
  }
  __syncthreads();
  uint32_t* out = part + ((uint64_t)s * nb + bin) * kBinIds;
  for (uint32_t i = tid; i < kBinIds; i += 1024) out[i] = hist[i];
}

__global__ __launch_bounds__(TB) void k_bin_sum(const uint32_t* __restrict__ part, uint32_t bits,
                                                uint32_t S, uint32_t n, uint32_t* __restrict__ h) {
  const uint64_t all = 1ull << bits;
  for (uint64_t i = gtid(); i < all; i += gstride()) {
    uint32_t c = 0;
    for (uint32_t s = 0; s < S; ++s) c += part[s * all + i];
    const uint32_t id = ((uint32_t)i * kHashInv) & (uint32_t)(all - 1);
    if (c && id < n) h[id] += c;
  }
}

constexpr uint64_t kMinBinned = 1u << 20;

// ---- compaction of keys ----------------------------------------------------------
// A wave takes kWaveKeys consecutive keys: k_keep_count counts the kept ones, a scan
// of the counts places them, k_keep_write writes them.  Two reads of the keys
// at memory speed: 6.2 * 10^7 keys 0.36 ms, where a single pass with look-back
// took 1.9.
constexpr uint32_t kWaveKeys = 1024;

// kept: flags[i], or (null) the first of equal keys
__device__ inline bool kept(const uint64_t* __restrict__ key, const uint8_t* __restrict__ flags,
                            uint64_t i, uint64_t k) {
  return flags ? flags[i] != 0 : i == 0 || key[i - 1] != k;
}

__global__ __launch_bounds__(TB) void k_keep_count(const uint64_t* __restrict__ key,
                                                   const uint8_t* __restrict__ flags, uint64_t n,
                                                   uint64_t nw, uint64_t* __restrict__ cnt) {
  const uint32_t lane = threadIdx.x & 63;
  for (uint64_t w = gtid() >> 6; w <= nw; w += gstride() >> 6) {
    uint32_t c = 0;
#pragma unroll 8
    for (uint32_t s = 0; s < kWaveKeys; s += 64) {
      const uint64_t i = w * kWaveKeys + s + lane;
      c += (uint32_t)__popcll(dev::lanes(i < n && kept(key, flags, i, flags ? 0 : key[i])));
    }
    if (lane == 0) cnt[w] = c;  // (entry nw: none)
  }
}

__global__ __launch_bounds__(TB) void k_keep_write(const uint64_t* __restrict__ key,
                                                   const uint8_t* __restrict__ flags, uint64_t n,
                                                   uint64_t nw, const uint64_t* __restrict__ at,
                                                   uint32_t shift, uint64_t* __restrict__ out) {
  const uint64_t low = (1ull << shift) - 1;
  const uint32_t lane = threadIdx.x & 63;
  for (uint64_t w = gtid() >> 6; w < nw; w += gstride() >> 6) {
    uint64_t to = at[w];
#pragma unroll 8
    for (uint32_t s = 0; s < kWaveKeys; s += 64) {
      const uint64_t i = w * kWaveKeys + s + lane;
      const uint64_t k = i < n ? key[i] : 0;
      const bool take = i < n && kept(key, flags, i, k);
      const uint64_t mask = dev::lanes(take);
      if (take) out[to + dev::lanes_below(mask, 0u)] = (k >> shift) << 32 | (k & low);
      to += (uint32_t)__popcll(mask);
    }
  }
}

// ---- largest id ----------------------------------------------------------------
// top[block]: the largest of its share of a (and b, unless null).  One launch and
// one copy for both arrays; the library's reduction took 34 us for each 20,000
// ids, in one workgroup.
constexpr uint32_t kMaxThreads = 1024;

__global__ __launch_bounds__(kMaxThreads) void k_max_ids(const uint32_t* __restrict__ a,
                                                         const uint32_t* __restrict__ b, uint64_t m,
                                                         uint32_t* __restrict__ top) {
  __shared__ uint32_t red[kMaxThreads / 64];
  uint32_t x = 0;
  for (uint64_t i0 = gtid(); i0 < m; i0 += 4 * gstride()) {
#pragma unroll
    for (uint32_t u = 0; u < 4; ++u) {
      const uint64_t i = i0 + u * gstride();
      if (i < m) x = max(x, b ? max(a[i], b[i]) : a[i]);
    }
  }
  for (int off = 32; off > 0; off >>= 1) x = max(x, (uint32_t)__shfl_xor((int)x, off, 64));
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = x;
  __syncthreads();
  if (threadIdx.x == 0) {
    for (uint32_t w = 1; w < kMaxThreads / 64; ++w) x = max(x, red[w]);
    top[blockIdx.x] = x;
  }
}

}  // namespace

int max_ids(tc_ctx* c, const uint32_t* a, const uint32_t* b, uint64_t m, uint32_t* result) {
  *result = 0;
  if (m == 0) return TC_OK;
  constexpr uint32_t kMaxBlocks = 1024;
  const uint32_t G = (uint32_t)std::min<uint64_t>(
      std::min<uint64_t>((m + kMaxThreads - 1) / kMaxThreads, 2ull * c->num_cus), kMaxBlocks);
  TCX_TRY(c->prim_out.reserve(4 * kMaxBlocks));
  uint32_t* top = c->prim_out.as<uint32_t>();
  hipLaunchKernelGGL(k_max_ids, dim3(G), dim3(kMaxThreads), 0, c->stream, a, b, m, top);
  TCX_HIP(hipGetLastError());
  uint32_t h[kMaxBlocks];
  TCX_TRY(fetch(c, h, top, 4 * G));
  *result = *std::max_element(h, h + G);
  return TC_OK;
}

int count_ids(tc_ctx* c, const uint32_t* a, const uint32_t* b, uint64_t m, uint32_t n,
              uint32_t* h) {
  if (m == 0) return TC_OK;
  uint32_t bits = kBinBits;
  while (bits < 32 && (1ull << bits) < n) ++bits;
  const uint64_t ids = b ? 2 * m : m;
  const uint32_t nb = bits - kBinBits < 9 ? 1u << (bits - kBinBits) : kMaxBins + 1;
  const uint64_t tiles = (m + kTileIds - 1) / kTileIds, nt = b ? 2 * tiles : tiles;
  const uint32_t S = std::max<uint32_t>(1, 512 / nb);
  DevBuf bin, border, part;
  // (without the memory for the bins the atomics do)
  if (ids >= kMinBinned && nb <= kMaxBins && nt <= 0x7FFFFFFFull &&
      bin.reserve(2 * nt * kTileIds) == TC_OK && border.reserve(2 * nt * (nb + 1)) == TC_OK &&
      part.reserve((4ull * S) << bits) == TC_OK) {
    for (uint32_t i = 0; i < (b ? 2u : 1u); ++i)
      hipLaunchKernelGGL(k_bin_ids, dim3((unsigned)tiles), dim3(kTileThreads), 0, c->stream,
                         i ? b : a, m, n, bits, nb, bin.as<uint16_t>() + i * tiles * kTileIds,
                         border.as<uint16_t>() + i * tiles * (nb + 1));
    // tiles a wave of a workgroup has
    const uint32_t share = (uint32_t)((nt / S + 16) / 16);
    hipLaunchKernelGGL(k_bin_hist, dim3(nb * S), dim3(1024), 0, c->stream, bin.as<uint16_t>(),
                       border.as<uint16_t>(), (uint32_t)nt, nb, S,
                       std::min<uint32_t>(64, (share + 3) / 4 * 4), part.as<uint32_t>());
    hipLaunchKernelGGL(k_bin_sum, dim3(grid_for(1ull << bits)), dim3(TB), 0, c->stream,
                       part.as<uint32_t>(), bits, S, n, h);
    TCX_HIP(hipGetLastError());
    return TC_OK;
  }
  const unsigned G = (unsigned)std::min<uint64_t>(grid_for(m), (uint64_t)c->num_cus * 4u);
  hipLaunchKernelGGL(dev::k_count_ids<8192>, dim3(G), dim3(256), 0, c->stream, a, b, m, n, h);
  TCX_HIP(hipGetLastError());
  return TC_OK;
}

int compact_u64(tc_ctx* c, const uint64_t* in, const uint8_t* flags, uint64_t n, uint64_t* out,
                uint64_t* n_out, int shift, uint64_t* last) {
  const uint64_t nw = (n + kWaveKeys - 1) / kWaveKeys;
  DevBuf cnt, at;
  TCX_TRY(cnt.reserve(8 * (nw + 1)));
  TCX_TRY(at.reserve(8 * (nw + 1)));
  hipLaunchKernelGGL(k_keep_count, dim3(grid_for(64 * (nw + 1))), dim3(TB), 0, c->stream, in,
                     flags, n, nw, cnt.as<uint64_t>());
  TCX_HIP(hipGetLastError());
  TCX_TRY(exclusive_scan_u64(c, cnt.as<uint64_t>(), at.as<uint64_t>(), nw + 1));
  hipLaunchKernelGGL(k_keep_write, dim3(grid_for(64 * nw)), dim3(TB), 0, c->stream, in, flags, n,
                     nw, at.as<uint64_t>(), (uint32_t)shift, out);
  TCX_HIP(hipGetLastError());
  return fetch2(c, n_out, at.as<uint64_t>() + nw, last, in + n - 1);
}

}  // namespace tcx

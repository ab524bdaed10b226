// Internal declarations shared by the engine's translation units.
#pragma once

#include <hip/hip_runtime.h>

#include <chrono>
#include <cstdint>
#include <cstdio>
#include <memory>
#include <string>
#include <utility>
#include <vector>

#include "../../include/tc_amd.h"

namespace tcx {

// Most oriented edges a CSR may hold: 32-bit offsets, with the last list's
// 64-entry chunks (up to 512 entries past a list's first) still below 2^32.
constexpr uint64_t kMaxCsrEntries = 0xFFFFFFFFull - 512;

// ---- error plumbing ------------------------------------------------------
void set_error(const char* fmt, ...);
int fail(int status, const char* fmt, ...);

#define TCX_HIP(call)                                                        \
  do {                                                                       \
    hipError_t _e = (call);                                                  \
    if (_e != hipSuccess)                                                    \
      return ::tcx::fail(_e == hipErrorOutOfMemory ? TC_ERR_NOMEM : TC_ERR_HIP, \
                         "%s failed: %s (%s:%d)", #call, hipGetErrorString(_e), \
                         __FILE__, __LINE__);                                \
  } while (0)

#define TCX_TRY(expr)          \
  do {                         \
    int _s = (expr);           \
    if (_s != TC_OK) return _s; \
  } while (0)

// ---- device memory --------------------------------------------------------
// Freed blocks of one context, kept for its next buffers (alloc.cpp).  All of
// a context's work is on its one stream, so a block that a freed buffer leaves
// behind is safe for the next buffer of the same context at once.
struct Pool;
// While one lives, this thread's buffers come from the context's pool (NULL,
// or no scope: from hipMalloc).  Entry points that allocate open one.
struct PoolScope {
  explicit PoolScope(const tc_ctx* c);
  ~PoolScope();
  PoolScope(const PoolScope&) = delete;
  PoolScope& operator=(const PoolScope&) = delete;
 private:
  Pool* before;
};
// (null: out of host memory)
std::shared_ptr<Pool> pool_create(int device, uint64_t total_mem);
// The blocks that the context keeps, and those of destroyed ones, back to the
// system.
void pool_release(tc_ctx* c);
// The context's stream is idle: its blocks go to the device's other contexts,
// and back to the system with the last of them.
void pool_retire(std::shared_ptr<Pool> pool);

// Host-to-device copy of pageable memory on the context's stream; the host
// memory has been read when it returns.
int upload(tc_ctx* c, void* dst, const void* src, size_t bytes);
// Device-to-host copy through the context's pinned page (at most kPinBytes);
// waits for the stream.
constexpr size_t kPinBytes = 32768;
int fetch(tc_ctx* c, void* out, const void* src, size_t bytes);
// Two words with one wait (out2 may be null: one).
int fetch2(tc_ctx* c, uint64_t* out, const uint64_t* src, uint64_t* out2, const uint64_t* src2);

// ---- device buffer ------------------------------------------------------
// Owns one region; grows on demand (contents are not kept).
struct DevBuf {
  void* p = nullptr;
  size_t bytes = 0;
  std::shared_ptr<Pool> pool;  // where the region goes back to (null: hipFree)
  DevBuf() = default;
  DevBuf(const DevBuf&) = delete;
  DevBuf& operator=(const DevBuf&) = delete;
  ~DevBuf() { release(); }
  int reserve(size_t want);
  void release();
  template <class T> T* as() const { return static_cast<T*>(p); }
};

inline void swap(DevBuf& a, DevBuf& b) {
  std::swap(a.p, b.p);
  std::swap(a.bytes, b.bytes);
  std::swap(a.pool, b.pool);
}

}  // namespace tcx

struct tc_ctx {
  int device = 0;
  hipStream_t stream = nullptr;
  hipEvent_t ev0 = nullptr, ev1 = nullptr;
  std::shared_ptr<tcx::Pool> pool;
  void* pin = nullptr;      // kPinBytes of pinned host memory
  hipEvent_t lev[17] = {};  // per-launch timing marks (created on first use)
  uint64_t total_mem = 0;
  int num_cus = 256;
  int wall_clock_khz = 100000;  // device wall_clock64() rate
  tcx::DevBuf temp;     // rocprim temp storage
  tcx::DevBuf scratch;  // small per-call scratch (counters, bitmaps)
  tcx::DevBuf accum;    // uint64 accumulators
  tcx::DevBuf prim_out; // 64-byte result slot of the device-wide primitives
  tcx::DevBuf bitmaps;  // Bisson per-workgroup bitmaps, all-zero between calls
  uint64_t bitmap_words = 0;
};

namespace tcx {
// Out-list rows in 16-byte units and the work lists and tasks over them
// (lists16.h).
struct Rows16 {
  DevBuf row;                      // uint2[n]: first unit of the row, units
  DevBuf col;                      // entries, rows padded to whole units
  DevBuf se;                       // uint2[entries]: row of each work-list entry's list
  DevBuf who;                      // uint32[tasks]: owner (its graph, in a batch)
  DevBuf cred;                     // uint32[entries], when built for per-vertex counts
  DevBuf act;                      // uint4[tasks + 1]: entry range, owner's row
  DevBuf slice;                    // uint2[nslice + 1]: first (task, entry) of each slice
  uint64_t units = 0, entries = 0, tasks = 0;
  uint32_t nslice = 0;
  void release() {
    for (DevBuf* b : {&row, &col, &se, &who, &cred, &act, &slice}) b->release();
  }
};
struct Lists16 {
  uint64_t version = ~0ull;        // the CSR it was built (or found unsuitable) for
  bool usable = false;
  bool credit = false;             // built for per-vertex counts too
  bool listed = false;             // with the hub's work lists (else id and cnt to build them)
  DevBuf id, cnt;                  // uint16[n] 16-bit ids (none: all are their own), uint32[n]
  Rows16 hub, tail;                // entries with 16-bit ids, the others (32-bit)
  void release() {
    usable = false;
    for (DevBuf* b : {&id, &cnt}) b->release();
    hub.release();
    tail.release();
  }
};

// Push lists (a task streams the rows of all its out-neighbours) over the hub
// rows of a usable layer, else over the rows of l32, with Hu's and Bisson's
// slices of them.
struct Push16 {
  uint64_t version = ~0ull;
  DevBuf se, act;                  // as in Rows16
  uint64_t tasks = 0;
  DevBuf hu_slice, slice;
  uint32_t hu_blocks = 0, hu_nslice = 0, nslice = 0;
  void release() {
    version = ~0ull;
    for (DevBuf* b : {&se, &act, &hu_slice, &slice}) b->release();
  }
};

// Per-graph schedules, rebuilt when the oriented CSR changes.
struct SchedCache {
  uint64_t version = ~0ull;
  uint32_t hu_nblocks = 0;
  DevBuf hu_start;                 // int32[nblocks+1]
  bool auto_ok = false;
  uint32_t auto_wmax = 0, auto_hmin = 0;  // thresholds the AUTO lists were built for
  DevBuf auto_small;               // vertices with 2 <= d+ <= 64, id order
  DevBuf auto_large;               // d+ in (64, 2048], by descending work
  DevBuf auto_huge;                // d+ > 2048, by descending work
  uint64_t n_small = 0, n_large = 0, n_huge = 0;
  // AUTO over work lists: W(x) CSR (wl_rp, wl_col) and the task lists
  bool wl_ok = false;
  uint32_t wl_wmax = 0, wl_hmin = 0, wl_lmax = 0;
  DevBuf wl_rp, wl_col;            // uint32[n+1], uint32[entries]
  DevBuf wl_se;                    // uint2[entries]: (rp[y], rp[y+1]) of wl_col's y
  DevBuf wl_small, wl_large, wl_huge, wl_lane;
  DevBuf wl_ell;                   // uint32[8 n]: out-lists of <= 8 entries, kEmpty-padded rows
  uint64_t nw_small = 0, nw_large = 0, nw_huge = 0, nw_lane = 0;
  uint64_t wl_entries = 0;         // edges kept in the work lists
  Lists16 l16;
  Lists16 l32;                     // all entries 32-bit (in tail); usable: with work lists
  Push16 push16;
  uint64_t no_rows_version = ~0ull;  // the CSR that l32 or push16 found no room for
  // counts of this CSR so far that did without list rows (up to a bound)
  uint32_t hu_counts = 0, fox_counts = 0, vertex_counts = 0;
  double wl_bytes = 0;             // bytes one count streams (see count.hip)
  bool rows_ok = false;
  DevBuf rows;                     // rows with d+ >= 2
  uint64_t nrows = 0;
  uint32_t fox_lanes = 0;
  bool fox_rearr = false;
  DevBuf fox_eids;                 // edge ids grouped by lanes-per-edge bin
  std::vector<uint64_t> fox_off;   // bin offsets (bins+1)
  uint64_t builds = 0;             // schedules built so far (each waits for the device)
  // learned schedule (per model id)
  uint64_t learned_version = ~0ull, learned_model = ~0ull;
  DevBuf l_blk, l_wav, l_huge, l_lan;
  uint64_t nl_blk = 0, nl_wav = 0, nl_huge = 0, nl_lan = 0;
  uint32_t learned_mask = 0;  // cells whose tasks run narrow
  // learned k-clique plan (per k and model id)
  uint64_t kcl_version = ~0ull, kcl_model = ~0ull;
  uint32_t kcl_k = 0;
  DevBuf kcl_path, kcl_key;
  // k-clique roots, widest first, and how many have d+ > i (see kcl_order)
  uint64_t kcl_order_version = ~0ull;
  DevBuf kcl_order;
  std::vector<uint32_t> kcl_wider;
  // degeneracy-oriented copy of the graph for k-clique counting when the
  // caller's orientation leaves roots wider than the LDS bit matrix
  uint64_t kcl_degen_version = ~0ull;
  std::shared_ptr<tc_graph> kcl_degen;
};
}  // namespace tcx

struct tc_graph {
  tc_ctx* ctx = nullptr;
  uint32_t n = 0;           // rows of the oriented CSR (after pruning, if any)
  uint32_t n_raw = 0;       // every raw record id is below this
  uint64_t m_raw = 0;
  bool csr_only = false;    // built from a CSR (stage file, TriCore parts): no raw records
  tcx::DevBuf src, dst;     // raw records (uint32 each)
  // oriented CSR
  int orient_mode = -1;
  uint64_t m_or = 0;
  uint32_t max_out = 0;
  tcx::DevBuf rowptr;       // uint32[n+1]
  tcx::DevBuf col;          // uint32[m_or]
  tcx::DevBuf esrc;         // uint32[m_or]  source of each CSR edge
  // uint32[n] a degree of each vertex (of the raw records, the simple graph or
  // the CSR's in-edges, whichever the orientation had at hand) and the CSR it
  // goes with; vertex_degrees() makes it when there is none
  tcx::DevBuf vdeg;
  uint64_t vdeg_version = ~0ull;
  tcx::DevBuf vkey;         // int32[n] ADIR priority / KCORE core number
  uint64_t sum_out_sq = 0, sum_in_out = 0;
  // tc_graph_device_csr gave the CSR's addresses out: work on any stream may
  // read it, so its memory is let go only when the device is idle
  mutable bool exported = false;
  // cached schedules (valid for the current CSR)
  uint64_t sched_version = 0;
  tcx::SchedCache sc;
};

namespace tcx {

// ---- primitives (prims.hip) ---------------------------------------------
// Ascending by bits [begin_bit, end_bit), stable.
int sort_u64(tc_ctx* c, uint64_t* keys, uint64_t* tmp, uint64_t n, int end_bit,
             uint64_t** sorted, int begin_bit = 0);
int sort_pairs_u64_u32(tc_ctx* c, uint64_t* keys, uint64_t* ktmp, uint32_t* vals,
                       uint32_t* vtmp, uint64_t n, int end_bit, uint64_t** skeys,
                       uint32_t** svals);
int sort_pairs_u32_u32(tc_ctx* c, uint32_t* keys, uint32_t* ktmp, uint32_t* vals,
                       uint32_t* vtmp, uint64_t n, int end_bit, uint32_t** skeys,
                       uint32_t** svals);
// (shift, last: as for compact_u64; shift 32 below kMinCompact keys)
int unique_u64(tc_ctx* c, const uint64_t* in, uint64_t* out, uint64_t n,
               uint64_t* n_out, int shift = 32, uint64_t* last = nullptr);
int exclusive_scan_u32(tc_ctx* c, const uint32_t* in, uint32_t* out, uint64_t n);
int exclusive_scan_u64(tc_ctx* c, const uint64_t* in, uint64_t* out, uint64_t n);
int inclusive_scan_i64(tc_ctx* c, const int64_t* in, int64_t* out, uint64_t n);
int sum_u64(tc_ctx* c, const uint64_t* in, uint64_t n, uint64_t* result);
int min_i32(tc_ctx* c, const int32_t* in, uint64_t n, int32_t* result);
int select_flagged_u32(tc_ctx* c, const uint32_t* in, const uint8_t* flags,
                       uint32_t* out, uint64_t n, uint64_t* n_out);
int select_indices(tc_ctx* c, const uint8_t* flags, uint64_t n, uint32_t* out,
                   uint64_t* n_out);
int select_flagged_u64(tc_ctx* c, const uint64_t* in, const uint8_t* flags,
                       uint64_t* out, uint64_t n, uint64_t* n_out);

// ---- passes over long arrays (passes.hip) ----------------------------------
// h[x] += occurrences of x < n in a[0, m) (and b[0, m) when b is not null).
int count_ids(tc_ctx* c, const uint32_t* a, const uint32_t* b, uint64_t m, uint32_t n,
              uint32_t* h);
// The keys with flags[i] set, or (flags null) the first of each run of equal
// keys, in order; out must not be in.  Keys a << shift | b come out as
// a << 32 | b.  last (optional) receives the last key of in.
int compact_u64(tc_ctx* c, const uint64_t* in, const uint8_t* flags, uint64_t n, uint64_t* out,
                uint64_t* n_out, int shift = 32, uint64_t* last = nullptr);
// The largest of a[0, m) (and b[0, m) when b is not null), 0 for m = 0.
int max_ids(tc_ctx* c, const uint32_t* a, const uint32_t* b, uint64_t m, uint32_t* result);
// Keys from which on compact_u64 takes over from the single pass (two more
// launches, so small inputs keep it).
constexpr uint64_t kMinCompact = 1u << 20;

// ---- graph helpers (graph.hip) -------------------------------------------
int build_csr_from_keys(tc_ctx* c, tc_graph* g, uint64_t* keys, uint64_t nkeys,
                        int end_bit);
int compute_csr_stats(tc_ctx* c, tc_graph* g);
int vertex_degrees(tc_ctx* c, tc_graph* g);
int build_sym(tc_ctx* c, tc_graph* g, DevBuf& rowptr, DevBuf& col, uint64_t* m2);
// A new graph holding a device copy of g's raw records (not oriented); its
// vertex count is the records' largest id + 1.  A graph without raw records
// (csr_only) gives its oriented CSR's edges instead.
int graph_clone_records(tc_ctx* c, const tc_graph* g, tc_graph** out);

// ---- work lists of the AUTO engine (count.hip) ---------------------------
// Builds (or keeps) the default work-list schedule of g: sc.wl_rp / wl_col
// and the fixed rule's task lists.
int worklists(tc_ctx* c, tc_graph* g);

// ---- the 16-bit list layer (lists16.hip) -----------------------------------
// Builds (or keeps) g's layer when its lists suit it and there is memory for it
// (g->sc.l16.usable).  credit: for per-vertex counts too.
int lists16(tc_ctx* c, tc_graph* g, bool credit = false);
// The layer where usable, else (l32) the same over 32-bit rows of all entries.
int lists16or32(tc_ctx* c, tc_graph* g, const Lists16** use);
// Bytes that one count over a layer with work lists streams.
int rows_bytes(tc_ctx* c, const Lists16& L, double* bytes);
// After a failure of lists16or32, hu16 or bisson16: where the rows have no room
// (memory, or 2^32 units) they are let go, the CSR is counted without them
// from now on, and the status is TC_OK.
int without_rows(tc_graph* g, int status);
// Enqueues the count over them; acc: kAccBytes16 bytes, cleared; sum16 adds the
// copied-back accumulators.
constexpr size_t kAccBytes16 = 8 * 64 * 16;
int count16(tc_ctx* c, const Lists16& L, uint32_t grid, unsigned long long* acc,
            uint32_t* launches);
unsigned long long sum16(const unsigned long long* acc);
// Push lists with slices for Hu's vertex blocks start[0 .. nblocks] (device
// array), or of equally many edges each (Bisson's method).
int hu16(tc_ctx* c, tc_graph* g, const int32_t* start, uint32_t nblocks);
int bisson16(tc_ctx* c, tc_graph* g);
int count_push16(tc_ctx* c, tc_graph* g, const DevBuf& slice, uint32_t nslice, uint32_t grid,
                 unsigned long long* acc, uint32_t* launches);
// tri[u] += the triangles whose first vertex is u, over a layer built with
// credit; cursor: kCurBytes16 bytes, cleared.
constexpr size_t kCurBytes16 = 64 * 128;
int count16_vertices(tc_ctx* c, tc_graph* g, uint32_t* cursor, unsigned long long* tri);
// The same for a batch's union graph: 16-bit ids are the ids within each
// graph (vertex v of graph gid[v], which starts at voff[gid[v]]; device
// arrays), so every graph must have at most 65,535 vertices.  Counts go to
// counts[graph]; cursor: kCurBytes16 bytes, cleared.
int lists16_batch(tc_ctx* c, tc_graph* g, const uint32_t* gid, const uint32_t* voff);
int count16_graphs(tc_ctx* c, tc_graph* g, uint32_t grid, uint32_t* cursor,
                   unsigned long long* counts);

inline float ms_since(std::chrono::steady_clock::time_point t0) {
  return std::chrono::duration<float, std::milli>(std::chrono::steady_clock::now() - t0).count();
}

// Event marks around count launches: mark() before each launch, stop() where
// other work follows one (else the next mark ends its interval), end() after
// the last; finish(), once the stream has been waited for, gives the total and
// the longest launch.
struct LaunchMarks {
  tc_ctx* c;
  int n = 0;                // intervals
  int ev = 0;               // events recorded
  int first[16], last[16];  // an interval's events
  bool open = false;
  explicit LaunchMarks(tc_ctx* cc) : c(cc) {}
  int record() {
    if (!c->lev[ev]) TCX_HIP(hipEventCreate(&c->lev[ev]));
    TCX_HIP(hipEventRecord(c->lev[ev], c->stream));
    return TC_OK;
  }
  int mark() {
    if (ev >= 16) return TC_OK;  // later launches fold into the last interval
    TCX_TRY(record());
    if (open) last[n - 1] = ev;
    first[n++] = ev++;
    open = true;
    return TC_OK;
  }
  int stop() {
    if (!open || ev >= 16) return TC_OK;
    TCX_TRY(record());
    last[n - 1] = ev++;
    open = false;
    return TC_OK;
  }
  int end() {
    if (!open) return TC_OK;
    TCX_TRY(record());
    last[n - 1] = ev;
    open = false;
    return TC_OK;
  }
  int finish(tc_timing* tm) {
    tm->ms_count = 0;
    tm->ms_dominant = 0;
    for (int i = 0; i < n; ++i) {
      float ms = 0;
      TCX_HIP(hipEventElapsedTime(&ms, c->lev[first[i]], c->lev[last[i]]));
      tm->ms_count += ms;
      if (ms > tm->ms_dominant) {
        tm->ms_dominant = ms;
        tm->dominant_kernel = (uint32_t)i;
      }
    }
    return TC_OK;
  }
};

// ---- cost model and per-vertex counts (mlp.hip, count.hip) ---------------
// Predicted log2 costs Y[n][2] for device features X[n][8]; fails when the
// model belongs to another context.
int model_predict(tc_ctx* c, tc_model* m, const float* dX, uint32_t n, float* dY);
// Identity of the model's current parameters (changes with every update).
uint64_t model_id(const tc_model* m);
// tri[u] = |{v -> w : v, w in N+(u)}|, the edges of the sub-graph of N+(u)
// (uint64 per vertex, device array of n entries).
int per_vertex_counts(tc_ctx* c, tc_graph* g, unsigned long long* tri);

// ---- allocation-free counting (noalloc.hip) --------------------------------
// Looks up the device address of the static scratch array on `device` (the
// device must be current); called once per device by tc_ctx_create.
int noalloc_setup(int device);

// ---- A-order (aorder.cpp, host heap) -------------------------------------
int aorder_perm_from_outdeg(const uint32_t* rtd, uint32_t n, uint32_t* perm,
                            const tc_bw_model& model);
void bw_model_reference(tc_bw_model* m);

// ---- host parallel-for ----------------------------------------------------
void parallel_for(uint64_t n, void (*fn)(uint64_t begin, uint64_t end, void* arg),
                  void* arg, unsigned max_threads = 0);

inline int bit_width_u32(uint32_t x) {
  int b = 0;
  while (x) { ++b; x >>= 1; }
  return b;
}

constexpr int kWave = 64;

}  // namespace tcx
